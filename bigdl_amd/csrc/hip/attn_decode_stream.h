// Decode attention whose K and V^T arrive in whole 128-byte lines, by DMA into LDS (included by attn_decode.hip,
// which also states the cache layout and the products' operand order).
//
// What bounds it is the K / V stream, and what decides the rate of that stream is the pattern: fragments loaded straight into
// registers are 16 rows x 64 bytes a request, and two requests (of different wavefronts, for V^T) share every 128-byte line.  524 MB of
// e5m2 keys and values (64 sequences x 32 heads, 1000 keys) read that way by an otherwise empty kernel take 92 us (99 non-temporal), in
// whole lines 90, in whole lines and non-temporal 80.  Hence:
//  * a block is NW x 64 bytes of every V^T row (64 e5m2 or 32 fp16 keys a wavefront).  Scores are split over the wavefronts by keys,
//    O over them by channels, so that what a wavefront requests -- its keys' rows, its channels' rows -- is its own and needs no
//    barrier; the probabilities change hands in LDS (`rows` x 64 keys a wavefront), double-buffered, one barrier a block.  O needs no merge.
//  * the requests hold no registers: K of the next block leaves as soon as this one's keys are in registers, V^T the same, so each
//    wavefront has 8 - 16 KiB under way and a CU (eight wavefronts, 160 KiB of LDS) 64 - 128; the 27 bytes / ns that a CU can draw
//    times 2 us of loaded latency are 54.
//  * the first block is requested before anything else but q.  The new key and value are put into their block in LDS, so nobody waits
//    for the append; the 64 bytes of a V^T row that hold the new value are stored whole.
// Measured, register form -> this one: that case 120 -> 100 us a launch (without the append 95 -> 89, so the rest are the 262144 stores
// of 64 bytes; whole lines and non-temporal stores cost more; of the loads' 84 nothing is left but the stream: without the products it
// takes as long); 12 sequences x 8 heads of 128, fp16, 1900 keys in two ranges 32 -> 25.5.  Two blocks under way per wavefront instead
// of one: equal to 40 % slower (fewer wavefronts a CU); eight wavefronts a workgroup: up to 8 % faster in long single ranges, 10 - 50 %
// slower elsewhere.
// 16-byte chunks of a row stand in LDS under chunk ^ (row bits), by permuting the source addresses inside each line.
#pragma once

namespace bigdl {

__device__ __forceinline__ void attn_dma16(__amdgpu_buffer_rsrc_t b, char* lds, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(b, (__attribute__((address_space(3))) void*)lds, 16, off, 0, 0, 2 /* non-temporal */);
}
constexpr int attn_vm_lgkm0(int n) { return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4); }       // s_waitcnt vmcnt(n) lgkmcnt(0)

template <int D, bool FP8, int NW, int RT>
constexpr size_t attn_stream_lds(int rows) {
  return (size_t)NW * (D * 128) + 2 * NW * rows * (FP8 ? 128 : 64) + 3 * NW * RT * 64;
}

// RT = 16-row tiles of query rows (G query heads x the launch's new tokens, of which MULTI has several).  A row's result does not depend
// on the rows beside it.
template <int D, bool FP8, int NW, int RT, bool MULTI>
__global__ __launch_bounds__(NW * 64, 2) void attn_stream_kernel(const int* p_past, _Float16* p_qkv, int p_ld, int p_splits, int p_Hq,
                                                                              int p_Hkv, int p_Lmax, void* p_kc, void* p_vc, AttnArgs a) {
  a.past_len = p_past; a.qkv = p_qkv; a.ld = p_ld; a.splits = p_splits; a.Hq = p_Hq; a.Hkv = p_Hkv; a.Lmax = p_Lmax;
  constexpr int ES = FP8 ? 1 : 2;
  constexpr int DC = D / 32;                 // k-steps of the scores
  constexpr int CH = D / NW, DTW = CH / 16;  // channels and 16-channel tiles of O per wavefront
  constexpr int KW = 64 / ES;                // keys per wavefront and block
  constexpr int KL = KW / 4, NU = KW / 16;
  constexpr int BK = NW * KW;
  constexpr int RB = D * ES;                 // bytes of a key
  constexpr int RV = NW * 64;                // bytes of a V^T row in a block
  constexpr int NR = D / 16;                 // requests per wavefront: K of a block, V^T of a block
  // e5m2 bytes straight into the fp8 matrix instruction (q and probabilities as two e4m3 terms), as in the register form: heads of 128
  // (16 bytes of a key are two k-steps); heads of 64 are widened to fp16, as they are there
  constexpr bool F8M = FP8 && D == 128;
  static_assert(CH >= 16, "one 16-channel tile per wavefront at least");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rr = lane & 15, g = lane >> 4;
  const int split = blockIdx.x, hkv = blockIdx.y, b = blockIdx.z;
  const int G = a.Hq / a.Hkv, q_total = MULTI ? a.q_total : 1, rows = MULTI ? G * a.q_cnt : G;
  auto token = [&](int row) { return MULTI ? a.q_off + row / G : 0; };
  auto head = [&](int row) { return hkv * G + (MULTI ? row % G : row); };
  constexpr int PB = FP8 ? 128 : 64;         // LDS bytes of a row's probabilities, one wavefront's keys
  char* sk = smem + wave * (D * 128);                                   // this wavefront's keys of a block, then its V^T rows
  char* svt = sk + D * 64;
  char* sp = smem + NW * (D * 128);                                    // [2][NW][row][PB]
  float* s_m = (float*)(sp + 2 * NW * rows * PB);                       // [2][NW][RT * 16]
  float* s_l = s_m + 2 * NW * RT * 16;                                  // [NW][RT * 16]

  const int past = a.past_len[b];
  const int kv_len = min(past + q_total, a.Lmax);
  const int nblk = (kv_len + BK - 1) / BK;
  const int per = (nblk + a.splits - 1) / a.splits;
  const int blk0 = split * per, blk1 = min(nblk, blk0 + per);
  const int64_t base = ((int64_t)b * a.Hkv + hkv) * (int64_t)a.Lmax * RB;
  char* kc = (char*)p_kc + base;
  char* vc = (char*)p_vc + base;
  const int half_rot = a.rot >> 1;
  const bool appends = a.rope != nullptr || a.rot == 0;
  const bool append = appends && !MULTI && past < a.Lmax && past >= blk0 * BK && past < blk1 * BK;     // one token: into its block in LDS
  const int kw_new = (past % BK) / KW;       // the wavefront with the new key

  // ---- requests ----
  auto swz_k = [&](int kl) { return RB >= 128 ? (kl & 3) | (((kl / KL) & 1) << 2) : ((kl >> 1) & 1) | (((kl / KL) & 1) << 1); };
  const uint32_t head_bytes = (uint32_t)a.Lmax * RB;
  const __amdgpu_buffer_rsrc_t kbuf = __builtin_amdgcn_make_buffer_rsrc(kc, 0, head_bytes, 0x00027000);
  const __amdgpu_buffer_rsrc_t vbuf = __builtin_amdgcn_make_buffer_rsrc(vc, 0, head_bytes, 0x00027000);
  constexpr uint32_t NONE = 0x80000000u;     // beyond every buffer: nothing is fetched (the launcher keeps heads below 2 GiB)
  auto request_k = [&](int kb, int end) {
    const bool on = kb + wave * KW < end;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int kl = i * (1024 / RB) + lane / (RB / 16);
      const uint32_t off = (uint32_t)(kb + wave * KW + kl) * RB + (((lane % (RB / 16)) ^ swz_k(kl)) << 4);
      attn_dma16(kbuf, sk + i * 1024, on ? off : NONE);
    }
  };
  auto request_v = [&](int kb, int end) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int ch = i * (16 / NW) + lane / (4 * NW);
      const int gc = (lane % (4 * NW)) ^ (ch & 7);
      const uint32_t off = (uint32_t)(wave * CH + ch) * (uint32_t)(a.Lmax * ES) + (uint32_t)(kb * ES) + (gc << 4);
      attn_dma16(vbuf, svt + i * 1024, kb + (gc >> 2) * KW < end ? off : NONE);
    }
  };

  // first head channel of this lane's 8 values in k-step c (as in the register form: the rotate-half partner is k-step c + DC / 2)
  auto chan = [](int c, int g) { return F8M ? 64 * (c >> 1) + 16 * g + 8 * (c & 1) : 32 * c + 8 * g; };
  const bool rotate = a.rope != nullptr;
  const _Float16* krow = a.qkv + (int64_t)b * q_total * a.ld + (int64_t)(a.Hq + hkv) * D;
  // the channel pair (i0, i1) of the new keys that this lane rotates
  const int pair = min(lane, D / 2 - 1);
  const bool rot_pair = rotate && pair < half_rot;
  const int i0 = !rot_pair ? max(a.rot, 0) + 2 * (pair - max(half_rot, 0)) : a.interleaved ? 2 * pair : pair;
  const int i1 = rot_pair && !a.interleaved ? pair + half_rot : i0 + 1;
  auto table_row = [&](int tok) {
    const int pos = max(min(a.position_ids ? a.position_ids[b * q_total + tok] : past + tok, a.rope_max_pos - 1), 0);
    return a.rope + (int64_t)pos * half_rot * 2;
  };
  auto rotated = [&](float u, float w, float2 cs, float& y0, float& y1) {
    y0 = rot_pair ? fmaf(u, cs.x, -(w * cs.y)) : u;
    y1 = rot_pair ? fmaf(w, cs.x, u * cs.y) : w;
  };
  // several new tokens: those of this range go to the cache first
  if (MULTI && appends && a.q_off == 0) {
    for (int t = wave; t < q_total; t += NW) {
      const int p = past + t;
      if (p < blk0 * BK || p >= blk1 * BK || p >= a.Lmax) continue;
      const _Float16* kt = krow + (int64_t)t * a.ld;
      const _Float16* vt = kt + (int64_t)a.Hkv * D;
      if (lane < D / 2) {
        float y0, y1;
        rotated((float)kt[i0], (float)kt[i1], rot_pair ? *(const float2*)(table_row(t) + 2 * pair) : float2{1.0f, 0.0f}, y0, y1);
        if constexpr (FP8) {
          ((uint8_t*)kc)[(int64_t)p * D + i0] = f16_to_e5m2((_Float16)y0);
          ((uint8_t*)kc)[(int64_t)p * D + i1] = f16_to_e5m2((_Float16)y1);
        } else {
          ((_Float16*)kc)[(int64_t)p * D + i0] = (_Float16)y0;
          ((_Float16*)kc)[(int64_t)p * D + i1] = (_Float16)y1;
        }
      }
      for (int d = lane; d < D; d += 64) {
        if constexpr (FP8) ((uint8_t*)vc)[(int64_t)d * a.Lmax + p] = f16_to_e5m2(vt[d]);
        else ((_Float16*)vc)[(int64_t)d * a.Lmax + p] = vt[d];
      }
    }
    __syncthreads();
  }
  // ---- q, its rotation, the new key and value, then the first block (all without a branch: what arrives is counted) ----
  half8 qraw[RT][DC];
  typedef float __attribute__((ext_vector_type(4), aligned(8))) pairs2;      // two pairs of a table that may start anywhere
  float4v cs[RT][DC][2];     // [2 i], [2 i + 1]: cosine and sine of 8 / 2 channel pairs each (without a rotation: any readable numbers)
  int row[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    row[t] = min(16 * t + rr, rows - 1);
    const int tok = token(row[t]);
    const _Float16* qp = a.qkv + ((int64_t)b * q_total + tok) * a.ld + (int64_t)head(row[t]) * D;
#pragma unroll
    for (int c = 0; c < DC; ++c) qraw[t][c] = *(const half8*)(qp + chan(c, g));
    const float* tab = rotate ? table_row(tok) : (const float*)qp;
#pragma unroll
    for (int i = 0; i < DC; ++i) {
      const int at = a.interleaved ? (chan(i, g) < a.rot ? chan(i, g) : 0) : 2 * chan(i >> 1, g) + 8 * (i & 1);
      const float* p = tab + (rotate ? at : 0);
      cs[t][i][0] = *(const pairs2*)p;
      cs[t][i][1] = *(const pairs2*)(p + 4);
    }
  }
  const _Float16 x0 = krow[i0], x1 = krow[i1];
  const float2 kcs = *(const float2*)(rot_pair ? table_row(0) + 2 * pair : (const float*)a.qkv);
  const _Float16 nv = krow[(int64_t)a.Hkv * D + wave * CH + min(lane, CH - 1)];
  const int first_end = blk0 < blk1 ? kv_len : 0;
  request_k(blk0 * BK, first_end);
  request_v(blk0 * BK, first_end);
  __builtin_amdgcn_sched_barrier(0);

  const float qscale = a.softcap > 0.0f ? a.scale : a.scale * 1.4426950408889634f;
  half8 qf[RT][F8M ? 1 : DC];
  uint2v qh[RT][F8M ? DC : 1], ql[RT][F8M ? DC : 1];
  float q_unscale[RT], slope[RT];
  int lim[RT], lo_lim[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const bool valid = 16 * t + rr < rows;
    float qv[DC][8];
#pragma unroll
    for (int c = 0; c < DC; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) qv[c][j] = valid ? (float)qraw[t][c][j] : 0.0f;
    if (rotate) {
      if (a.interleaved) {
#pragma unroll
        for (int c = 0; c < DC; ++c) {
          if (chan(c, g) < a.rot) {
#pragma unroll
            for (int j = 0; j < 8; j += 2) {
              const float co = cs[t][c][j >> 2][j & 3], si = cs[t][c][j >> 2][(j & 3) + 1], u = qv[c][j], w = qv[c][j + 1];
              qv[c][j] = u * co - w * si;
              qv[c][j + 1] = w * co + u * si;
            }
          }
        }
      } else {
#pragma unroll
        for (int c = 0; c < DC / 2; ++c) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float4v p = cs[t][2 * c + (j >> 2)][(j >> 1) & 1];
            const float co = p[2 * (j & 1)], si = p[2 * (j & 1) + 1], u = qv[c][j], w = qv[c + DC / 2][j];
            qv[c][j] = u * co - w * si;
            qv[c + DC / 2][j] = w * co + u * si;
          }
        }
      }
    }
    q_unscale[t] = 1.0f;
    if constexpr (F8M) {
      float am = 0.0f;
#pragma unroll
      for (int c = 0; c < DC; ++c)
#pragma unroll
        for (int j = 0; j < 8; ++j) am = fmaxf(am, fabsf(qv[c][j]));
      am = fmaxf(am, __shfl_xor(am, 16));
      am = fmaxf(am, __shfl_xor(am, 32));
      const float f = am > 0.0f ? P8_SCALE / am : 0.0f;
      q_unscale[t] = am * (qscale / P8_SCALE);
#pragma unroll
      for (int c = 0; c < DC; ++c) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = qv[c][j] * f;
        split_e4m3(x, qh[t][c], ql[t][c]);
      }
    } else {
#pragma unroll
      for (int c = 0; c < DC; ++c) {
        half8 v;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = (_Float16)(qv[c][j] * qscale);
        qf[t][c] = v;
      }
    }
    const int last = past + token(row[t]);
    lim[t] = valid ? last : -1;
    lo_lim[t] = a.window > 0 && valid ? max(0, last - a.window + 1) : 0;
    slope[t] = a.alibi != nullptr ? a.alibi[head(row[t])] * 1.4426950408889634f : 0.0f;
  }

  float m_all[RT], l_run[RT];      // running maximum of the row, the same in every wavefront; sum over this lane's keys relative to it
  float psum[RT];                  // of this block: this lane's keys relative to the wavefront's own maximum (m_new)
  float4v o[RT][DTW];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    m_all[t] = NEG_BIG;
    l_run[t] = 0.0f;
#pragma unroll
    for (int d = 0; d < DTW; ++d) o[t][d] = float4v{0, 0, 0, 0};
  }

  for (int blk = blk0; blk < blk1; ++blk) {
    const int kb = blk * BK, kbw = kb + wave * KW;
    const bool more = blk + 1 < blk1;
    const int par = (blk - blk0) & 1;
    // ---- this wavefront's keys (V^T of the block is behind them) ----
    __builtin_amdgcn_s_waitcnt(attn_vm_lgkm0(NR));
    __builtin_amdgcn_sched_barrier(0);
    if (append && !more && wave == kw_new && lane < D / 2) {
      const int kl = (past % BK) % KW;
      auto put = [&](int c, float x) {
        char* dst = sk + kl * RB + ((((c * ES) >> 4) ^ swz_k(kl)) << 4) + ((c * ES) & 15);
        if constexpr (FP8) {
          const uint8_t e = f16_to_e5m2((_Float16)x);
          *(uint8_t*)dst = e;
          ((uint8_t*)kc)[(int64_t)past * D + c] = e;
        } else {
          *(_Float16*)dst = (_Float16)x;
          ((_Float16*)kc)[(int64_t)past * D + c] = (_Float16)x;
        }
      };
      float y0, y1;
      rotated((float)x0, (float)x1, kcs, y0, y1);
      put(i0, y0);
      put(i1, y1);
    }
    const bool mine = kbw < kv_len;
    half8 kf[FP8 ? 1 : NU][FP8 ? 1 : DC];
    uint2v kr[FP8 ? NU : 1][FP8 ? DC : 1];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int kl = KL * (rr >> 2) + 4 * u + (rr & 3);
      const char* src = sk + kl * RB;
      if constexpr (F8M) {
#pragma unroll
        for (int c2 = 0; c2 < DC / 2; ++c2) {
          const uint4v w = *(const uint4v*)(src + (((4 * c2 + g) ^ swz_k(kl)) << 4));
          kr[u][2 * c2] = uint2v{w[0], w[1]};
          kr[u][2 * c2 + 1] = uint2v{w[2], w[3]};
        }
      } else if constexpr (FP8) {
#pragma unroll
        for (int c = 0; c < DC; ++c) kr[u][c] = *(const uint2v*)(src + (((2 * c + (g >> 1)) ^ swz_k(kl)) << 4) + 8 * (g & 1));
      } else {
#pragma unroll
        for (int c = 0; c < DC; ++c) kf[u][c] = *(const half8*)(src + (((4 * c + g) ^ swz_k(kl)) << 4));
      }
    }
    __builtin_amdgcn_s_waitcnt(attn_vm_lgkm0(63));
    __builtin_amdgcn_sched_barrier(0);
    if (more) request_k(kb + BK, kv_len);
    // (the row tiles side by side, not one after the other: 64 groups of two tiles of 64 channels, 1000 keys 19.8 -> 17.6)
    float m_new[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      m_new[t] = NEG_BIG;
      psum[t] = 0.0f;
    }
    if (mine) {
      const int kfirst = kbw + KL * g;
      float sv[RT][KL];
#pragma unroll
      for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          float4v su = {0, 0, 0, 0};
#pragma unroll
          for (int c = 0; c < DC; ++c) {
            if constexpr (F8M) {
              su = mfma_bf8_fp8(kr[u][c], qh[t][c], su);
              su = mfma_bf8_fp8(kr[u][c], ql[t][c], su);
            } else if constexpr (FP8) {
              su = mfma16(dec_e5m2(kr[u][c].x, kr[u][c].y), qf[t][c], su);
            } else {
              su = mfma16(kf[u][c], qf[t][c], su);
            }
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) sv[t][4 * u + q] = F8M ? su[q] * q_unscale[t] : su[q];
        }
      if (a.softcap > 0.0f) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
          for (int q = 0; q < KL; ++q) sv[t][q] = a.softcap * tanhf(sv[t][q] / a.softcap) * 1.4426950408889634f;
      }
      if (a.alibi != nullptr) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
          for (int q = 0; q < KL; ++q) sv[t][q] += slope[t] * (float)(kfirst + q - lim[t]);
      }
      if (a.mask) {
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          if (16 * t + rr >= rows) continue;
          const _Float16* mp = a.mask + ((int64_t)b * q_total + token(row[t])) * a.mask_ld + kfirst;
#pragma unroll
          for (int q = 0; q < KL; ++q)
            if (kfirst + q < a.mask_ld) sv[t][q] += (float)mp[q] * 1.4426950408889634f;
        }
      }
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int q = 0; q < KL; ++q) {
          const int key = kfirst + q;
          if (key > lim[t] || key < lo_lim[t]) sv[t][q] = NEG_BIG;
          m_new[t] = fmaxf(m_new[t], sv[t][q]);
        }
#pragma unroll
      for (int t = 0; t < RT; ++t) m_new[t] = fmaxf(m_new[t], __shfl_xor(m_new[t], 16));
#pragma unroll
      for (int t = 0; t < RT; ++t) m_new[t] = fmaxf(m_new[t], __shfl_xor(m_new[t], 32));
      // Relative to these KW keys' own maximum: in 16 bits or two e4m3 terms a weight loses bits far below what it is relative to.
      // 1000 keys, one of them with e^9 (e5m2) or e^14 (fp16) times the others' weights and a value of zero, error against float64:
      // relative to the running maximum of all keys 0.0031 - 0.0076, of each wavefront's keys 0.0014 - 0.0033, so 0.0010 - 0.0018
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int q = 0; q < KL; ++q) {
          sv[t][q] = sv[t][q] <= NEG_BIG ? 0.0f : (F8M ? P8_SCALE : 1.0f) * __builtin_amdgcn_exp2f(sv[t][q] - m_new[t]);
          psum[t] += sv[t][q];
        }
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        char* pw = sp + ((par * NW + wave) * rows + 16 * t + rr) * PB + 16 * g;
        const bool valid = 16 * t + rr < rows;
        if constexpr (F8M) {
          uint2v h0, l0, h1, l1;
          split_e4m3(*(const float(*)[8]) & sv[t][0], h0, l0);
          split_e4m3(*(const float(*)[8]) & sv[t][8], h1, l1);
          if (valid) {
            *(uint4v*)pw = uint4v{h0.x, h0.y, h1.x, h1.y};
            *(uint4v*)(pw + 64) = uint4v{l0.x, l0.y, l1.x, l1.y};
          }
        } else {
#pragma unroll
          for (int h = 0; h < KL / 8; ++h) {
            half8 p;
#pragma unroll
            for (int q = 0; q < 8; ++q) p[q] = (_Float16)sv[t][8 * h + q];
            if (valid) *(half8*)(pw + 64 * h) = p;
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < RT; ++t)
      if (g == 0) s_m[((par * NW + wave) * RT + t) * 16 + rr] = m_new[t];
    // ---- everybody's probabilities, this wavefront's channels ----
    if (more) __builtin_amdgcn_s_waitcnt(attn_vm_lgkm0(NR));
    else __builtin_amdgcn_s_waitcnt(attn_vm_lgkm0(0));
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (append && !more) {
      const int at = (past % BK) * ES;
      if (lane < CH) {
        char* dst = svt + lane * RV + (((at >> 4) ^ (lane & 7)) << 4) + (at & 15);
        if constexpr (FP8) *(uint8_t*)dst = f16_to_e5m2(nv);
        else *(_Float16*)dst = nv;
      }
#pragma unroll
      for (int j = 0; j < DTW; ++j) {
        const int ch = 16 * j + (lane >> 2), ck = 4 * (at >> 6) + (lane & 3);
        const uint4v w = *(const uint4v*)(svt + ch * RV + ((ck ^ (ch & 7)) << 4));
        __builtin_amdgcn_raw_buffer_store_b128(w, vbuf, (uint32_t)(wave * CH + ch) * (uint32_t)(a.Lmax * ES) + (uint32_t)(kb * ES + 16 * ck), 0,
                                               17 /* written through: 64 x 32 heads, 1000 e5m2 keys 107 -> 103 us */);
      }
    }
    uint4v vr[DTW][NW], ph[RT][NW], pl[RT][FP8 ? NW : 1];
    float mw[RT][NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        mw[t][w] = s_m[((par * NW + w) * RT + t) * 16 + rr];
        const char* pr = sp + ((par * NW + w) * rows + row[t]) * PB + 16 * g;
        ph[t][w] = *(const uint4v*)pr;
        if constexpr (FP8) pl[t][w] = *(const uint4v*)(pr + 64);
      }
#pragma unroll
      for (int d = 0; d < DTW; ++d) vr[d][w] = *(const uint4v*)(svt + (16 * d + rr) * RV + (((4 * w + g) ^ (rr & 7)) << 4));
    }
    __builtin_amdgcn_s_waitcnt(attn_vm_lgkm0(63));
    __builtin_amdgcn_sched_barrier(0);
    if (more) request_v(kb + BK, kv_len);
    auto times = [&](int t, int d, int w, float4v c) {
      if constexpr (FP8 && !F8M) {
        c = mfma16(dec_e5m2(vr[d][w][0], vr[d][w][1]), __builtin_bit_cast(half8, ph[t][w]), c);
        return mfma16(dec_e5m2(vr[d][w][2], vr[d][w][3]), __builtin_bit_cast(half8, pl[t][w]), c);
      } else if constexpr (F8M) {
        const uint2v v0 = {vr[d][w][0], vr[d][w][1]}, v1 = {vr[d][w][2], vr[d][w][3]};
        c = mfma_bf8_fp8(v0, uint2v{ph[t][w][0], ph[t][w][1]}, c);
        c = mfma_bf8_fp8(v1, uint2v{ph[t][w][2], ph[t][w][3]}, c);
        c = mfma_bf8_fp8(v0, uint2v{pl[t][w][0], pl[t][w][1]}, c);
        return mfma_bf8_fp8(v1, uint2v{pl[t][w][2], pl[t][w][3]}, c);
      } else {
        return mfma16(__builtin_bit_cast(half8, vr[d][w]), __builtin_bit_cast(half8, ph[t][w]), c);
      }
    };
    // each wavefront's share is scaled by its own maximum against the row's (in the vector unit: a row never depends on the rows beside it)
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      float m_next = m_all[t];
#pragma unroll
      for (int w = 0; w < NW; ++w) m_next = fmaxf(m_next, mw[t][w]);
      const float alpha = __builtin_amdgcn_exp2f(m_all[t] - m_next);
      l_run[t] = l_run[t] * alpha + psum[t] * __builtin_amdgcn_exp2f(m_new[t] - m_next);
      m_all[t] = m_next;
#pragma unroll
      for (int d = 0; d < DTW; ++d) o[t][d] *= alpha;
    }
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      if (kb + w * KW >= kv_len) break;             // (bytes that nobody wrote)
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        const float f = __builtin_amdgcn_exp2f(mw[t][w] - m_all[t]);
#pragma unroll
        for (int d = 0; d < DTW; ++d) o[t][d] += times(t, d, w, float4v{0, 0, 0, 0}) * f;
      }
    }
  }

  // ---- the rows' sums ----
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    float l = l_run[t];
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (g == 0) s_l[(wave * RT + t) * 16 + rr] = l;
  }
  __syncthreads();
  const int bh = b * gridDim.y + hkv;
  const bool single = a.splits == 1;
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    float lt = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) lt += s_l[(w * RT + t) * 16 + rr];
    if (16 * t + rr >= rows) continue;
    if (single) {
      const float inv = lt > 0.0f ? 1.0f / lt : 0.0f;
#pragma unroll
      for (int d = 0; d < DTW; ++d) {
        half4 hv;
#pragma unroll
        for (int q = 0; q < 4; ++q) hv[q] = (_Float16)(o[t][d][q] * inv);
        *(half4*)(a.out + out_at(b * q_total + token(row[t]), head(row[t]) * D + wave * CH + 16 * d + 4 * g, a.Hq * D, a.frag_mt)) = hv;
      }
    } else {
      const __amdgpu_buffer_rsrc_t parts = partials_of<D, RT>(a, bh);
      auto leave = [&](auto scope) {
#pragma unroll
        for (int d = 0; d < DTW; ++d) put_partial<D, RT, decltype(scope)::value>(parts, split, 16 * t + rr, wave * CH + 16 * d + 4 * g, o[t][d]);
        if (wave == 0 && g == 0) put_partial<D, RT, decltype(scope)::value>(parts, split, 16 * t + rr, D, float2{m_all[t], lt});
      };
      if (a.defer_combine) leave(std::integral_constant<int, 0>{});
      else leave(std::integral_constant<int, AGENT_SCOPE>{});
    }
  }
  if (single || a.defer_combine) return;
  combine_splits<D, RT, NW * 64>(a, bh, hkv * G, b * q_total + (MULTI ? a.q_off : 0), rows, G, (int*)s_m);
}

}  // namespace bigdl
