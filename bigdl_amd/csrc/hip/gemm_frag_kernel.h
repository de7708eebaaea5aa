// Dequant-fused product on x in fragment order for gfx950:  y[M,N] = f(x[M,K] . dequant(W)[N,K]^T), 33 to 512 rows, and up to
// FRAG_MAX_ROWS where K is no multiple of 128: short prompts, wide decode batches, module calls.
//
// What bounds products of so many rows is neither the weights (28 MB for Llama-2-7B's qkv, 6 us) nor the matrix cores alone (64 rows: 5 us).
// In rows it is x, which every workgroup pulls through its CU's L1: rates per CU, x in L2, 70 GB/s for requests of 8 rows x 128 bytes, 29
// for MFMA fragments straight from rows (16 rows x 64 bytes), 105 - 120 for whole contiguous KiB.  In the last form what remains is mostly
// instructions: without any memory access 73 - 87 % of the time (77 x 14336 pair 30.4 of 35.1 us, 203 x 4672 x 4544 19.6 of 26).  Hence:
//  * x comes in fragment order: [k / 32][row / 16][lane][8 halves], 1 KiB that a wavefront requests at once and multiplies as it
//    arrives -- no LDS, no swizzle, no barrier in the loop.  A pass of 3.5 us puts rows into that order (frag_pack_kernel; for
//    bf16 rows in place of their conversion), unless the producer of x writes it so.
//  * One workgroup a CU owns MT x NS tiles of 16 x 16 and all of K (or a split of it); its wavefronts take the k-tiles in turn, so
//    every byte of x and of the weights reaches the CU once, and the sums meet in LDS at the end.  MT follows the row count, so
//    that 77 rows are one block of 80 and not two of 64; planner in gemm_frag.hip.
//  * Eight wavefronts where the tile leaves 256 registers enough, else four with 512.
//  * The weight is the A operand: a lane holds four neighbouring columns of a row, stored together.
//  * Row blocks of one weight panel run on the same XCD, one after the other, and load weights through its L2 (non-temporal loads,
//    which it does not keep, are for the only row block: 203 rows, three blocks: 24.0 -> 22.4 us; 64 rows, one: 16.0 <- 15.6).
// One MI355X, us, kernels of before (few-row / tile kernel) -> this one, without the pass over x: gate / up pair of 14336 x 4096,
// 77 rows, asym_int4 67.6 -> 32; 4672 x 4544, 203 rows, sym_int8 38.7 -> 22; sym_int4 4096 x 4096 at 64 / 256 / 400 rows 12.4 -> 9.6,
// 23.1 -> 14.3, 31.3 -> 20.1; 4096 x 11008 at 256 rows 39.2 -> 29.1.  Depth of look-ahead, 4 / 8 / 16
// wavefronts, the order of arithmetic and loads and decoding between the products of the fragment before change it by 3 %.
#pragma once
#include "gemm_rows_kernel.h"

namespace bigdl {

// out_type of an output in fragment order, fp16: x of the next product
constexpr int OUT_FRAG = 3;

struct FragArgs {
  const _Float16* xp;     // [KT * 4][mt_all][64 lanes][8]: see frag_pack_kernel
  const void* w;          // T16 [N, K]
  const void* w2;         // pair form: second weight, same shape and format
  void* out;              // [M, ldo]
  float* partial;         // [splitk][M][N] (x 2 in the pair form) fp32 when splitk > 1
  const void* bias;
  const void* bias2;
  const void* residual;
  int M, N, K, mt_all, ldo, act, out_type;
  int splitk, kt_per_split;
  int vec;                // rows of out / residual take 4-column accesses
};

// registers of a wavefront: accumulators, XD steps of x, WD k-tiles of weights, and addresses and the decoding (for the formats with
// high bits measured from the compiler's allocation).  256 with eight wavefronts; with four 512, of which 448 are planned for: not
// every value can sit in the accumulation half.  A tiling that spills costs: 6 x 4 tiles of fp6, 16384 x 4096, on eight wavefronts
// with 52 registers in scratch 40.2 us, on four 30.1; 3 x 6 and 5 x 8 of fp6 37.8 -> 35.8 and 60.4 -> 50.8; 4 x 6 of sym_int5 32.8 -> 30.9.
constexpr int frag_tile_vgprs(int qt) { return lo_bits_of(qt) + hi_bits_of(qt) + 2 + (has_min_of(qt) ? 2 : 0); }
constexpr int frag_decode_vgprs(int qt, int ns) { return qt == Q_FP6 ? 16 + 10 * ns : qt == Q_SYM_INT5 ? 10 + 6 * ns : 40; }
constexpr int frag_need(int qt, int mt, int ns, int xd, int wd) {
  return 4 * mt * ns + 4 * mt * xd + wd * ns * frag_tile_vgprs(qt) + frag_decode_vgprs(qt, ns);
}
constexpr int frag_nw(int qt, int mt, int ns) { return frag_need(qt, mt, ns, 2, 2) <= 256 ? 8 : 4; }
constexpr int frag_xd(int qt, int mt, int ns) { return frag_need(qt, mt, ns, 4, 2) <= (frag_nw(qt, mt, ns) == 8 ? 256 : 448) ? 4 : 2; }
// partial sums of a wavefront are mt * ns KiB; as many wavefronts park theirs at once as fit
constexpr int frag_red(int mt, int ns, int nw) { return mt * ns * nw <= 144 ? nw : nw / 2; }
constexpr int frag_lds(int mt, int ns, int nw) { return frag_red(mt, ns, nw) * mt * ns * 1024; }

template <int QT, int MT, int NS, int NW, int XD, int AUX>
__global__ __launch_bounds__(NW * 64, NW / 4) void gemm_frag_kernel(FragArgs a) {
  constexpr int WD = 2;                              // k-tiles of weights on their way or in use
  constexpr int NR = frag_red(MT, NS, NW);
  constexpr int NA = (NS + 1) / 2;                   // weight tiles addressed through the first set of planes
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* red = (float*)smem;                         // [NR][NS * MT][64][4]

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int KT = (a.K + 127) >> 7;
  const int ntiles = (a.N + 15) >> 4;
  const bool pair = a.w2 != nullptr;
  const int NO = pair ? NS / 2 : NS;                 // column tiles of the output a workgroup owns
  const int nblocks = (ntiles + NO - 1) / NO, mblocks = (a.mt_all + MT - 1) / MT;
  int tid;                                           // consecutive ids go to one XCD
  {
    const int nblk = gridDim.x, b = blockIdx.x, q = nblk >> 3, rr = nblk & 7, xcd = b & 7;
    tid = (xcd < rr ? xcd * (q + 1) : rr * (q + 1) + (xcd - rr) * q) + (b >> 3);
  }
  const int mb = tid % mblocks, rest = tid / mblocks;
  const int nb = rest % nblocks, sp = rest / nblocks;
  const int kt0 = sp * a.kt_per_split, kt1 = min(KT, kt0 + a.kt_per_split);

  // planes of the first NA weight tiles and of the others (pair form: the same columns of w2)
  const int nb0 = nb * NO, nb1 = pair ? nb0 : min(nb0 + NA, ntiles - 1);
  RowsPlanes<QT> pl, ph;
  pl.init(t16_planes(a.w, QT, a.N, a.K), (int64_t)nb0 * KT, min(NA, ntiles - nb0) * KT);
  ph.init(t16_planes(pair ? a.w2 : a.w, QT, a.N, a.K), (int64_t)nb1 * KT, min(NA, ntiles - nb1) * KT);
  int tbase[NS];
#pragma unroll
  for (int n = 0; n < NS; ++n) tbase[n] = n < NA ? min(n, ntiles - 1 - nb0) * KT : min(n - NA, ntiles - 1 - nb1) * KT;

  // this wavefront's k-tiles: kt0 + wave, + NW, ...  Past them the lane offsets point behind the buffers (zeros, no memory access)
  const int nk = kt1 - kt0 > wave ? (kt1 - kt0 - wave + NW - 1) / NW : 0;
  auto kmap = [&](int i) { return min(kt0 + wave + i * NW, KT - 1); };
  auto past = [&](int i) { return i < nk ? 0u : ROWS_OUT; };

  Tile<QT> tt[WD][NS];
  auto fetch_w = [&](Tile<QT> (&t)[NS], int i) {
    const int kt = kmap(i);
    const uint32_t out = past(i);
#pragma unroll
    for (int n = 0; n < NS; ++n) {
      if (n < NA) pl.template load<AUX>(t[n], tbase[n] + kt, lane, out);
      else ph.template load<AUX>(t[n], tbase[n] + kt, lane, out);
    }
  };
  const int mt0 = mb * MT;
  const rows_rsrc xb = rows_buffer(a.xp, KT * 4 * a.mt_all * 1024);
  int xtile[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) xtile[j] = min(mt0 + j, a.mt_all - 1) * 1024;
  half8 xr[XD][MT];                                  // steps of x on their way or in use
  auto fetch_x = [&](half8 (&x)[MT], int i, int s) {       // step s (may run past 3: a later k-tile) of k-tile i
    const int ii = i + (s >> 2);
    const int row = (kmap(ii) * 4 + (s & 3)) * a.mt_all * 1024;
    const uint32_t at = lane * 16 + past(ii);
#pragma unroll
    for (int j = 0; j < MT; ++j) x[j] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(xb, at, row + xtile[j], 0));
  };

  // what the first step needs, then the rest of the look-ahead
  fetch_x(xr[0], 0, 0);
  rows_issued();
  fetch_w(tt[0], 0);
  rows_issued();
#pragma unroll
  for (int s = 1; s < XD; ++s) {
    fetch_x(xr[s], 0, s);
    rows_issued();
  }
#pragma unroll
  for (int d = 1; d < WD; ++d) {
    fetch_w(tt[d], d);
    rows_issued();
  }

  float4v acc[NS][MT];
#pragma unroll
  for (int n = 0; n < NS; ++n)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[n][j] = float4v{0, 0, 0, 0};

  for (int i = 0; i < nk; i += WD) {
#pragma unroll
    for (int d = 0; d < WD; ++d) {
      // (only arithmetic stands under a condition: a load there would cost the counts of the waits)
      const bool live = d == 0 || i + d < nk;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (live) {
#pragma unroll
          for (int n = 0; n < NS; ++n) {
            const half8 wf = rows_scaled<QT>(tt[d][n], rows_fragment<QT>(tt[d][n], s, g), s);
#pragma unroll
            for (int j = 0; j < MT; ++j) acc[n][j] = mfma16(wf, xr[(4 * d + s) % XD][j], acc[n][j]);     // D[n = 4 g + q][m = r]
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch_x(xr[(4 * d + s) % XD], i + d, s + XD);
        if (s == 3) fetch_w(tt[d], i + d + WD);
        rows_issued();
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // ---- sum over the wavefronts' k-tiles through LDS
  auto park = [&](int at) {
#pragma unroll
    for (int n = 0; n < NS; ++n)
#pragma unroll
      for (int j = 0; j < MT; ++j) *(float4v*)(red + ((at * NS * MT + n * MT + j) * 64 + lane) * 4) = acc[n][j];
  };
  if constexpr (NR < NW) {
    if (wave >= NR) park(wave - NR);
    __syncthreads();
    if (wave < NR) {
#pragma unroll
      for (int n = 0; n < NS; ++n)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[n][j] += *(const float4v*)(red + ((wave * NS * MT + n * MT + j) * 64 + lane) * 4);
      park(wave);        // (the slot this wavefront alone has just read)
    }
  } else {
    park(wave);
  }
  __syncthreads();

  const bool partial_out = a.splitk > 1;
  const int items = NO * MT, second = NA * MT;
  for (int it = wave; it < items; it += NW) {
    const int n = it / MT, j = it % MT;
    float4v v = {0, 0, 0, 0}, u = {0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < NR; ++w) {
      v += *(const float4v*)(red + ((w * NS * MT + it) * 64 + lane) * 4);
      if (pair) u += *(const float4v*)(red + ((w * NS * MT + second + it) * 64 + lane) * 4);
    }
    const int nt = !pair && n >= NA ? nb1 + n - NA : nb0 + n;
    if (nt >= ntiles || nb0 + n >= ntiles) continue;
    const int col = nt * 16 + 4 * g, m = (mt0 + j) * 16 + r;
    if (m >= a.M || col >= a.N) continue;
    const int cols = min(4, a.N - col);
    if (partial_out) {
      const int64_t at = ((int64_t)sp * a.M + m) * a.N + col, at2 = ((int64_t)(a.splitk + sp) * a.M + m) * a.N + col;
      if ((a.N & 3) == 0) {
        *(float4v*)(a.partial + at) = v;
        if (pair) *(float4v*)(a.partial + at2) = u;
        continue;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q >= cols) break;
        a.partial[at + q] = v[q];
        if (pair) a.partial[at2 + q] = u[q];
      }
      continue;
    }
    // Four elements to a branch, and the usual gate by a reciprocal: asked for each element, what the call is like took most of an item's
    // time (one wavefront a SIMD issues an instruction in 5 cycles).  us, before -> now: head 64 x 32000 x 4096 sym_int4 31.4 -> 28.9, pair of
    // 11008 x 4096 23.1 -> 22.4, 203 x 4672 x 4544 sym_int8 25.9 -> 25.1, 77 x 6144 x 4096 asym_int4 13.4 -> 13.0
    float y[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) y[q] = v[q];
    if (a.bias != nullptr) {
#pragma unroll
      for (int q = 0; q < 4; ++q) y[q] += (float)((const _Float16*)a.bias)[min(col + q, a.N - 1)];
    }
    if (a.act == ACT_SILU) {
#pragma unroll
      for (int q = 0; q < 4; ++q) y[q] = silu_rcp(y[q]);
    } else if (a.act != ACT_NONE) {
#pragma unroll
      for (int q = 0; q < 4; ++q) y[q] = act_apply(a.act, y[q]);
    }
    if (pair) {
      if (a.bias2 != nullptr) {
#pragma unroll
        for (int q = 0; q < 4; ++q) u[q] += (float)((const _Float16*)a.bias2)[min(col + q, a.N - 1)];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) y[q] *= u[q];
    }
    if (a.out_type == OUT_FRAG) {
      *(half4*)((_Float16*)a.out + frag_at(m, col, a.mt_all)) = half4{(_Float16)y[0], (_Float16)y[1], (_Float16)y[2], (_Float16)y[3]};
      continue;
    }
    const int64_t oi = (int64_t)m * a.ldo + col;
    if (a.vec && a.out_type != OUT_F32) {
      if (a.out_type == OUT_F16) {
        if (a.residual) {
          const half4 h = *(const half4*)((const _Float16*)a.residual + oi);
#pragma unroll
          for (int q = 0; q < 4; ++q) y[q] += (float)h[q];
        }
        *(half4*)((_Float16*)a.out + oi) = half4{(_Float16)y[0], (_Float16)y[1], (_Float16)y[2], (_Float16)y[3]};
      } else {
        if (a.residual) {
#pragma unroll
          for (int q = 0; q < 4; ++q) y[q] += load_out<OUT_BF16>(a.residual, oi + q);
        }
        uint2v p;
        p.x = (uint32_t)f32_to_bf16_bits(y[0]) | ((uint32_t)f32_to_bf16_bits(y[1]) << 16);
        p.y = (uint32_t)f32_to_bf16_bits(y[2]) | ((uint32_t)f32_to_bf16_bits(y[3]) << 16);
        *(uint2v*)((uint16_t*)a.out + oi) = p;
      }
    } else if (a.vec) {
      float4v f = {y[0], y[1], y[2], y[3]};
      if (a.residual) f += *(const float4v*)((const float*)a.residual + oi);
      *(float4v*)((float*)a.out + oi) = f;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q >= cols) break;
        float z = y[q];
        if (a.out_type == OUT_F16) {
          if (a.residual) z += load_out<OUT_F16>(a.residual, oi + q);
          store_out<OUT_F16>(a.out, oi + q, z);
        } else if (a.out_type == OUT_BF16) {
          if (a.residual) z += load_out<OUT_BF16>(a.residual, oi + q);
          store_out<OUT_BF16>(a.out, oi + q, z);
        } else {
          if (a.residual) z += load_out<OUT_F32>(a.residual, oi + q);
          store_out<OUT_F32>(a.out, oi + q, z);
        }
      }
    }
  }
}

template <int QT, int MT, int NS>
static int gemm_frag_launch_t(const FragArgs& a, hipStream_t st) {
  constexpr int NW = frag_nw(QT, MT, NS), XD = frag_xd(QT, MT, NS);
  constexpr int lds = frag_lds(MT, NS, NW);
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  if (a.w2 != nullptr && (NS & 1)) return -4;
  const int no = a.w2 != nullptr ? NS / 2 : NS;
  const int nblocks = ((a.N + 15) / 16 + no - 1) / no, mblocks = (a.mt_all + MT - 1) / MT;
  auto k = mblocks == 1 ? gemm_frag_kernel<QT, MT, NS, NW, XD, ROWS_NT> : gemm_frag_kernel<QT, MT, NS, NW, XD, 0>;
  if (!gemv_allow_lds((const void*)k, lds)) return -101;
  hipLaunchKernelGGL(k, dim3(nblocks * mblocks * a.splitk), dim3(NW * 64), lds, st, a);
  return HIP_CHECK_LAUNCH();
}

// the tilings that exist (the planner in gemm_frag.hip chooses among them)
// (without five that the planner would choose for 2 % of random shapes, all within 3 % of another)
constexpr bool frag_has(int mt, int ns) {
  return mt == 3 ? ns == 2 || ns == 3 || ns == 4 || ns == 6 : mt == 4 ? ns == 2 || ns == 3 || ns == 4 || ns == 6 || ns == 8
       : mt == 5 ? ns == 3 || ns == 4 || ns == 6 || ns == 8 : mt == 6 ? ns == 2 || ns == 4 || ns == 6 : (mt == 7 || mt == 8) && (ns == 3 || ns == 4);
}
template <int QT, int MT>
static int gemm_frag_launch_mt(const FragArgs& a, int ns, hipStream_t st) {
  if constexpr (frag_has(MT, 2)) if (ns == 2) return gemm_frag_launch_t<QT, MT, 2>(a, st);
  if constexpr (frag_has(MT, 3)) if (ns == 3) return gemm_frag_launch_t<QT, MT, 3>(a, st);
  if constexpr (frag_has(MT, 4)) if (ns == 4) return gemm_frag_launch_t<QT, MT, 4>(a, st);
  if constexpr (frag_has(MT, 6)) if (ns == 6) return gemm_frag_launch_t<QT, MT, 6>(a, st);
  if constexpr (frag_has(MT, 8)) if (ns == 8) return gemm_frag_launch_t<QT, MT, 8>(a, st);
  return -4;
}
template <int QT>
static int gemm_frag_launch_qt(const FragArgs& a, int mt, int ns, hipStream_t st) {
  switch (mt) {
    case 3: return gemm_frag_launch_mt<QT, 3>(a, ns, st);
    case 4: return gemm_frag_launch_mt<QT, 4>(a, ns, st);
    case 5: return gemm_frag_launch_mt<QT, 5>(a, ns, st);
    case 6: return gemm_frag_launch_mt<QT, 6>(a, ns, st);
    case 7: return gemm_frag_launch_mt<QT, 7>(a, ns, st);
    case 8: return gemm_frag_launch_mt<QT, 8>(a, ns, st);
    default: return -4;
  }
}

}  // namespace bigdl
