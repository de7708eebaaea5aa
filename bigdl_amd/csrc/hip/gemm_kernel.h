// Dequant-fused MFMA GEMM for mid-size row counts on gfx950:  y[M,N] = f(x[M,K] . dequant(W)[N,K]^T) for the products of
// 33 - 256 rows where the few-row kernel is not expected to be ahead (dense_cost in gemm_lowbit.hip), for more rows where the
// prompt kernel does not take K, and its grouped (mixture-of-experts) form where every 64/128-row block of x belongs to one expert.
//
// Takes the place of the reference's closed xe_linear.forward_new for prefill-sized inputs / xe_batch.batch_forward
// (call sites python/llm/src/ipex_llm/transformers/low_bit_linear.py:657-668) and of the per-expert Python loop of
// python/llm/src/ipex_llm/transformers/models/qwen2_moe.py:400-445.
//
// Why a second kernel next to the skinny one (gemv_kernel.h): above 64 rows x no longer fits next to the K-split
// partials in LDS and re-reading it per 16-row weight tile would make the kernel L2 bound.  Here a workgroup owns
// a BM x 128 output tile:
//  * x tile [BM][128 k] goes global -> VGPR -> LDS in full 256-byte rows, double buffered, XOR-swizzled per 16-byte
//    slot (slot ^= row & 15) so that the ds_read_b128 of an A fragment is bank-conflict free;
//  * the T16 weight layout already is the MFMA B-operand order, so each of the 4 wavefronts streams its own two
//    16-row weight tiles HBM -> VGPR (no LDS, no redundancy inside the workgroup), dequantises them with the same
//    register bit tricks as the skinny kernel, folds the block scale in as a packed fp16 multiply, and reuses
//    every B fragment for all BM/16 row tiles (8 MFMAs per dequantised fragment at BM = 128);
//  * v_mfma_f32_16x16x32_f16 accumulates over all of K in fp32 registers; one barrier per 128-deep k tile;
//  * small grids split K across workgroups (fp32 slabs + a reduce/epilogue kernel) to cover the 256 CUs.
#pragma once
#include "gemv_kernel.h"

// Hooks of benchmark/gemm_probe.hip (all 0 in the library build):
// GEMM_STAMP = 1: every wavefront writes 100 MHz wall-clock stamps to g_gemm_stamps ([workgroup][wavefront][32]:
// 0 entry, 1 first x tile staged, 2 + i after k iteration i, 31 exit).
// GEMM_ABL (results are wrong): 1 = no MFMA, 2 = no dequantization, 4 = no LDS fragment reads, 8 = no x loads in the
// k loop, 16 = no weight loads in the k loop, 32 = no epilogue (one store per wavefront),
// 64 = no weight loads before the loop, 128 = no x requests before the loop (loader form).
#ifndef GEMM_STAMP
#define GEMM_STAMP 0
#endif
#ifndef GEMM_ABL
#define GEMM_ABL 0
#endif
#if GEMM_STAMP
__device__ unsigned long long* g_gemm_stamps = nullptr;      // [2048 workgroups][16][32], set by the probe
#define GEMM_STAMP_AT(i)                                                                                        \
  do {                                                                                                          \
    __builtin_amdgcn_sched_barrier(0);                                                                          \
    const unsigned long long t_ = __builtin_amdgcn_s_memrealtime();                                             \
    if (lane == 0 && (i) < 32 && g_gemm_stamps != nullptr && blockIdx.x + gridDim.x * blockIdx.y < 2048)        \
      g_gemm_stamps[((size_t)(blockIdx.x + gridDim.x * blockIdx.y) * 16 + wave) * 32 + (i)] = t_;               \
    __builtin_amdgcn_sched_barrier(0);                                                                          \
  } while (0)
#else
#define GEMM_STAMP_AT(i)
#endif
// look-ahead of the weight stream in k-tiles (even)
#ifndef GEMM_DEPTH
#define GEMM_DEPTH 4
#endif

namespace bigdl {

// s_waitcnt immediate that waits for all but the n youngest vector-memory operations only (gfx9 encoding: vmcnt in bits
// [3:0] and [15:14], expcnt [6:4] and lgkmcnt [11:8] left at their maxima)
constexpr int gemm_waitcnt_vm(int n) { return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4) | (0xF << 8); }

struct GemmArgs {
  const _Float16* x;      // [*, ldx]
  const void* w;          // T16 buffer ([N, K], or experts stacked by rows in grouped mode)
  void* out;              // [Mtot, ldo]
  float* partial;         // [splitk][Mtot][N] fp32 when splitk > 1
  const void* bias;       // [N] fp16 or null (dense mode)
  const void* residual;   // [Mtot, ldo] or null
  int M, N, K, ldx, ldo, act, out_type;
  int splitk, kt_per_split;
  // grouped mode (blk_expert != null): m-block b covers sorted rows [blk_row0[b], +blk_rows[b]) of expert
  // blk_expert[b] (< 0: unused block); x row of sorted row i is x_rows[i] (null: i); out row is i
  const int* blk_expert;
  const int* blk_row0;
  const int* blk_rows;
  const int* x_rows;
  const float* row_scale;  // [Mtot] multiplied into the output rows (routing weights), or null
  int n_total;             // rows of the stacked weight buffer
  // RMSNorm folded into the product: x is multiplied by gamma (+ gamma_offset) while it is staged and the result rows by
  // rsqrt(row_ssq[m] / K + eps) before bias / activation; row_ssq holds the sums of squares of the rows of x (written by
  // the reduce kernel of the product that produced x: ssq_out)
  const _Float16* gamma;
  float gamma_offset, eps;
  const float* row_ssq;
  float* ssq_out;          // [Mtot], accumulated (atomics) by the reduce kernel from the rows it writes; zeroed by the caller
  // pair form (gate / up): blockIdx.z = 1 multiplies by w2 and writes its partials `pair_stride` floats further on; the
  // reduce kernel then writes act(first + bias) * (second + bias2)
  const void* w2;
  const void* bias2;
  int64_t pair_stride;
  int force_partial;       // write fp32 partials even with one K split (pair form, ssq_out)
};

// MT = 16-row tiles of x per workgroup, NT = 16-column weight tiles per wavefront (4 wavefronts side by side)
// NORM: x is multiplied by gamma while it is staged (compile-time, so that the gamma load is unconditional: a load
// under a run-time condition costs the counted waits of the whole loop)
// NW = wavefronts per workgroup, side by side along N.  8 wavefronts of one weight tile each (NT = 1) cover the same 128
// columns as 4 of two, in under 128 VGPRs: four wavefronts per SIMD instead of two hide the load -> dequantize -> MFMA ->
// barrier chain of a k-tile behind each other, which is what the few-row shapes of batched decode lack.
// LW: one more wavefront per workgroup does nothing but bring the x tiles in (global -> LDS directly, three stages), so
// that the compute wavefronts request and wait for weight tiles only (a wavefront's vector loads retire in order: one
// that requests both operands takes delivery of an x tile only after the older weight requests).  Measured on the
// Llama-2-7B shapes at 64 rows: 117 -> 109 us for the four products of a layer.  Needs K % 128 == 0, no folded norm.
// Where the time of these launches goes at 64 rows (qkv, 288 workgroups of 11 k-tiles, 22 us): 4.5 us for the kernel
// with an empty loop and no loads, 4 - 8 us until the first four weight tiles of every wavefront have arrived (the
// 128-byte scale requests cost more than the 1 KiB code requests next to them), 2.5 us for the eleven k-tiles, 6.5 us
// for the fp32 partials (9.4 MB) -- then 4.8 us of reduce kernel.  Eight wavefronts of one tile each, deeper weight
// look-ahead, more K splits, rotated k order, tile-major slabs and one 512-byte scale request per four k-tiles (with
// ds_bpermute redistribution) were all measured within 5 % or slower.
template <int QT, int MT, int NT, bool NORM = false, int NW = 4, bool LW = false>
__global__ __launch_bounds__((NW + (LW ? 1 : 0)) * 64, 2) void gemm_t16_kernel(GemmArgs a) {
  static_assert(!(LW && NORM), "the loader wavefront copies x as it is");
  constexpr int NSTAGE = LW ? 3 : 2;
  constexpr int BM = MT * 16;
  constexpr int BN = NW * NT * 16;
  constexpr int RP = NW * 4;       // x rows staged per pass (16 threads per 256-byte row)
  constexpr int NP = BM / RP;      // passes per x tile
  static_assert(BM % RP == 0 && RP % 16 == 0, "whole passes; the swizzle of a row is that of its pass-0 row");
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* As = smem;                                               // [NSTAGE][BM][256 B]

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  GEMM_STAMP_AT(0);
  const int r = lane & 15, g = lane >> 4;
  const int KT = (a.K + 127) >> 7;
  const int nblocks = (a.N + BN - 1) / BN;
  const int nb = blockIdx.x % nblocks, sp = blockIdx.x / nblocks;
  const int mb = blockIdx.y;

  int row0 = mb * BM, rows = min(BM, a.M - row0);
  int64_t wt = 0;
  int n_planes = a.N;
  if (a.blk_expert != nullptr) {
    const int e = a.blk_expert[mb];
    if (e < 0) return;
    row0 = a.blk_row0[mb];
    rows = a.blk_rows[mb];
    wt = (int64_t)e * (a.N >> 4);
    n_planes = a.n_total;
  }
  const int kt0 = sp * a.kt_per_split, kt1 = min(KT, kt0 + a.kt_per_split);
  const bool second = a.w2 != nullptr && blockIdx.z == 1;
  const T16Planes pl = t16_planes(second ? a.w2 : a.w, QT, n_planes, a.K);

  // this wavefront's weight tile rows (clamped: a tile past N is loaded from the last valid one and never stored)
  const int ntiles = (a.N + 15) >> 4;
  int nt_idx[NT];
  int64_t tbase[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    nt_idx[n] = nb * (BN / 16) + wave * NT + n;
    tbase[n] = (wt + min(nt_idx[n], ntiles - 1)) * KT;
  }

  const int klast = max(kt1 - 1, kt0);
  auto kmap = [&](int k) { return min(k, klast); };     // tiles past the end: the last one again (never used)
  if constexpr (LW) {
    if (wave == NW) {
      // ---- loader wavefront.  One instruction moves 4 rows of a tile (64 lanes x 16 bytes); lane i brings what belongs
      // in slot i % 16 of row i / 16, i.e. k chunk (i % 16) ^ (row % 16) (the swizzle of the fragment reads, applied to
      // the source address because the LDS side of the instruction is lane-linear).  Rows past the block re-read its last
      // row (their products are never stored).  Tile i + 2 is requested into stage (i + 2) % 3 -- last read in iteration
      // i - 1, which every wavefront has left -- then the wait leaves exactly those requests open: tile i + 1 is in LDS
      // before the barrier that ends iteration i.
      constexpr int NLD = BM / 4;
      uint32_t xo[NLD];
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        const int row = min(4 * i + (lane >> 4), max(rows - 1, 0));
        const int64_t xr = a.x_rows != nullptr ? a.x_rows[row0 + row] : row0 + row;
        xo[i] = (uint32_t)(xr * a.ldx) + (uint32_t)((((lane & 15) ^ (4 * i + (lane >> 4))) & 15) << 3);
      }
      auto request = [&](int kt, int stage) {
        const _Float16* src = a.x + (int64_t)kt * 128;
        char* dst = As + stage * BM * 256;
#pragma unroll
        for (int i = 0; i < NLD; ++i)
          __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) const void*)(src + xo[i]),
                                           (__attribute__((address_space(3))) void*)(dst + i * 1024), 16, 0, 0);
      };
      // (bare s_barrier: __syncthreads() carries a fence that makes the compiler wait for EVERY outstanding LDS-bound
      // load, the tile just requested included)
      auto tile_ready_barrier = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(gemm_waitcnt_vm(NLD));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      };
      if constexpr (!(GEMM_ABL & 128)) {
        request(kmap(kt0), 0);
        request(kmap(kt0 + 1), 1);
      }
      tile_ready_barrier();
      int st = 2;
      for (int k = kt0; k < kt1; ++k) {
        if constexpr (!(GEMM_ABL & 8)) request(kmap(k + 2), st);
        st = st == 2 ? 0 : st + 1;
        tile_ready_barrier();
      }
      return;
    }
  }

  // x staging: thread t moves 16 bytes of row (16 p + t / 16), slot t % 16, for p = 0 .. MT-1
  const int srow = threadIdx.x >> 4, sslot = threadIdx.x & 15;
  // element offsets into x (32 bits: the host checks rows * ldx < 2^31).  Rows past the block read the block's last
  // row and are zeroed afterwards: every load below is unconditional, from a clamped address.  A load under a
  // condition leaves the compiler without a static count of younger loads in flight, and it then waits for ALL of
  // them (s_waitcnt vmcnt(0)) before the LDS store of the x tile, including the weight tiles just requested four
  // k-tiles ahead, which put a full memory round trip into every k-tile.
  uint32_t xsrc[NP];
  bool xok[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int row = min(RP * p + srow, max(rows - 1, 0));
    xok[p] = RP * p + srow < rows;
    const int64_t xr = a.x_rows != nullptr ? a.x_rows[row0 + row] : row0 + row;
    xsrc[p] = (uint32_t)(xr * a.ldx);
  }
  const int swz = ((sslot ^ srow) & 15) << 4;   // (RP p + srow) & 15 == srow & 15
  // x tiles travel global -> registers -> LDS two k-tiles ahead of their use: tile t sits in register set t & 1
  // from iteration t - 2 and is written to LDS stage t & 1 at the end of iteration t - 1
  uint4v areg[2][NP];
  uint4v greg[2];                              // NORM: gamma of the k slot of the tile in the same register set
  auto gload_a = [&](uint4v (&dst)[NP], uint4v& gdst, int kt) {
    const int k = kt * 128 + sslot * 8;
    const int kc = min(k, a.K - 8);           // K % 32 == 0: the clamped address is a whole valid 16-byte slot
    const bool kin = k < a.K;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      // zeroing by mask, not by a select the compiler could turn back into a branch around the load
      const uint32_t keep = 0u - (uint32_t)(kin & xok[p]);
      const uint4v v = *(const uint4v*)(a.x + xsrc[p] + kc);
      dst[p] = v & uint4v{keep, keep, keep, keep};
    }
    // gamma of the tile's k slot travels with the tile and is applied when the tile is written to LDS (using it here
    // would make this the point where the x loads are waited for)
    if constexpr (NORM) gdst = *(const uint4v*)(a.gamma + kc);
  };
  auto store_a = [&](uint4v (&src)[NP], const uint4v& gsrc, int stage) {
    char* base = As + stage * BM * 256 + srow * 256 + swz;
    if constexpr (NORM) {
      const half8 g8 = __builtin_bit_cast(half8, gsrc) + (_Float16)a.gamma_offset;
#pragma unroll
      for (int p = 0; p < NP; ++p) *(half8*)(base + p * RP * 256) = __builtin_bit_cast(half8, src[p]) * g8;
    } else {
#pragma unroll
      for (int p = 0; p < NP; ++p) *(uint4v*)(base + p * RP * 256) = src[p];
    }
  };

  float4v acc[MT][NT];
#pragma unroll
  for (int j = 0; j < MT; ++j)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[j][n] = float4v{0, 0, 0, 0};

  // weight tiles: a ring of DEPTH k-tiles per wavefront in flight (HBM latency under load is several k-tiles of
  // MFMA work at small M; one tile of look-ahead left the MFMA pipe waiting on vmcnt)
  constexpr int DEPTH = GEMM_DEPTH;
  static_assert(DEPTH % 2 == 0, "the x stage index is taken from the unrolled position");
  Tile<QT> tt[DEPTH][NT];
  auto fetch_b = [&](Tile<QT> (&t)[NT], int kt) {
#pragma unroll
    for (int n = 0; n < NT; ++n) load_tile<QT>(t[n], pl, tbase[n] + kt, lane);
  };
  auto compute = [&](Tile<QT> (&t)[NT], int stage) {
    const char* abase = As + stage * BM * 256 + r * 256;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      half8 bf[NT];
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        if constexpr (GEMM_ABL & 2) {
          bf[n] = __builtin_bit_cast(half8, uint4v{t[n].lo0[s], t[n].lo0[(s + 1) & 3], __builtin_bit_cast(uint32_t, half2v{t[n].d[s], t[n].d[s]}), 0x3c003c00u});
          continue;
        }
        const half8 code = decode_step<QT>(t[n], s);
        _Float16 d = t[n].d[s];
        if constexpr (post_scale<QT>() != 1.0f) d = (_Float16)fminf((float)d * post_scale<QT>(), 65504.0f);
        if constexpr (has_min<QT>()) bf[n] = code * d + t[n].m[s];
        else bf[n] = code * d;
      }
      const int aoff = (((4 * s + g) ^ r) & 15) << 4;
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        half8 af;
        if constexpr (GEMM_ABL & 4) af = __builtin_bit_cast(half8, uint4v{(uint32_t)(aoff + j + stage), 0x3c003c00u, 0x3c003c00u, 0x3c003c00u});
        else af = *(const half8*)(abase + j * 16 * 256 + aoff);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          if constexpr (GEMM_ABL & 1) {
            const uint4v x = __builtin_bit_cast(uint4v, af) ^ __builtin_bit_cast(uint4v, bf[n]);
            acc[j][n][0] += __uint_as_float((x[0] ^ x[1] ^ x[2] ^ x[3]) & 0x3f800000u);
          } else {
            acc[j][n] = mfma16(af, bf[n], acc[j][n]);
          }
        }
      }
    }
  };

  // prologue.  Tile indices past the end are clamped to the last tile of the range (a redundant load of data that
  // is already on its way) so that the number of loads per iteration is fixed.
  if constexpr (LW) {
    // ---- compute wavefronts next to a loader: weights only; x tile k sits in stage (k - kt0) % 3
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if constexpr (!(GEMM_ABL & 64)) fetch_b(tt[d], kmap(kt0 + d));
    __syncthreads();
    GEMM_STAMP_AT(1);
    int st = 0;
    for (int kt = kt0; kt < kt1; kt += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        const int k = kt + d;                 // block-uniform
        if (k >= kt1) break;
        compute(tt[d], st);
        st = st == 2 ? 0 : st + 1;
        if constexpr (!(GEMM_ABL & 16)) fetch_b(tt[d], kmap(k + DEPTH));
        __syncthreads();
        GEMM_STAMP_AT(2 + k - kt0);
      }
    }
  } else {
  gload_a(areg[0], greg[0], kmap(kt0));
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) fetch_b(tt[d], kmap(kt0 + d));
  store_a(areg[0], greg[0], 0);
  gload_a(areg[1], greg[1], kmap(kt0 + 1));
  __syncthreads();
  GEMM_STAMP_AT(1);
  for (int kt = kt0; kt < kt1; kt += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int k = kt + d;                 // block-uniform
      if (k >= kt1) break;
      if constexpr (!(GEMM_ABL & 8)) gload_a(areg[d & 1], greg[d & 1], kmap(k + 2));           // (k - kt0) & 1 == d & 1: DEPTH is even
      compute(tt[d], d & 1);
      if constexpr (!(GEMM_ABL & 16)) fetch_b(tt[d], kmap(k + DEPTH));
      if constexpr (!(GEMM_ABL & 8)) store_a(areg[(d + 1) & 1], greg[(d + 1) & 1], (d + 1) & 1);
      __syncthreads();
      GEMM_STAMP_AT(2 + k - kt0);
    }
  }
  }

  // epilogue
  if constexpr (GEMM_ABL & 32) {               // measurement: one store per wavefront instead of the tile
    float v = 0.0f;
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int n = 0; n < NT; ++n) v += acc[j][n][0] + acc[j][n][1] + acc[j][n][2] + acc[j][n][3];
    // (where the workgroup ran: HW_ID and XCC_ID, for the probe's placement count)
    if (lane == 0 && wave == 0) {
      ((uint32_t*)a.partial)[(int64_t)blockIdx.x * 2] = __builtin_amdgcn_s_getreg((31 << 11) | 4) | (v == 12345.0f ? 1u << 31 : 0u);
      ((uint32_t*)a.partial)[(int64_t)blockIdx.x * 2 + 1] = __builtin_amdgcn_s_getreg((31 << 11) | 20);
    }
    return;
  }
  const int64_t mtot = a.M;
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int ncol = nt_idx[n] * 16 + r;
    if (nt_idx[n] >= ntiles || ncol >= a.N) continue;
    float bias = 0.0f;
    const bool partial_out = a.splitk > 1 || a.force_partial;
    if (a.bias != nullptr && !partial_out) bias = (float)((const _Float16*)a.bias)[ncol];
#pragma unroll
    for (int j = 0; j < MT; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int m = 16 * j + 4 * g + q;
        if (m >= rows) continue;
        const int64_t orow = row0 + m;
        float v = acc[j][n][q];
        if (partial_out) {
          a.partial[(second ? a.pair_stride : 0) + ((int64_t)sp * mtot + orow) * a.N + ncol] = v;
          continue;
        }
        if (a.row_ssq != nullptr) v *= rsqrtf(a.row_ssq[orow] / (float)a.K + a.eps);
        v = act_apply(a.act, v + bias);
        if (a.row_scale != nullptr) v *= a.row_scale[orow];
        const int64_t oi = orow * a.ldo + ncol;
        if (a.out_type == OUT_F16) {
          if (a.residual) v += load_out<OUT_F16>(a.residual, oi);
          store_out<OUT_F16>(a.out, oi, v);
        } else if (a.out_type == OUT_BF16) {
          if (a.residual) v += load_out<OUT_BF16>(a.residual, oi);
          store_out<OUT_BF16>(a.out, oi, v);
        } else {
          if (a.residual) v += load_out<OUT_F32>(a.residual, oi);
          store_out<OUT_F32>(a.out, oi, v);
        }
      }
    }
  }
  GEMM_STAMP_AT(31);
}

template <int QT, int MT, int NT, bool NORM = false, int NW = 4, bool LW = false>
static int gemm_launch_mt(const GemmArgs& a, int mblocks, hipStream_t st) {
  constexpr int BM = MT * 16;
  const size_t lds = (LW ? 3 : 2) * BM * 256;
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)gemm_t16_kernel<QT, MT, NT, NORM, NW, LW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return -101;
    attr_set = true;
  }
  const int bn = NW * 16 * NT;
  const int nblocks = (a.N + bn - 1) / bn;
  const dim3 grid(nblocks * a.splitk, mblocks, a.w2 != nullptr ? 2 : 1);
  hipLaunchKernelGGL((gemm_t16_kernel<QT, MT, NT, NORM, NW, LW>), grid, dim3((NW + (LW ? 1 : 0)) * 64), lds, st, a);
  return HIP_CHECK_LAUNCH();
}

// bm: rows per block (64 / 128); bn: columns per block (128).  64-column blocks were measured too (more workgroups
// streaming weights at few rows): slower or equal on every Llama-2-7B projection shape.  Up to 32 rows the dense products
// run on gemm_rows_kernel.h, more where gemm_lowbit.hip expects it to be ahead.
template <int QT>
static int gemm_launch_qt(const GemmArgs& a, int bm, int bn, int mblocks, hipStream_t st) {
  if (bn != 128) return -4;
  if (a.gamma != nullptr) {
    if (bm == 64) return gemm_launch_mt<QT, 4, 2, true>(a, mblocks, st);
    if (bm == 128) return gemm_launch_mt<QT, 8, 2, true>(a, mblocks, st);
    return -4;
  }
  static const int lw = getenv("BIGDL_GEMM_LOADER") ? atoi(getenv("BIGDL_GEMM_LOADER")) : 1;
  if (lw && (a.K & 127) == 0) {
    if (bm == 64) return gemm_launch_mt<QT, 4, 2, false, 4, true>(a, mblocks, st);
  }
  if (bm == 64) return gemm_launch_mt<QT, 4, 2>(a, mblocks, st);
  if (bm == 128) return gemm_launch_mt<QT, 8, 2>(a, mblocks, st);
  return -4;
}

}  // namespace bigdl
