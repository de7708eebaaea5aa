// Dequant-fused MFMA GEMM for prompt-sized row counts (M > 256) on gfx950:  y[M,N] = f(x[M,K] . dequant(W)[N,K]^T).
//
// The prompt-side counterpart of the reference's closed xe_linear.forward_new
// (python/llm/src/ipex_llm/transformers/low_bit_linear.py:657-668): the weights stay in their low-bit T16 tiles in HBM
// and are expanded on the way to the matrix cores, so a prompt pass neither writes nor re-reads an fp16 copy of the
// model and calls no library GEMM.
//
// Structure (one workgroup = 2 x 4 wavefronts = one BM x BN output tile, K walked in 64-deep tiles):
//  * x tile [BM][64 k] goes global -> LDS directly (buffer_load .. lds, 16 bytes per lane), up to two tiles ahead, three buffers.
//    The LDS image is lane-linear as the instruction requires; the bank swizzle (16-byte slot ^= row & 7) is applied
//    to the per-lane SOURCE address and again on the fragment reads.
//  * the weight tile [BN][64 k] is expanded ONCE per workgroup: every wavefront owns a share of the block's 16-row weight
//    tile rows, loads their raw T16 tiles (codes + block scales, 16-byte loads, one whole 128-deep tile per two k tiles)
//    two tiles ahead, expands them with the register bit tricks of the skinny kernels, folds the block scale in as a
//    packed fp16 multiply and writes the fp16 fragments to the other LDS buffer with one 16-byte store per unit.
//  * one instruction stream per wavefront (comments at the loop): behind the MFMAs on an x fragment the next k step's
//    fragment is read into its place, and a share of the expansion and at most one memory request ride between two groups
//    of MFMAs.  Two wavefronts a SIMD fill each other's gaps; one barrier per 64-deep tile.
//  * fragments: both operands are read with ds_read_b128 from 128-byte rows; slot ^= row & 7 makes the four 16-lane
//    groups of the read and the eight 8-lane groups of the expansion's ds_write_b128 conflict free.
//  * the weight fragment is the MFMA's A operand, so a lane holds 4 consecutive output columns of one row; the epilogue
//    stages the wavefront's tile through LDS and stores whole 128-byte row segments; the gate / up pair form combines the
//    two products of a column there (act(g) * u), so neither reaches memory.
//  * the block index is remapped so that the workgroups of one XCD share x and weight panels in its L2.
// What bounds it: power.  8192 x 8192 x 8192 in fp16 runs the library's product at 1.42 GHz (87 % of the MFMA cycles, 1300 - 1350
// TFLOP/s; 2110 with zeros), this kernel at 1.5 - 1.6; the cycles of the 256 x 256 loop are 15 % over the MFMAs'.
// The earlier form ran the two row halves as a ping-pong pair, load and MFMA segments in turn with a barrier behind each (4 a tile) and
// a tile's requests in one burst, behind which every wavefront stood still.  Old -> new, us, weights of 4 layers in turn: sym_int4
// 7680 rows x 14336 x 4096 827 -> 715, 1024 x 4096 x 4096 48.5 -> 43.6, nf4 924 -> 777 and 55.5 -> 50.4, fp6 1041 -> 900 and 63 -> 54.7.
// Measured and dropped: stream-K over 256 x 256 tiles (every CU the same number of k tiles whatever the tile count; the
// 256 KiB fp32 slab per shared tile costs more than the idle CUs it removes: 130 instead of 98 us on the qkv shape), wavefront
// priorities (none / slower), weights expanded by both row halves in registers (no LDS for them, but twice the vector work: int4 3 - 6 %
// ahead of the ping-pong form, nf4 14 - 18 % behind), 32 x 32 x 16 MFMAs (alone 1650 TFLOP/s on normal data, 16 x 16 x 32 1870).
#pragma once
#include "gemm_kernel.h"

namespace bigdl {

typedef __attribute__((address_space(3))) void lds_void_t;

// LDS bytes of the tile buffers: three x + two weight buffers, or the epilogue's staging area (rows padded by 16 bytes)
constexpr int prompt_lds_tiles(int BM, int BN, int NW, int MTW, int NTW) {
  const int a = (3 * BM + 2 * BN) * 128, b = NW * MTW * 16 * (32 * NTW + 16);
  return a > b ? a : b;
}

// s_waitcnt immediates (gfx9 encoding: vmcnt [3:0] + [15:14], expcnt [6:4], lgkmcnt [11:8])
constexpr int waitcnt_vm(int n) { return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4) | (0xF << 8); }
constexpr int waitcnt_vm_lgkm0(int n) { return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4); }

// one expansion unit = the 8 codes per lane of one (16-row weight tile, 32-deep k step) -> the fp16 fragment with the
// block scale (and minimum) folded in.  `s` is the step inside the T16 tile (0 .. 3), static.
template <int QT, int S>
__device__ __forceinline__ half8 unit_expand(const Tile<QT>& t) {
  const half8 code = decode_step<QT>(t, S);
  _Float16 d = t.d[S];
  if constexpr (post_scale<QT>() != 1.0f) d = (_Float16)fminf((float)d * post_scale<QT>(), 65504.0f);
  if constexpr (has_min<QT>()) return code * d + t.m[S];
  return code * d;
}

// (buffer operations: a scalar offset plus a lane constant is the whole address, and their arrival is counted, while a global load to
// LDS makes the compiler wait for everything in flight at the next use of a loaded register)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_of(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0xffffffff, 0x00027000);
}
// 16 bytes per lane from a buffer (lane offset + wavefront offset) to consecutive LDS
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t b, char* lds, uint32_t lane_off, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(b, (lds_void_t*)lds, 16, lane_off, off, 0, 0);
}
// the planes of one row of T16 tiles
struct RowPlanes { __amdgpu_buffer_rsrc_t lo, hi, sc, mn; };
template <int QT>
__device__ __forceinline__ RowPlanes row_planes(const T16Planes& p, int64_t tile) {
  RowPlanes b;
  b.lo = buf_of(p.lo + tile * (lo_bits_of(QT) * 256));
  if constexpr (hi_bits_of(QT) > 0) b.hi = buf_of(p.hi + tile * (hi_bits_of(QT) * 256));
  b.sc = buf_of(p.sc + tile * 64);
  if constexpr (has_min<QT>()) b.mn = buf_of(p.mn + tile * 64);
  return b;
}
// requests of load_raw (vmcnt is counted by them below)
template <int QT>
constexpr int raw_loads() { return lo_bits_of(QT) / 4 + (hi_bits_of(QT) > 0) + 1 + has_min<QT>(); }
template <int QT>
__device__ __forceinline__ void load_raw(Tile<QT>& t, const RowPlanes& p, int tile, int lane) {
  t.lo0 = __builtin_amdgcn_raw_buffer_load_b128(p.lo, lane * 16, tile * (lo_bits_of(QT) * 256), 0);
  if constexpr (lo_bits_of(QT) == 8) t.lo1 = __builtin_amdgcn_raw_buffer_load_b128(p.lo, lane * 16, tile * 2048 + 1024, 0);
  if constexpr (hi_bits_of(QT) == 1) t.hi0 = __builtin_amdgcn_raw_buffer_load_b32(p.hi, lane * 4, tile * 256, 0);
  if constexpr (hi_bits_of(QT) == 2) {
    const uint2v h = __builtin_amdgcn_raw_buffer_load_b64(p.hi, lane * 8, tile * 512, 0);
    t.hi0 = h.x;
    t.hi1 = h.y;
  }
  t.d = __builtin_bit_cast(half4, __builtin_amdgcn_raw_buffer_load_b64(p.sc, (lane & 15) * 8, tile * 128, 0));
  if constexpr (has_min<QT>()) t.m = __builtin_bit_cast(half4, __builtin_amdgcn_raw_buffer_load_b64(p.mn, (lane & 15) * 8, tile * 128, 0));
}

// WM x WN wavefronts; a wavefront owns MTW x NTW 16 x 16 output tiles
template <int QT, int WM, int WN, int MTW, int NTW>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_prompt_kernel(GemmArgs a) {
  constexpr int NW = WM * WN;
  constexpr int BM = WM * MTW * 16, BN = WN * NTW * 16;
  constexpr int NA = BM / (8 * NW);                 // requests per wavefront and x tile
  // weight tile rows (16 rows each) of the block over the wavefronts: FULL whole rows per wavefront, and with 1.5 rows per
  // wavefront (BN = 192 on 8 wavefronts) a pair of wavefronts shares a third row, one k half of the T16 tile each
  constexpr int RT = BN / 16;
  constexpr int FULL = RT / NW, HALF = (RT % NW) ? 1 : 0;
  constexpr int SLOTS = FULL + HALF;
  constexpr int RL = SLOTS * raw_loads<QT>();        // weight requests per wavefront and T16 tile
  // (large tiles of formats that need more registers: the fragment reads stay behind the MFMAs they replace, or the loop spills: fp6
  // 256 x 256 2x slower, int8 and int5 6 - 10 %; where they fit, reads in between are up to 3 % faster)
  constexpr bool TIGHT = MTW * NTW >= 24 && (lo_bits_of(QT) == 8 || hi_bits_of(QT) > 0);
  static_assert(NW == 8 && BM % (8 * NW) == 0 && RT % 2 == 0 && (RT % NW == 0 || 2 * RT == 3 * NW), "tile does not divide over the wavefronts");
  constexpr int ABYTES = BM * 128, BBYTES = BN * 128;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* const As = smem;                            // [3][BM][128 B]
  char* const Bs = smem + 3 * ABYTES;               // [2][BN][128 B]

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int r = lane & 15, g = lane >> 4;
  const int KT = a.K >> 7;                          // host: K % 128 == 0
  // pair form (a.w2: gate / up): the block's first RT / 2 weight tile rows come from w, the others from the same rows of
  // w2, and the epilogue writes act(first) * second: BN / 2 output columns per block
  const bool pair = a.w2 != nullptr;
  const int BNO = pair ? BN / 2 : BN;
  const int nmb = (a.M + BM - 1) / BM, nnb = (a.N + BNO - 1) / BNO;

  // XCD-aware tile order: blocks b and b + 8 share an L2; consecutive tile ids go to one XCD (bijective also when the grid
  // is not a multiple of 8).  Where the tiles of a product outnumber the CUs, the ids run through bands of four row blocks,
  // column by column: the 32 workgroups of an XCD then share 4 x panels (16 bits an element) and 8 weight panels (4 - 8 bits)
  // instead of reading 32 x panels each for itself.  7700 rows: 14336 x 4096 pair 1697 -> 1655 us, 6144 x 4096 351 -> 342 us; bands
  // of 2 and 8 within 1 %.  Fewer tiles run down the columns: in bands 1024 x 4096 at 2048 rows took 38.3 us instead of 33.8,
  // 2048 x 2048 28.6 instead of 27.2, 4096 x 11008 183 instead of 177.
  const int BAND = nmb * nnb > 256 ? 4 : nmb;
  int tid;
  {
    const int nblk = gridDim.x, b = blockIdx.x, q = nblk >> 3, rr = nblk & 7, xcd = b & 7;
    tid = (xcd < rr ? xcd * (q + 1) : rr * (q + 1) + (xcd - rr) * q) + (b >> 3);
  }
  const int sp = tid / (nmb * nnb), in_split = tid - sp * (nmb * nnb);
  const int band = in_split / (BAND * nnb), band_rows = min(BAND, nmb - band * BAND);
  const int in_band = in_split - band * (BAND * nnb);
  const int mb = band * BAND + in_band % band_rows, nb = in_band / band_rows;
  const int row0 = mb * BM, rows = min(BM, a.M - row0);
  const int kt0 = sp * a.kt_per_split, kt1 = min(KT, kt0 + a.kt_per_split);
  const int nkt = kt1 - kt0, T = 2 * nkt;            // T16 k tiles / 64-deep tiles of this workgroup

  // ---- x tile (32-bit byte offsets from the block's first row: M * ldx < 2^31); instruction p of wavefront (wm, wn) fills rows
  // 8 (p WN + wn) .. + 7 of its half; lane i brings the 16 bytes that belong in slot i % 8 of row i / 8, i.e. k slot
  // (i % 8) ^ (i / 8) of that row (rows past the block re-read its last row: never stored)
  uint32_t xoff[NA];
#pragma unroll
  for (int p = 0; p < NA; ++p) {
    const int row = wm * (BM / WM) + (p * WN + wn) * 8 + (lane >> 3);
    xoff[p] = ((uint32_t)min(row, rows - 1) * (uint32_t)a.ldx + (uint32_t)((((lane & 7) ^ (lane >> 3)) & 7) << 3)) * 2u;
  }
  const auto xb = buf_of(a.x + (int64_t)row0 * a.ldx + kt0 * 128);
  auto stage_a = [&](int t, int buf, int p) {
    char* dst = As + buf * ABYTES + (wm * (BM / WM) + wn * 8) * 128;     // wave-uniform; the instruction adds lane * 16
    lds_dma16(xb, dst + p * WN * 1024, xoff[p], t * 128);
  };

  // ---- weight tile rows of this wavefront (block-relative index; a row past N is loaded from the last valid one and never
  // stored) and their raw data: one whole T16 tile (128 k = two 64-deep tiles) per slot
  const int ntiles = (a.N + 15) >> 4;
  int slot_rt[SLOTS];
  RowPlanes wp[SLOTS];
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    if constexpr (HALF) slot_rt[i] = (wave >> 1) * 3 + (i < FULL ? (wave & 1) : 2);
    else slot_rt[i] = wave * FULL + i;
    const bool second = pair && slot_rt[i] >= RT / 2;
    const int trow = pair ? nb * (RT / 2) + slot_rt[i] - second * (RT / 2) : nb * RT + slot_rt[i];
    wp[i] = row_planes<QT>(t16_planes(second ? a.w2 : a.w, QT, a.N, a.K), (int64_t)min(trow, ntiles - 1) * KT + kt0);
  }
  const int half_sel = wave & 1;                     // which k half of the shared row this wavefront expands
  Tile<QT> rawC[SLOTS], rawN[SLOTS];                 // T16 tile being expanded / the next one (in flight)

  // fragment slot of k step s for this lane: (4 s + g) ^ (r & 7); s = 1 flips bit 2
  const int fsw0 = ((g ^ (r & 7)) & 7) << 4;
  const int frag_off[2] = {r * 128 + fsw0, r * 128 + (fsw0 ^ 64)};

  // unit u (k step u % 2 of slot u / 2) of a 64-deep tile of parity h, from rawC to the weight buffer h; the shared row's units
  // exist only in the wavefront that owns that k half
  auto expand = [&](auto hc, int u) {
    constexpr int h = decltype(hc)::value;
    const int i = u >> 1;
    if (i >= FULL && half_sel != h) return;          // wave-uniform
    half8 v;
    if (u & 1) v = unit_expand<QT, 2 * h + 1>(rawC[i]);
    else v = unit_expand<QT, 2 * h>(rawC[i]);
    *(half8*)(Bs + h * BBYTES + slot_rt[i] * 2048 + frag_off[u & 1]) = v;
  };

  float4v acc[MTW][NTW];
#pragma unroll
  for (int j = 0; j < MTW; ++j)
#pragma unroll
    for (int n = 0; n < NTW; ++n) acc[j][n] = float4v{0, 0, 0, 0};

  typedef std::integral_constant<int, 0> I0;
  typedef std::integral_constant<int, 1> I1;
  typedef std::integral_constant<int, 2> I2;
  typedef std::integral_constant<int, 3> I3;
  auto lds_w = [&](int buf, int s) { return Bs + buf * BBYTES + wn * (NTW * 2048) + frag_off[s]; };
  auto lds_x = [&](int buf, int s) { return As + buf * ABYTES + wm * (MTW * 2048) + frag_off[s]; };
  auto frag = [&](const char* p, int i) { return *(const half8*)(p + i * 2048); };

  // ---- the loop.  Tile t (x buffer t % 3, weight buffer t % 2) runs as two k steps of MTW groups of NTW MFMAs.  Fragments: x in one
  // register set that rolls (group j's is replaced behind its last use), weights in two.  At the turn between the two steps of
  // tile t every read of tile t is done and every store of tile t + 1, hence:
  //  * second step of t, first of t + 1: tile t + 2 is expanded into weight buffer t % 2; second step: x tile t + 3 is requested
  //    into x buffer t % 3.  Both are last read in the first step of t, before the turn (lgkmcnt(0), barrier);
  //  * what the second step of t reads of tile t + 1: its expansion ended in the first step of t, its x was requested a tile and a
  //    half ago (vmcnt: what is younger may still be under way).
  half8 wf[2][NTW], xf[MTW];
  // k step S (0 .. 3 of the T16 tile) of tile t = 2 kt + S / 2
  auto step = [&](auto sc, int t, int xcur, int xnext, int xfree) {
    constexpr int S = decltype(sc)::value;
    constexpr bool first = (S & 1) == 0;               // first k step of a tile
    // what is read for the next k step, and the weight tile under expansion: t + 1 in the first k step (its second half of
    // units), t + 2 in the second
    const char* px = first ? lds_x(xcur, 1) : lds_x(xnext, 0);
    const char* pw = first ? lds_w(S >> 1, 1) : lds_w((S >> 1) ^ 1, 0);
    typedef std::integral_constant<int, first ? (S >> 1) ^ 1 : (S >> 1)> H;
#pragma unroll
    for (int j = 0; j < MTW; ++j) {
#pragma unroll
      for (int n = 0; n < NTW; ++n) acc[j][n] = mfma16(wf[S & 1][n], xf[j], acc[j][n]);     // D[n = 4 g + q][m = r]
      if constexpr (TIGHT) __builtin_amdgcn_sched_barrier(0);
      xf[j] = frag(px, j);
#pragma unroll
      for (int n = 0; n < NTW; ++n)
        if (n * MTW / NTW == j) wf[~S & 1][n] = frag(pw, n);
#pragma unroll
      for (int u = 0; u < SLOTS; ++u)
        if ((2 * u + 1) * MTW / (2 * SLOTS) == j) expand(H{}, first ? SLOTS + u : u);
      if constexpr (!first) {
#pragma unroll
        for (int p = 0; p < NA; ++p)
          if (p * MTW / NA == j) stage_a(min(t + 3, T - 1), xfree, p);
      }
      if constexpr (S == 2) {
#pragma unroll
        for (int i = 0; i < SLOTS; ++i)
          if (i * MTW / SLOTS == j) load_raw<QT>(rawN[i], wp[i], min((t >> 1) + 2, nkt - 1), lane);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto turn = [&](auto nc) {
    // own reads and stores done, the next x tile landed
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(decltype(nc)::value));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) load_raw<QT>(rawC[i], wp[i], 0, lane);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int p = 0; p < NA; ++p) stage_a(0, 0, p);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int p = 0; p < NA; ++p) stage_a(1, 1, p);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) load_raw<QT>(rawN[i], wp[i], min(1, nkt - 1), lane);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int p = 0; p < NA; ++p) stage_a(min(2, T - 1), 2, p);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < 2 * SLOTS; ++u) expand(I0{}, u);
#pragma unroll
  for (int u = 0; u < SLOTS; ++u) expand(I1{}, u);
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(2 * NA + RL));
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int j = 0; j < MTW; ++j) xf[j] = frag(lds_x(0, 0), j);
#pragma unroll
  for (int n = 0; n < NTW; ++n) wf[0][n] = frag(lds_w(0, 0), n);
  int b0 = 0;
  for (int t = 0; t < T; t += 2) {
    const int b1 = b0 == 2 ? 0 : b0 + 1, b2 = b1 == 2 ? 0 : b1 + 1;
    step(I0{}, t, b0, b1, b2);
    turn(std::integral_constant<int, NA>{});           // younger than x tile t + 1: x tile t + 2 (and raw weights that rawC takes now)
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) rawC[i] = rawN[i];
    step(I1{}, t, b0, b1, b0);
    step(I2{}, t + 1, b1, b2, b0);
    turn(std::integral_constant<int, NA + RL>{});      // younger than x tile t + 2: x tile t + 3, raw weights
    step(I3{}, t + 1, b1, b2, b1);
    b0 = b2;
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));   // the look-ahead of the last tile: requests (clamped), reads and expansion

  // ---- epilogue.  A lane holds 4 consecutive output columns (n = 16 tile + 4 g + q) of row m = 16 j + r.
  // Two forms: fp32 partial slabs (K splits, or an output the staged form does not cover: the reduce kernel of
  // gemm_lowbit.hip then applies bias / activation / residual), or the staged 16-bit output.
  // (pair form: the wavefronts of the second column half hold the second product of the first half's columns)
  const int wn_out = pair ? wn % (WN / 2) : wn;
  const bool second_half = pair && wn >= WN / 2;
  const int ocol0 = nb * BNO + wn_out * (NTW * 16), orow0 = row0 + wm * (MTW * 16);
  const int64_t mtot = a.M;
  if (!pair && (a.splitk > 1 || a.force_partial)) {
#pragma unroll
    for (int n = 0; n < NTW; ++n) {
      const int ncol = ocol0 + 16 * n + 4 * g;
      if (ncol >= a.N) continue;
#pragma unroll
      for (int j = 0; j < MTW; ++j) {
        const int64_t orow = orow0 + 16 * j + r;
        if (orow >= row0 + rows) continue;
        float* dst = a.partial + ((int64_t)sp * mtot + orow) * a.N + ncol;
        if (ncol + 4 <= a.N && (a.N & 3) == 0) *(float4v*)dst = acc[j][n];
        else {
#pragma unroll
          for (int q = 0; q < 4; ++q)             // (static register indices: a run-time index would put acc in scratch)
            if (ncol + q < a.N) dst[q] = acc[j][n][q];
        }
      }
    }
    return;
  }
  // staged form (host: 16-bit output, N % 8 == 0, ldo % 8 == 0, 16-byte aligned out / residual): bias added to the fp32
  // accumulators, rounded to the output type, the wavefront's tile transposed through LDS ([16 MTW rows][16 NTW
  // columns], rows padded by 16 bytes), then whole row segments (16 bytes per lane) leave with activation and residual
  // applied (a rolled loop: the activation's code exists once)
  constexpr int RB = 32 * NTW + 16;
  char* stg = smem + wave * (MTW * 16 * RB);
  __builtin_amdgcn_s_barrier();                      // every wavefront's last look-ahead tile has landed and been read
#pragma unroll
  for (int n = 0; n < NTW; ++n) {
    const int ncol = ocol0 + 16 * n + 4 * g;
    float bias[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const _Float16* bsrc = (const _Float16*)(second_half ? a.bias2 : a.bias);
    if (bsrc != nullptr && ncol < a.N) {
      const half4 b4 = *(const half4*)(bsrc + ncol);
#pragma unroll
      for (int q = 0; q < 4; ++q) bias[q] = (float)b4[q];
    }
#pragma unroll
    for (int j = 0; j < MTW; ++j) {
      uint2v pk;
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) v[q] = acc[j][n][q] + bias[q];
      if (a.out_type == OUT_F16) {
        pk = __builtin_bit_cast(uint2v, half4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]});
      } else {
        pk.x = (uint32_t)f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16);
        pk.y = (uint32_t)f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16);
      }
      *(uint2v*)(stg + (16 * j + r) * RB + (16 * n + 4 * g) * 2) = pk;
    }
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(63));
  constexpr int CH = 2 * NTW;                        // 16-byte chunks per row
  static_assert((MTW * 16 * CH) % 64 == 0, "row chunks do not divide over the lanes");
  const bool plain = a.act == ACT_NONE && a.residual == nullptr && !pair;
  constexpr int ITS = MTW * 16 * CH / 64;
  int it0 = 0, it1 = ITS;
  const char* stg2 = stg;
  if (pair) {
    // the two wavefronts that hold a tile's first and second products take half of its rows each: wavefronts w and w + 4
    // share a SIMD, so with the first-product wavefronts alone two of the four SIMDs did all exponentials and divisions
    // (14336 x 4096 pair, 7700 rows: 1655 -> 1610 us)
    __builtin_amdgcn_s_barrier();                    // the partner's tile is complete in LDS
    if (second_half) { it0 = ITS / 2; stg -= (WN / 2) * (MTW * 16 * RB); }
    else it1 = ITS / 2;
    stg2 = stg + (WN / 2) * (MTW * 16 * RB);
  }
  // the 16-bit pairs of a 16-byte chunk, f(first, second) each
  auto chunk = [&](uint4v p, uint4v q, auto f) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float lo, hi, qlo, qhi;
      if (a.out_type == OUT_F16) {
        const half2v h = u2h(p[e]), hq = u2h(q[e]);
        lo = (float)h[0]; hi = (float)h[1]; qlo = (float)hq[0]; qhi = (float)hq[1];
      } else {
        lo = bf16_bits_to_f32((uint16_t)(p[e] & 0xffffu)); hi = bf16_bits_to_f32((uint16_t)(p[e] >> 16));
        qlo = bf16_bits_to_f32((uint16_t)(q[e] & 0xffffu)); qhi = bf16_bits_to_f32((uint16_t)(q[e] >> 16));
      }
      lo = f(lo, qlo);
      hi = f(hi, qhi);
      if (a.out_type == OUT_F16) p[e] = h2u(half2v{(_Float16)lo, (_Float16)hi});
      else p[e] = (uint32_t)f32_to_bf16_bits(lo) | ((uint32_t)f32_to_bf16_bits(hi) << 16);
    }
    return p;
  };
  // fn(own chunk, the same chunk of the partner's tile or the residual) -> what is stored
  auto rows_out = [&](auto fn) {
#pragma unroll 2
    for (int it = it0; it < it1; ++it) {
      const int idx = it * 64 + lane, row = idx / CH, ch = idx % CH;
      const int col = ocol0 + ch * 8;
      if (orow0 + row >= row0 + rows || col >= a.N) continue;
      const uint4v p = *(const uint4v*)(stg + row * RB + ch * 16);
      const int64_t oi = (int64_t)(orow0 + row) * a.ldo + col;
      uint4v q = uint4v{0, 0, 0, 0};
      if (pair) q = *(const uint4v*)(stg2 + row * RB + ch * 16);
      else if (a.residual != nullptr) q = *(const uint4v*)((const uint16_t*)a.residual + oi);
      *(uint4v*)((uint16_t*)a.out + oi) = fn(p, q);
    }
  };
  // act(first) * second on the rounded 16-bit values (what a separate activation kernel would read).  The usual gate has a loop of
  // its own: with the choice of the activation inside, an element took twice the instructions
  if (pair && a.act == ACT_SILU) rows_out([&](uint4v p, uint4v q) { return chunk(p, q, [](float x, float u) { return silu_rcp(x) * u; }); });
  else if (pair) rows_out([&](uint4v p, uint4v q) { return chunk(p, q, [&](float x, float u) { return act_apply(a.act, x) * u; }); });
  else if (plain) rows_out([](uint4v p, uint4v) { return p; });
  else rows_out([&](uint4v p, uint4v q) { return chunk(p, q, [&](float x, float u) { return act_apply(a.act, x) + u; }); });
}

template <int QT, int WM, int WN, int MTW, int NTW>
static int gemm_prompt_launch_cfg(const GemmArgs& a, hipStream_t st) {
  constexpr int NW = WM * WN, BM = WM * MTW * 16, BN = WN * NTW * 16;
  const size_t lds = prompt_lds_tiles(BM, BN, NW, MTW, NTW);
  static bool attr_set = false;
  if (!attr_set) {
    if (hipFuncSetAttribute((const void*)gemm_prompt_kernel<QT, WM, WN, MTW, NTW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
      return -101;
    attr_set = true;
  }
  const int bno = a.w2 != nullptr ? BN / 2 : BN;
  const int tiles = ((a.M + BM - 1) / BM) * ((a.N + bno - 1) / bno);
  hipLaunchKernelGGL((gemm_prompt_kernel<QT, WM, WN, MTW, NTW>), dim3(tiles * a.splitk), dim3(64 * NW), lds, st, a);
  return HIP_CHECK_LAUNCH();
}

// configurations in the order of gemm_prompt.hip's table: 256 x 256, 256 x 192, 128 x 128, 256 x 128, 192 x 256, 192 x 128
#define PROMPT_NCFG 6
template <int QT>
static int gemm_prompt_launch(const GemmArgs& a, int cfg, hipStream_t st) {
  switch (cfg) {
    case 0: return gemm_prompt_launch_cfg<QT, 2, 4, 8, 4>(a, st);
    case 1: return gemm_prompt_launch_cfg<QT, 2, 4, 8, 3>(a, st);
    case 2: return gemm_prompt_launch_cfg<QT, 2, 4, 4, 2>(a, st);
    case 3: return gemm_prompt_launch_cfg<QT, 2, 4, 8, 2>(a, st);
    case 4: return gemm_prompt_launch_cfg<QT, 2, 4, 6, 4>(a, st);
    case 5: return gemm_prompt_launch_cfg<QT, 2, 4, 6, 2>(a, st);
    default: return -4;
  }
}

}  // namespace bigdl
