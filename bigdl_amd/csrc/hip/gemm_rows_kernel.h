// Dequant-fused product for a few rows of x on gfx950:  y[M,N] = f(x[M,K] . dequant(W)[N,K]^T), up to 64 rows (blocks of
// 16 * MT rows above that).  Batched decode, short prompts and speculative verification run on it, as far as they do not on the product
// on x in fragment order (gemm_frag_kernel.h: most products of more than 64 rows); up to 16 rows it folds
// the RMSNorm of x in, and a gate / up pair is one launch with act(g) * u in its epilogue.
//
// What bounds it: the weights (28 MB for Llama-2-7B's qkv, 5.6 us at the 5 TB/s that 256 CUs draw) and, from about 32 rows on, x,
// which every workgroup reads whole: 512 KiB for 64 rows of 4096, at about 57 GB/s a CU.  Hence the structure:
//  * One workgroup of 8 wavefronts per CU owns NT 16-column tiles and all of K; the wavefronts take k-tiles in turn, so a
//    weight tile and an x tile belong to one wavefront each: no barriers, no sharing, until the partial sums meet in LDS
//    once, at the end.  No K split across workgroups and so no fp32 slabs and no reduce launch (the tile kernel of
//    gemm_kernel.h spends 6.5 us on the slabs and 4.7 us on the reduce of a 64-row qkv), except where K is so long that
//    the x of a whole K outweighs them (planner in gemm_rows.hip).
//  * NT follows from the column count so that the grid is one turn of the CUs: fewer columns per workgroup would mean more
//    workgroups reading the same x (64 rows, qkv: NT = 1 / 2 / 3: 32 / 29 / 17 us; 3 is 256 workgroups).
//  * x is read in whole 128-byte lines (8 rows x 128 bytes a request) and turned into MFMA fragments through a private LDS
//    patch.  Fragments read straight from memory are 64-byte pieces of 16 rows: the same kernel took 21 instead of 17 us.
//  * Loads are ordered by hand (rows_issued) and go through buffer descriptors: scalar offsets instead of 64-bit vector
//    addresses (which spilled), and what lies outside x or past the last k-tile costs no memory access.
// Measured, one MI355X, sym_int4, us, before (skinny kernel up to 16 rows, tile kernel above) -> this kernel: qkv 12288 x 4096 at
// 12 / 32 / 64 rows 15.3 -> 11.6, 19.8 -> 12.1, 25.3 -> 16.9; gate / up 11008 x 4096 28.1 -> 17.7, 26.2 -> 17.6, 33.4 -> 23.1; o
// 4096 x 4096 8.0 -> 8.0, 12.8 -> 9.0, 16.3 -> 11.9; down 4096 x 11008 16.5 -> 13.5, 17.7 -> 17.8, 22.0 -> 20.9 (two K splits).
// A decode step of 12 sequences of a Llama-3-8B-shaped q4_k model with 1900 keys each: 156 -> 108 us a layer.
#pragma once
#include "gemv_kernel.h"

namespace bigdl {

struct RowsArgs {
  const _Float16* x;      // [M, ldx]
  const void* w;          // T16 [N, K]
  const void* w2;         // pair form: second weight, same shape and format
  void* out;              // [M, ldo]
  float* partial;         // [splitk][M][N] (x 2 in the pair form) fp32 when splitk > 1
  const void* bias;
  const void* bias2;
  const void* residual;
  const _Float16* gamma;  // RMSNorm weight folded into x, or null
  float eps, gamma_offset;
  int M, N, K, ldx, ldo, act, out_type;
  int splitk, kt_per_split;
};

// The loads above this line are issued above it.  Without it the compiler sinks loads to their first use (its schedule
// aims at few registers): every one then waits for its own memory round trip.
__device__ __forceinline__ void rows_issued() { asm volatile("" ::: "memory"); }

constexpr int ROWS_NW = 8;            // wavefronts per workgroup
// partial sums of all wavefronts at once, or of one half after the other where they do not fit
constexpr bool rows_two_phase(int mt, int ns, int nw) { return nw * mt * ns > 144; }
constexpr int rows_red_kib(int mt, int ns, int nw) { return rows_two_phase(mt, ns, nw) ? nw * mt * ns / 2 : nw * mt * ns; }
constexpr int rows_lds(int mt, int ns, int nw) {
  return (rows_red_kib(mt, ns, nw) > nw * mt * 4 ? rows_red_kib(mt, ns, nw) : nw * mt * 4) * 1024 + (mt == 1 ? nw * mt * 64 : 0);
}

// halves of an x tile on their way in registers
constexpr int rows_x_halves(int mt, int ns) { return mt * ns > 16 || mt * ns == 12 ? 1 : 2; }
// k-tiles of weights requested ahead: about eight tiles per wavefront (72 KiB a CU), as far as the registers of two
// wavefronts per SIMD hold them
constexpr int rows_ahead(int qt, int mt, int ns) {
  const int tile = qt == Q_Q6_K ? 14 : lo_bits_of(qt) + hi_bits_of(qt) + 2 + (has_min_of(qt) ? 2 : 0);        // VGPRs of a weight tile
  const int other = ns * mt * 4 + 8 * mt * rows_x_halves(mt, ns) + (mt == 4 ? 30 : mt == 1 ? 6 * ns : 0) + (lo_bits_of(qt) == 8 || qt == Q_Q6_K ? 120 : has_min_of(qt) || hi_bits_of(qt) == 2 ? 84 : 72);
  int ahead = 1;
  while (ahead < 4 && (ahead < 2 || ahead * ns < 6) && other + (ahead + 1) * ns * tile <= 250) ++ahead;
  return ahead;
}

typedef __amdgpu_buffer_rsrc_t rows_rsrc;
__device__ __forceinline__ rows_rsrc rows_buffer(const void* p, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, bytes, 0x00027000);
}
constexpr int ROWS_NT = 2;            // cache policy of a buffer load: non-temporal
// a lane offset past the end of every buffer here (a gigabyte at most): the load returns zeros, no memory access
constexpr uint32_t ROWS_OUT = 0x40000000;
static_assert(ROWS_OUT + ROWS_OUT == 0x80000000u, "a row and a column that are both outside: no overflow (the type is unsigned)");

// one weight tile through buffer loads: every address is a scalar offset plus a lane constant
template <int QT>
struct RowsPlanes {
  rows_rsrc lo, hi, sc, mn;
  __device__ __forceinline__ void init(const T16Planes& p, int64_t tile0, int tiles) {
    lo = rows_buffer(p.lo + tile0 * (lo_bits_of(QT) * 256), tiles * (lo_bits_of(QT) * 256));
    if constexpr (hi_bits_of(QT) > 0) hi = rows_buffer(p.hi + tile0 * (hi_bits_of(QT) * 256), tiles * (hi_bits_of(QT) * 256));
    sc = rows_buffer(p.sc + tile0 * 64, tiles * 128);
    if constexpr (has_min_of(QT)) mn = rows_buffer(p.mn + tile0 * 64, tiles * 128);
  }
  // out: 0, or ROWS_OUT for a tile that does not exist (zeros, no memory access)
  template <int AUX = ROWS_NT>
  __device__ __forceinline__ void load(Tile<QT>& t, int tile, int lane, uint32_t out) const {
    t.lo0 = __builtin_amdgcn_raw_buffer_load_b128(lo, lane * 16 + out, tile * (lo_bits_of(QT) * 256), AUX);
    if constexpr (lo_bits_of(QT) == 8) t.lo1 = __builtin_amdgcn_raw_buffer_load_b128(lo, lane * 16 + 1024 + out, tile * 2048, AUX);
    if constexpr (hi_bits_of(QT) == 1) t.hi0 = __builtin_amdgcn_raw_buffer_load_b32(hi, lane * 4 + out, tile * 256, AUX);
    if constexpr (hi_bits_of(QT) == 2) {
      const uint2v h = __builtin_amdgcn_raw_buffer_load_b64(hi, lane * 8 + out, tile * 512, AUX);
      t.hi0 = h.x;
      t.hi1 = h.y;
    }
    const uint32_t r8 = (lane & 15) * 8 + out;
    t.d = __builtin_bit_cast(half4, __builtin_amdgcn_raw_buffer_load_b64(sc, r8, tile * 128, AUX));
    if constexpr (has_min_of(QT)) t.m = __builtin_bit_cast(half4, __builtin_amdgcn_raw_buffer_load_b64(mn, r8, tile * 128, AUX));
  }
};

// How a lane's share of a weight tile becomes MFMA operands.  T16 formats: fragment s holds k = 32 s + 8 g + j, one 32-element
// scale block per fragment.
template <int QT>
__device__ __forceinline__ half8 rows_fragment(const Tile<QT>& t, int s, int) { return decode_step<QT>(t, s); }
template <int QT>
__device__ __forceinline__ float rows_scale(const Tile<QT>& t, int s) { return (float)t.d[s] * post_scale<QT>(); }
template <int QT>
__device__ __forceinline__ half8 rows_scaled(const Tile<QT>& t, half8 code, int s) {
  _Float16 d = t.d[s];
  if constexpr (post_scale<QT>() != 1.0f) d = (_Float16)fminf((float)d * post_scale<QT>(), 65504.0f);
  if constexpr (has_min<QT>()) return code * d + t.m[s];
  return code * d;
}
template <int QT>
__device__ __forceinline__ int rows_chunk(int s, int g) { return 4 * (s & 1) + g; }     // 16-byte chunk of half an x tile

// q6_k as the file's blocks hold it (210 bytes for 256 elements of a row: 128 of low nibbles, 64 of high bit pairs, 16 int8
// sub-scales, fp16 d): a k-tile is half a block.  Lane group g takes bytes 16 g .. of the half's low nibbles -- 64 contiguous
// bytes a row and request -- so that fragment s holds k = 32 ((g >> 1) + 2 (s >> 1)) + 16 (g & 1) + 8 (s & 1) + j, all of it
// in sub-block g + 4 (s >> 1).  Code times sub-scale is exact in fp16 up to 2048 and within 2^-11 above (12 % of a normal
// matrix's weights); d multiplies the fp32 product, once for the two steps of a half k-tile.  Error of a weight, rms: 1.6e-4,
// where the expansion to fp16 has 2.1e-4.
// Blocks start at even bytes, every other one between two dwords.  16-byte loads from there are split by the address unit
// (4096 x 11008, 1 row: 34 us, 25 this way); so the dwords around them are loaded and shifted into place.  The last dword's address steps
// back where it is not needed: nothing outside the block is touched.
typedef uint4v rows_raw16 __attribute__((aligned(4)));
typedef uint2v rows_raw8 __attribute__((aligned(4)));
template <>
struct Tile<Q_Q6_K> {
  uint4v ql, qh;
  uint32_t ql4, qh4, sc2;     // the dword behind each
  uint2v sc;
  _Float16 d;
};
template <>
struct RowsPlanes<Q_Q6_K> {
  const uint8_t* row[4];      // this lane's weight row of every column tile
  template <int NT>
  __device__ __forceinline__ void init(const void* w, int first, int N, int K, int lane) {
#pragma unroll
    for (int n = 0; n < NT; ++n) row[n] = (const uint8_t*)w + (int64_t)min((first + n) * 16 + (lane & 15), N - 1) * (K / 256 * 210);
  }
  __device__ __forceinline__ void load(Tile<Q_Q6_K>& t, int n, int kt, int lane) const {
    const uint8_t* b = row[n] + (kt >> 1) * 210;
    const int h = kt & 1, g = lane >> 4, odd = (int)((uintptr_t)b & 2);
    const uint8_t* c = b - odd;          // (the pieces start at multiples of 8: they are all as far off a dword as the block)
    const uint8_t* last = c + 2 * odd;   // + 4 where the shift needs one more dword
    t.ql = *(const rows_raw16*)(c + 64 * h + 16 * g);
    t.ql4 = *(const uint32_t*)(last + 64 * h + 16 * g + 12);
    t.qh = *(const rows_raw16*)(c + 128 + 32 * h + 16 * (g & 1));
    t.qh4 = *(const uint32_t*)(last + 128 + 32 * h + 16 * (g & 1) + 12);
    t.sc = *(const rows_raw8*)(c + 192 + 8 * h);
    t.sc2 = *(const uint32_t*)(last + 192 + 8 * h + 4);
    t.d = *(const _Float16*)(b + 208);
  }
  // the tile with its pieces shifted into place
  __device__ __forceinline__ void settle(Tile<Q_Q6_K>& t, int n, int kt) const {
    const uint32_t odd = (uint32_t)((uintptr_t)(row[n] + (kt >> 1) * 210) & 2);
    t.ql = uint4v{__builtin_amdgcn_alignbyte(t.ql[1], t.ql[0], odd), __builtin_amdgcn_alignbyte(t.ql[2], t.ql[1], odd),
                  __builtin_amdgcn_alignbyte(t.ql[3], t.ql[2], odd), __builtin_amdgcn_alignbyte(t.ql4, t.ql[3], odd)};
    t.qh = uint4v{__builtin_amdgcn_alignbyte(t.qh[1], t.qh[0], odd), __builtin_amdgcn_alignbyte(t.qh[2], t.qh[1], odd),
                  __builtin_amdgcn_alignbyte(t.qh[3], t.qh[2], odd), __builtin_amdgcn_alignbyte(t.qh4, t.qh[3], odd)};
    t.sc = uint2v{__builtin_amdgcn_alignbyte(t.sc[1], t.sc[0], odd), __builtin_amdgcn_alignbyte(t.sc2, t.sc[1], odd)};
  }
};
template <>
__device__ __forceinline__ half8 rows_fragment<Q_Q6_K>(const Tile<Q_Q6_K>& t, int s, int g) {
  H8 r;
  const half2v off = {(_Float16)1056.0f, (_Float16)1056.0f};       // 1024 + 32
  const _Float16 sc = (_Float16)(float)(int8_t)(t.sc[s >> 1] >> (8 * g));
  const int up = 2 * (g >> 1) + 4 * (s >> 1);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t lo = t.ql[2 * (s & 1) + i] >> (4 * (s >> 1)), hi = t.qh[2 * (s & 1) + i] >> up;
    const uint32_t code = (lo & 0x0F0F0F0Fu) | ((hi & 0x03030303u) << 4);
    r.h2[2 * i] = (u2h(__builtin_amdgcn_perm(0x64646464u, code, 0x04010400u)) - off) * sc;
    r.h2[2 * i + 1] = (u2h(__builtin_amdgcn_perm(0x64646464u, code, 0x04030402u)) - off) * sc;
  }
  return r.v;
}
template <>
__device__ __forceinline__ int rows_chunk<Q_Q6_K>(int s, int g) { return 2 * g + (s & 1); }

// MT = 16-row tiles of x, NT = 16-column tiles of a weight per workgroup, WD = k-tiles of weights requested ahead.  What the
// first requests need is preloaded into scalar registers (build flag, see gemv_kernel.h).  4 decode steps of 4 layers, 12 sequences,
// Llama-3-8B shape: 1676 -> 1641 us; of 3 layers, 64 sequences, Llama-2-7B shape: 2798 -> 2772.
// Pairs of six or eight tiles: the look-ahead is one k-tile, and requested all at once behind it, it came a memory round trip late.  Each
// tile is requested again as soon as it has been multiplied (all four steps at once), and the other five or seven hide its way.  With minima or
// 8-bit codes only, us before -> now: asym_int4 14336 x 4096 at 4 / 12 rows 23.5 -> 21.5, 25.0 -> 23.9, 11008 x 4096 at 8 rows 19.0 -> 17.5;
// sym_int8 14336 x 4096 at 16 rows 28.8 -> 25.7, fp8_e4m3 at 12 rows 31.1 -> 28.2; other formats' tiles are smaller and take it +-1 %,
// single products of four tiles, whose look-ahead is two k-tiles, as well.
// (fp8_e5m2's six tiles take 171 registers so, with which no workgroup starts beside the last wavefront of another: 16.6 us for 15.9 where CUs
// have two workgroups, 21440 x 1024 at 6 rows.)
constexpr bool rows_rolls(int qt, int mt, int ns, bool pair) {
  return mt == 1 && qt != Q_Q6_K && pair && ns >= 6 && (has_min_of(qt) || lo_bits_of(qt) == 8) && !(qt == Q_FP8_E5M2 && ns == 6);
}
// ... and with 8-bit codes not where some wavefronts have no k-tile at all and the others one, with nothing to request again: SHORT.  fp8_e4m3
// 20896 x 768 at 12 rows, six / eight tiles, 15.2 / 19.2 us rolling 16.2 / 20.1, sym_int8 14.5 / 18.5 and 15.0 / 18.6, 23296 x 512 at 4 rows 11.9 and
// 12.2; 11000 x 1024 at 16 rows, a k-tile for each, 9.9 and 9.5.  With minima it pays there too (asym_int4 23296 x 512 12.7, rolling 11.6).
constexpr bool rows_has_short(int qt, int mt, int ns, bool pair) { return rows_rolls(qt, mt, ns, pair) && lo_bits_of(qt) == 8; }
template <int QT, int MT, int NT, bool PAIR, bool SHORT = false, int NW = ROWS_NW, int WD = rows_ahead(QT, MT, PAIR ? 2 * NT : NT)>
__global__ __launch_bounds__(NW * 64, (NW + 3) / 4) void gemm_rows_kernel(const _Float16* p_x, const void* p_w, const void* p_w2,
                                                                          const _Float16* p_gamma, int p_M, int p_N, int p_K,
                                                                          int p_ldx, int p_kt_per_split, float p_goff, RowsArgs a) {
  a.x = p_x; a.w = p_w; a.w2 = p_w2; a.gamma = p_gamma; a.M = p_M; a.N = p_N; a.K = p_K; a.ldx = p_ldx;
  a.kt_per_split = p_kt_per_split; a.gamma_offset = p_goff;
  constexpr int NS = PAIR ? 2 * NT : NT;             // weight tiles per k-tile
  constexpr bool POST = MT == 1;                     // block scale on the fp32 product instead of the fp16 code (q6_k: always)
  constexpr bool NORM = MT == 1;                     // the folded RMSNorm exists for up to 16 rows
  constexpr bool MINS = POST && has_min_of(QT);
  constexpr bool ROLL = !SHORT && rows_rolls(QT, MT, NS, PAIR);
  constexpr int XB = MT * 2048;                      // bytes of half a staged x tile: MT * 16 rows of 64 halves
  constexpr bool TWO = rows_two_phase(MT, NS, NW);
  constexpr int NR = TWO ? NW / 2 : NW;              // wavefronts whose partial sums are in LDS at once
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* red = (float*)smem;                         // [NR][MT * NS][64][4], once the x tiles [NW][2][XB] have been read
  float* ssq_sh = (float*)(smem + rows_lds(MT, NS, NW) - (NORM ? NW * MT * 64 : 0));     // [NW][MT * 16] (NORM)

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int KT = (a.K + 127) >> 7;
  const int ntiles = (a.N + 15) >> 4;
  const int nb = blockIdx.x, sp = blockIdx.z;
  const int kt0 = sp * a.kt_per_split, kt1 = min(KT, kt0 + a.kt_per_split);
  const int row0 = blockIdx.y * (MT * 16), rows = min(MT * 16, a.M - row0);

  RowsPlanes<QT> pl, pl2;
  constexpr bool RAW = QT == Q_Q6_K;
  static_assert(!RAW || !PAIR, "q6_k: single products");
  if constexpr (RAW) pl.template init<NT>(a.w, nb * NT, a.N, a.K, lane);
  else pl.init(t16_planes(a.w, QT, a.N, a.K), (int64_t)nb * NT * KT, min(NT, ntiles - nb * NT) * KT);
  if constexpr (PAIR) pl2.init(t16_planes(a.w2, QT, a.N, a.K), (int64_t)nb * NT * KT, min(NT, ntiles - nb * NT) * KT);
  int tbase[NT];                                     // first tile of the block's tile rows (past the last one: that again)
#pragma unroll
  for (int n = 0; n < NT; ++n) tbase[n] = min(n, ntiles - 1 - nb * NT) * KT;

  // this wavefront's k-tiles: kt0 + wave, + NW, ...  Past them the lane offsets point behind the buffers: such a load returns
  // zeros and moves nothing, so that the loop has one body (a kernel this short pays for every instruction that it fetches)
  // and every wait a fixed count of younger loads
  const int nk = kt1 - kt0 > wave ? (kt1 - kt0 - wave + NW - 1) / NW : 0;
  auto kmap = [&](int i) { return min(kt0 + wave + i * NW, KT - 1); };
  auto past = [&](int i) { return i < nk ? 0u : ROWS_OUT; };

  Tile<QT> tt[WD][NS];
  auto fetch_w = [&](Tile<QT> (&t)[NS], int i) {
    const int kt = kmap(i);
    const uint32_t out = past(i);
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      if constexpr (RAW) pl.load(t[n], n, kt, lane);        // (past the end: the last tile again, never multiplied)
      else pl.load(t[n], tbase[n] + kt, lane, out);
      if constexpr (PAIR) pl2.load(t[NT + n], tbase[n] + kt, lane, out);
    }
  };
  // x of half a k-tile: 2 * MT loads of 8 whole 128-byte row pieces, lane i bringing slot i % 8 of row 8 p + i / 8
  constexpr int NP = 2 * MT;
  const int srow = lane >> 3, slot = lane & 7;
  const rows_rsrc xb = rows_buffer(a.x + (int64_t)row0 * a.ldx, rows * a.ldx * 2);
  // without a norm the buffer of gamma is empty: its loads return zero, and the factor is 0 + 1
  const bool norm = NORM && a.gamma != nullptr;
  const rows_rsrc gb = rows_buffer(norm ? a.gamma : a.x, norm ? a.K * 2 : 0);
  const _Float16 goff = (_Float16)(norm ? a.gamma_offset : 1.0f);
  uint32_t xoff[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) xoff[p] = 8 * p + srow < rows ? (uint32_t)((8 * p + srow) * a.ldx * 2 + slot * 16) : ROWS_OUT;
  constexpr int XH = rows_x_halves(MT, NS);
  uint4v xr[XH][NP];
  uint4v gr[2];
  auto fetch_x = [&](int i, int h) {
    const int k = kmap(i) * 128 + h * 64;
    const uint32_t out = i < nk && k + slot * 8 < a.K ? 0u : ROWS_OUT;
#pragma unroll
    for (int p = 0; p < NP; ++p) xr[h % XH][p] = __builtin_amdgcn_raw_buffer_load_b128(xb, xoff[p] + out, k * 2, 0);
    if constexpr (NORM) gr[h] = __builtin_amdgcn_raw_buffer_load_b128(gb, slot * 16 + out, k * 2, 0);
  };
  char* xt = smem + wave * (2 * XB);                 // this wavefront's own: no barriers in the main loop
  float ssq[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) ssq[p] = 0.0f;
  auto stage_from = [&](auto& xs, auto& gs, int h) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      half8 v = __builtin_bit_cast(half8, xs[h % XH][p]);
      if constexpr (NORM) {
        ssq[p] += frag_sumsq(v);
        v = v * (__builtin_bit_cast(half8, gs[h]) + goff);
      }
      *(half8*)(xt + h * XB + (8 * p + srow) * 128 + ((slot ^ srow) << 4)) = v;
    }
  };
  auto stage_x = [&](int h) { stage_from(xr, gr, h); };
  // ROLL: one weight tile of k-tile i, so that the requests follow each other in the order of their use
  auto fetch_tile = [&](Tile<QT>& t, int n, int i) {
    if constexpr (!RAW) {
      const int kt = kmap(i);
      const uint32_t out = past(i);
      if (!PAIR || n < NT) pl.load(t, tbase[n % NT] + kt, lane, out);
      else if constexpr (PAIR) pl2.load(t, tbase[n % NT] + kt, lane, out);
    }
    rows_issued();
  };

  // x first (vector loads return in order), then the weights of the first WD k-tiles
  fetch_x(0, 0);
  if constexpr (XH == 2) fetch_x(0, 1);
  rows_issued();
  uint4v xr0[ROLL ? 2 : 1][NP], gr0[2];
  if constexpr (ROLL) {
    // (the loop's order from the start: its waits count what is younger on every way into it)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int p = 0; p < NP; ++p) xr0[h][p] = xr[h][p];
      if constexpr (NORM) gr0[h] = gr[h];
    }
#pragma unroll
    for (int d = 0; d < WD; ++d)
#pragma unroll
      for (int n = 0; n < NS; ++n) {
        fetch_tile(tt[d][n], n, d);
        if (d == WD - 1 && n == NS / 2) {
          fetch_x(1, 0);
          fetch_x(1, 1);
          rows_issued();
        }
      }
  } else {
#pragma unroll
    for (int d = 0; d < WD; ++d) {
      fetch_w(tt[d], d);
      rows_issued();
    }
  }

  float4v acc[NS][MT];
#pragma unroll
  for (int n = 0; n < NS; ++n)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[n][j] = float4v{0, 0, 0, 0};

  auto x_fragment = [&](int h, int s, int j) {
    return *(const half8*)(xt + h * XB + (16 * j + r) * 128 + ((rows_chunk<QT>(s, g) ^ (r & 7)) << 4));
  };
  // MINS: block sums of x in the layout of the product: a fragment of ones
  auto x_sum = [&](half8 xa) {
    const half8 one8 = {1, 1, 1, 1, 1, 1, 1, 1};
    return MINS ? mfma16(xa, one8, float4v{0, 0, 0, 0}) : float4v{0, 0, 0, 0};
  };
  // one fragment of a weight tile and x: code x x, scaled in fp32, + minimum x block sum.  ROLL: scale and minimum are converted by
  // themselves; full-rate multiply-adds follow, where the mixed form with a half operand issues at half the rate
  auto multiply = [&](float4v& c, const Tile<QT>& t, half8 xa, float4v sx, int s) {
    if constexpr (!RAW) {
      const half8 code = rows_fragment<QT>(t, s, g);
      float d = rows_scale<QT>(t, s);
      if constexpr (ROLL) asm("" : "+v"(d));
      const float4v p = mfma16(xa, code, float4v{0, 0, 0, 0});
#pragma unroll
      for (int q = 0; q < 4; ++q) c[q] = fmaf(p[q], d, c[q]);
      if constexpr (MINS) {
        float m = (float)t.m[s];
        if constexpr (ROLL) asm("" : "+v"(m));
#pragma unroll
        for (int q = 0; q < 4; ++q) c[q] = fmaf(sx[q], m, c[q]);
      }
    }
  };
  auto half_step = [&](Tile<QT> (&t)[NS], int h) {
    if constexpr (RAW) {
      half8 xa[2][MT];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) xa[i][j] = x_fragment(h, 2 * h + i, j);
#pragma unroll
      for (int n = 0; n < NS; ++n) {
        const half8 c0 = rows_fragment<QT>(t[n], 2 * h, g), c1 = rows_fragment<QT>(t[n], 2 * h + 1, g);
        const float d = (float)t[n].d;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          const float4v c = mfma16(xa[1][j], c1, mfma16(xa[0][j], c0, float4v{0, 0, 0, 0}));
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[n][j][q] = fmaf(c[q], d, acc[n][j][q]);
        }
      }
    } else if constexpr (POST) {
#pragma unroll
      for (int s = 2 * h; s < 2 * h + 2; ++s) {
        const half8 xa = x_fragment(h, s, 0);
        const float4v sx = x_sum(xa);
#pragma unroll
        for (int n = 0; n < NS; ++n) multiply(acc[n][0], t[n], xa, sx, s);
      }
    } else {
#pragma unroll
      for (int s = 2 * h; s < 2 * h + 2; ++s) {
        half8 xa[MT];
#pragma unroll
        for (int j = 0; j < MT; ++j) xa[j] = x_fragment(h, s, j);
#pragma unroll
        for (int n = 0; n < NS; ++n) {
          const half8 bf = rows_scaled<QT>(t[n], rows_fragment<QT>(t[n], s, g), s);
#pragma unroll
          for (int j = 0; j < MT; ++j) acc[n][j] = mfma16(xa[j], bf, acc[n][j]);
        }
      }
    }
  };
  // Half a k-tile of x is staged while the half before it is multiplied: registers -> LDS one half ahead, memory ->
  // registers three halves ahead (one where the accumulators leave no room).  (A wavefront's LDS operations execute in
  // order, so its two buffers need no waits.)
  if constexpr (ROLL) {
    stage_from(xr0, gr0, 0);
    stage_from(xr0, gr0, 1);
    for (int i = 0; i < nk; i += WD) {
#pragma unroll
      for (int d = 0; d < WD; ++d) {
        const bool live = d == 0 || i + d < nk;
        half8 xa[4];
        float4v sx[4];
        if (live) {
#pragma unroll
          for (int s = 0; s < 4; ++s) xa[s] = x_fragment(s >> 1, s, 0);
#pragma unroll
          for (int s = 0; s < 4; ++s) sx[s] = x_sum(xa[s]);
        }
#pragma unroll
        for (int n = 0; n < NS; ++n) {
          // (the empty statements pin the tile's arithmetic between its wait and its next request: moved together, the tiles' spill)
          asm volatile("" : "+v"(tt[d][n].lo0));
          if (live) {
#pragma unroll
            for (int s = 0; s < 4; ++s) multiply(acc[n][0], tt[d][n], xa[s], sx[s], s);
          }
          asm volatile("" : "+v"(acc[n][0]));
          __builtin_amdgcn_sched_barrier(0);
          fetch_tile(tt[d][n], n, i + d + WD);
          if (n == NS / 2) {
            stage_x(0);                              // (past the last k-tile: zeros)
            stage_x(1);
            fetch_x(i + d + 2, 0);
            fetch_x(i + d + 2, 1);
            rows_issued();
          }
        }
      }
    }
  } else {
    stage_x(0);
    if constexpr (XH == 2) fetch_x(1, 0);
    else fetch_x(0, 1);
    rows_issued();
    for (int i = 0; i < nk; i += WD) {
#pragma unroll
      for (int d = 0; d < WD; ++d) {
        // (only arithmetic stands under a condition: a load there would cost the counts of the waits)
        const bool live = d == 0 || i + d < nk, next = i + d + 1 < nk;
        if constexpr (RAW) {
          if (live)
#pragma unroll
            for (int n = 0; n < NT; ++n) pl.settle(tt[d][n], n, kmap(i + d));
        }
        if constexpr (XH == 2) {
          if (live) stage_x(1);
          fetch_x(i + d + 1, 1);
          rows_issued();
          if (live) half_step(tt[d], 0);
          if (next) stage_x(0);
          fetch_x(i + d + 2, 0);
          rows_issued();
          if (live) half_step(tt[d], 1);
        } else {
          if (live) half_step(tt[d], 0);
          if (live) stage_x(1);
          fetch_x(i + d + 1, 0);
          rows_issued();
          if (live) half_step(tt[d], 1);
          if (next) stage_x(0);
          fetch_x(i + d + 1, 1);
          rows_issued();
        }
        fetch_w(tt[d], i + d + WD);
        rows_issued();
      }
    }
  }

  // ---- sum over the wavefronts' k-tiles through LDS
  __syncthreads();
  auto park = [&](int at) {
#pragma unroll
    for (int n = 0; n < NS; ++n)
#pragma unroll
      for (int j = 0; j < MT; ++j) *(float4v*)(red + ((at * NS * MT + n * MT + j) * 64 + lane) * 4) = acc[n][j];
  };
  if constexpr (TWO) {
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
  if constexpr (NORM) {
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      float q = ssq[p];
      q += __shfl_xor(q, 1);
      q += __shfl_xor(q, 2);
      q += __shfl_xor(q, 4);
      if (slot == 0) ssq_sh[wave * MT * 16 + 8 * p + srow] = q;
    }
  }
  __syncthreads();

  const bool partial_out = a.splitk > 1;
  constexpr int ITEMS = NT * MT;                     // output tiles of 16 x 16
  for (int it = wave; it < ITEMS; it += NW) {
    const int n = it / MT, j = it % MT;
    const int nt = nb * NT + n;
    float4v v = {0, 0, 0, 0}, u = {0, 0, 0, 0};
#pragma unroll
    for (int w = 0; w < NR; ++w) {
      v += *(const float4v*)(red + ((w * NS * MT + n * MT + j) * 64 + lane) * 4);
      if constexpr (PAIR) u += *(const float4v*)(red + ((w * NS * MT + (NT + n) * MT + j) * 64 + lane) * 4);
    }
    const int col = nt * 16 + r;
    if (nt >= ntiles || col >= a.N) continue;
    float b1 = 0.0f, b2 = 0.0f;
    if (a.bias != nullptr && !partial_out) b1 = (float)((const _Float16*)a.bias)[col];
    if (PAIR && a.bias2 != nullptr && !partial_out) b2 = (float)((const _Float16*)a.bias2)[col];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int mr = 16 * j + 4 * g + q, m = row0 + mr;
      if (mr >= rows) continue;
      float y = v[q], z = u[q];
      if (partial_out) {
        a.partial[((int64_t)sp * a.M + m) * a.N + col] = y;
        if constexpr (PAIR) a.partial[((int64_t)(a.splitk + sp) * a.M + m) * a.N + col] = z;
        continue;
      }
      if (norm) {
        float s2 = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) s2 += ssq_sh[w * MT * 16 + mr];
        const float rs = rsqrtf(s2 / (float)a.K + a.eps);
        y *= rs;
        z *= rs;
      }
      y = act_apply(a.act, y + b1);
      if constexpr (PAIR) y *= z + b2;
      const int64_t oi = (int64_t)m * a.ldo + col;
      if (a.out_type == OUT_F16) {
        if (a.residual) y += load_out<OUT_F16>(a.residual, oi);
        store_out<OUT_F16>(a.out, oi, y);
      } else if (a.out_type == OUT_BF16) {
        if (a.residual) y += load_out<OUT_BF16>(a.residual, oi);
        store_out<OUT_BF16>(a.out, oi, y);
      } else {
        if (a.residual) y += load_out<OUT_F32>(a.residual, oi);
        store_out<OUT_F32>(a.out, oi, y);
      }
    }
  }
}

template <int QT, int MT, int NT, bool PAIR, bool SHORT = false>
static int gemm_rows_launch_t(const RowsArgs& a, hipStream_t st) {
  constexpr int NS = PAIR ? 2 * NT : NT, lds = rows_lds(MT, NS, ROWS_NW);
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  if constexpr (!SHORT && rows_has_short(QT, MT, NS, PAIR))
    if (a.kt_per_split < ROWS_NW) return gemm_rows_launch_t<QT, MT, NT, PAIR, true>(a, st);
  auto k = gemm_rows_kernel<QT, MT, NT, PAIR, SHORT>;
  if (!gemv_allow_lds((const void*)k, lds)) return -101;
  const int nblocks = ((a.N + 15) / 16 + NT - 1) / NT;
  hipLaunchKernelGGL(k, dim3(nblocks, (a.M + MT * 16 - 1) / (MT * 16), a.splitk), dim3(ROWS_NW * 64), lds, st, a.x, a.w, a.w2, a.gamma,
                     a.M, a.N, a.K, a.ldx, a.kt_per_split, a.gamma_offset, a);
  return HIP_CHECK_LAUNCH();
}

// the tilings that exist (the planner in gemm_rows.hip chooses among them)
constexpr bool rows_has(int mt, int nt, bool pair) {
  return pair ? (mt == 1 && nt >= 1 && nt <= 4) || (mt == 2 && (nt >= 1 && nt <= 3)) || (mt == 4 && nt >= 1 && nt <= 3)
              : (mt == 1 && nt >= 1 && nt <= 4) || (mt == 2 && nt >= 1 && nt <= 4) || (mt == 4 && nt >= 1 && nt <= 3);
}
template <int QT, int MT, bool PAIR>
static int gemm_rows_launch_mt(const RowsArgs& a, int nt, hipStream_t st) {
  if constexpr (rows_has(MT, 1, PAIR)) if (nt == 1) return gemm_rows_launch_t<QT, MT, 1, PAIR>(a, st);
  if constexpr (rows_has(MT, 2, PAIR)) if (nt == 2) return gemm_rows_launch_t<QT, MT, 2, PAIR>(a, st);
  if constexpr (rows_has(MT, 3, PAIR)) if (nt == 3) return gemm_rows_launch_t<QT, MT, 3, PAIR>(a, st);
  if constexpr (rows_has(MT, 4, PAIR)) if (nt == 4) return gemm_rows_launch_t<QT, MT, 4, PAIR>(a, st);
  return -4;
}
template <int QT>
static int gemm_rows_launch_qt(const RowsArgs& a, int mt, int nt, hipStream_t st) {
  const bool pair = a.w2 != nullptr;
  if constexpr (QT == Q_Q6_K) {
    if (pair) return -7;
    if (mt == 1) return gemm_rows_launch_mt<QT, 1, false>(a, nt, st);
    if (mt == 2) return gemm_rows_launch_mt<QT, 2, false>(a, nt, st);
    if (mt == 4) return gemm_rows_launch_mt<QT, 4, false>(a, nt, st);
    return -4;
  } else {
  if (mt == 1) return pair ? gemm_rows_launch_mt<QT, 1, true>(a, nt, st) : gemm_rows_launch_mt<QT, 1, false>(a, nt, st);
  if (mt == 2) return pair ? gemm_rows_launch_mt<QT, 2, true>(a, nt, st) : gemm_rows_launch_mt<QT, 2, false>(a, nt, st);
  if (mt == 4) return pair ? gemm_rows_launch_mt<QT, 4, true>(a, nt, st) : gemm_rows_launch_mt<QT, 4, false>(a, nt, st);
  return -4;
  }
}

}  // namespace bigdl
