// Planner and entry points of the low-bit product on x in fragment order (kernel: gemm_frag_kernel.h; one instantiation unit per
// weight format: gemm_frag_inst_*.hip), and the pass that puts x into that order.
#include "gemm_frag_kernel.h"
#include "gemm_frag.h"
#include <math.h>

namespace bigdl {
#define FRAG_FORMATS(X)                                                                                                     \
  X(Q_SYM_INT4, sym_int4) X(Q_ASYM_INT4, asym_int4) X(Q_WOQ_INT4, woq_int4) X(Q_FP4, fp4) X(Q_NF4, nf4)                     \
  X(Q_SYM_INT5, sym_int5) X(Q_ASYM_INT5, asym_int5) X(Q_FP6, fp6) X(Q_SYM_INT8, sym_int8) X(Q_FP8_E4M3, fp8_e4m3)           \
  X(Q_FP8_E5M2, fp8_e5m2)
#define FRAG_DECLARE(id, name) int gemm_frag_launch_##name(const FragArgs& a, int mt, int ns, hipStream_t st);
FRAG_FORMATS(FRAG_DECLARE)

// x [M, K] (fp16, or bf16: rounded to fp16) -> fragments of 16 rows x 32 columns, [k / 32][row / 16][lane][8 halves]: lane (g, r)
// of a fragment holds row r, columns 8 g .. 8 g + 7.  Rows past M and columns past K are zero.  One wavefront a fragment: 16
// pieces of 64 bytes in, 1 KiB out.
__global__ __launch_bounds__(256) void frag_pack_kernel(const void* x, _Float16* xp, int M, int K, int ldx, int mt_all, int frags, int bf16) {
  const int f = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (f >= frags) return;
  const int k = f / mt_all * 32 + (lane >> 4) * 8, m = f % mt_all * 16 + (lane & 15);
  half8 v = {0, 0, 0, 0, 0, 0, 0, 0};
  if (m < M && k < K) {
    const uint4v raw = *(const uint4v*)((const uint16_t*)x + (int64_t)m * ldx + k);
    v = __builtin_bit_cast(half8, raw);
    if (bf16) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[2 * i] = (_Float16)__uint_as_float(raw[i] << 16);
        v[2 * i + 1] = (_Float16)__uint_as_float(raw[i] & 0xffff0000u);
      }
    }
  }
  *(half8*)(xp + ((int64_t)f * 64 + lane) * 8) = v;
}
int frag_pack(const void* x, void* xp, int M, int K, int ldx, bool bf16, hipStream_t st) {
  const int mt = (M + 15) / 16, frags = (K + 127) / 128 * 4 * mt;
  hipLaunchKernelGGL(frag_pack_kernel, dim3((frags + 3) / 4), dim3(256), 0, st, x, (_Float16*)xp, M, K, ldx, mt, frags, (int)bf16);
  return HIP_CHECK_LAUNCH();
}

// Time of a tiling in us: a + turns * (turn + tile * mt * ns + k-tiles * (x * mt + w * ns + xw * mt * ns)) + load * k-tiles * mem * ns +
// part * (million partial sums written); load: workgroups a CU, turns: that number rounded up.  tile is the exchange of the sums and the
// stores, which a short K does not hide; mem is the memory's share of the weights, all workgroups' together.  Fitted per format to 20000
// launches on one MI355X: random shapes from 512 x 256 to 30000 x 14000 and pairs, 33 to 2048 rows, every tiling, 1 / 2 / 4 splits of
// K, caches flushed of the weights.  Off by 6 % on average, by more than 12 % for one launch in ten.  Without those two terms K below 1536
// came out up to half too fast: 437 rows of 11616 x 640 nf4 20 us, measured 37.
struct FragCost { float a, turn, tile, x, w, xw, mem, part; };
static FragCost frag_cost(int qtype) {
  switch (qtype) {
    case Q_SYM_INT4: return {3.01f, 1.26f, 0.219f, 0.0251f, 0.0192f, 0.0041f, 0.0184f, 0.72f};
    case Q_ASYM_INT4: case Q_WOQ_INT4: return {2.97f, 1.66f, 0.231f, 0.0270f, 0.0273f, 0.0033f, 0.0168f, 0.71f};
    case Q_FP4: return {2.98f, 1.27f, 0.226f, 0.0193f, 0.0254f, 0.0059f, 0.0184f, 0.67f};
    case Q_NF4: return {2.84f, 1.40f, 0.219f, 0.0146f, 0.0383f, 0.0069f, 0.0195f, 0.80f};
    case Q_SYM_INT5: return {2.76f, 1.43f, 0.240f, 0.0165f, 0.0490f, 0.0056f, 0.0194f, 0.64f};
    case Q_ASYM_INT5: return {3.08f, 1.29f, 0.257f, 0.0182f, 0.0547f, 0.0044f, 0.0221f, 0.94f};
    case Q_FP6: return {2.58f, 1.77f, 0.244f, 0.0098f, 0.0759f, 0.0064f, 0.0204f, 0.52f};
    case Q_SYM_INT8: return {2.77f, 1.76f, 0.227f, 0.0307f, 0.0344f, 0.0023f, 0.0208f, 0.42f};
    case Q_FP8_E4M3: return {2.93f, 1.52f, 0.240f, 0.0253f, 0.0419f, 0.0039f, 0.0199f, 0.37f};
    default: return {2.70f, 1.92f, 0.217f, 0.0337f, 0.0299f, 0.0016f, 0.0198f, 0.43f};        // fp8_e5m2
  }
}

FragPlan frag_plan(int M, int N, int K, int qtype, bool pair, bool may_split, bool sums_left) {
  const int KT = (K + 127) / 128, tiles = (N + 15) / 16, mt_all = (M + 15) / 16;
  FragPlan best = {0, 0, 1, KT, 1e30};
  if (frag_halves(M, K) * 2 >= ROWS_OUT) return best;
  const FragCost c = frag_cost(qtype);
  const int cus = gemv_cu_count();
  for (int mt = 3; mt <= 8; ++mt) {
    const int mblocks = (mt_all + mt - 1) / mt;
    for (int ns = 2; ns <= 8; ++ns) {
      if (!frag_has(mt, ns) || (pair && (ns & 1))) continue;
      const int64_t blocks = (int64_t)((tiles + (pair ? ns / 2 : ns) - 1) / (pair ? ns / 2 : ns)) * mblocks;
      for (int sk = 1; sk <= (may_split ? 4 : 1); sk *= 2) {
        const int per = (KT + sk - 1) / sk;
        if (sk > 1 && (KT < 8 * sk || (KT + per - 1) / per != sk)) break;
        const double load = (double)(blocks * sk) / cus;
        double us = c.a + ceil(load) * (c.turn + c.tile * mt * ns + per * (c.x * mt + c.w * ns + c.xw * mt * ns)) + load * per * c.mem * ns;
        // partial sums, and the launch that adds them up: 4 us on the GPU.  Where the host is behind it costs 3.5 us there, so a split has
        // to be ahead by that much (34 rows of 2048 x 5632 nf4 in a prompt of two layers: 282 us a pass, without the split 273)
        // Sums that are left to the norm behind cost what it takes to write and read them, and have to be 4 % ahead, for
        // the estimate's own error.  Of 400 random products of 33 - 512 rows in six formats that this splits, with their norm, none is more
        // than 1 % slower than whole, 17 % faster on average (64 x 4096 x 11008 sym_int4 23.1 -> 19.7 us, 77 x 4096 x 14336 asym_int4 29.6 -> 24.7,
        // 36 x 4096 x 14336 23.0 -> 20.1).  Priced at 1.0 us + 0.7 ps with 0.7 of a tile's exchange, 86 of 550 were 2 - 20 % slower than
        // whole (80 x 5120 x 2048 asym_int5 14.5 -> 17.5), nearly all of them whole in 160 - 256 workgroups and split into larger tiles.
        if (sums_left && sk > 1) us = (us + 2.0 + 0.4e-6 * sk * M * N) / 0.96;
        else if (sk > 1) us += 7.5 + 1e-6 * sk * M * N * (c.part + 1.0);
        if (us < best.us) best = {mt, ns, sk, per, us};
      }
    }
  }
  return best;
}

int frag_launch(const FragArgs& a_in, const FragPlan& p, int qtype, hipStream_t st) {
  FragArgs a = a_in;
  const uintptr_t at = (uintptr_t)a.out | (uintptr_t)a.residual;
  a.vec = (a.N & 3) == 0 && (a.ldo & 3) == 0 && (at & (a.out_type == OUT_F32 ? 15 : 7)) == 0;
  switch (qtype) {
#define FRAG_CASE(id, name) case id: return gemm_frag_launch_##name(a, p.mt, p.ns, st);
    FRAG_FORMATS(FRAG_CASE)
    default: return -2;
  }
}
}  // namespace bigdl

using namespace bigdl;

extern "C" int64_t bigdl_frag_halves(int M, int K) { return frag_halves(M, K); }

// K % 8 == 0, rows of x 16-byte aligned; x_type: OUT_F16 or OUT_BF16; xp: bigdl_frag_halves halves, 16-byte aligned
extern "C" int bigdl_frag_pack(const void* x, void* xp, int64_t halves, int M, int K, int ldx, int x_type, hipStream_t stream) {
  if (M <= 0 || K <= 0 || (K & 7) || (ldx & 7) || ((uintptr_t)x & 15) || ((uintptr_t)xp & 15) || halves < frag_halves(M, K)) return -1;
  if (x_type != OUT_F16 && x_type != OUT_BF16) return -3;
  return frag_pack(x, xp, M, K, ldx, x_type == OUT_BF16, stream);
}

// y = act(x W^T + bias) [* (x W2^T + bias2)] [+ residual] of x in fragment order, on an explicit tiling.  workspace: fp32,
// splitk * M * N (twice that with w2) when split: the partial sums stay there, nothing is written to out.  For tests and
// measurements; the public products choose by themselves.
extern "C" int bigdl_gemm_frag(const void* xp, int64_t halves, const void* w, const void* w2, void* out, const void* bias, const void* bias2,
                               const void* residual, float* workspace, int64_t workspace_floats, int M, int N, int K, int ldo,
                               int qtype, int act, int out_type, int mt, int ns, int splitk, hipStream_t stream) {
  qtype = t16_kernel_qtype(qtype);
  if (M <= 0 || N <= 0 || K <= 0 || (K & 31) || ((uintptr_t)xp & 15) || ((uintptr_t)w & 15) || (w2 && ((uintptr_t)w2 & 15)) || splitk < 1 ||
      halves < frag_halves(M, K) || frag_halves(M, K) * 2 >= ROWS_OUT)
    return -1;
  if (out_type < 0 || out_type > 2) return -3;
  const int KT = (K + 127) / 128;
  FragPlan p = {mt, ns, splitk, (KT + splitk - 1) / splitk, 0.0};
  p.splitk = (KT + p.kt_per_split - 1) / p.kt_per_split;
  if (p.splitk > 1 && (workspace == nullptr || workspace_floats < (w2 ? 2 : 1) * (int64_t)p.splitk * M * N)) return -5;
  FragArgs a = {};
  a.xp = (const _Float16*)xp; a.w = w; a.w2 = w2; a.out = out; a.partial = workspace; a.bias = bias; a.bias2 = bias2; a.residual = residual;
  a.M = M; a.N = N; a.K = K; a.mt_all = (M + 15) / 16; a.ldo = ldo; a.act = act; a.out_type = out_type;
  a.splitk = p.splitk; a.kt_per_split = p.kt_per_split;
  return frag_launch(a, p, qtype, stream);
}
