// Planner and entry point of the few-row low-bit product (kernel: gemm_rows_kernel.h; one instantiation unit per weight
// format: gemm_rows_inst_*.hip).
#include "gemm_rows_kernel.h"
#include "gemm_rows.h"

namespace bigdl {
#define ROWS_FORMATS(X)                                                                                                     \
  X(Q_SYM_INT4, sym_int4) X(Q_ASYM_INT4, asym_int4) X(Q_WOQ_INT4, woq_int4) X(Q_FP4, fp4) X(Q_NF4, nf4)                     \
  X(Q_SYM_INT5, sym_int5) X(Q_ASYM_INT5, asym_int5) X(Q_FP6, fp6) X(Q_SYM_INT8, sym_int8) X(Q_FP8_E4M3, fp8_e4m3)           \
  X(Q_FP8_E5M2, fp8_e5m2) X(Q_Q6_K, q6_k)
#define ROWS_DECLARE(id, name) int gemm_rows_launch_##name(const RowsArgs& a, int mt, int nt, hipStream_t st);
ROWS_FORMATS(ROWS_DECLARE)

static int tile_bytes(int qtype) {
  if (qtype == Q_Q6_K) return 16 * 105;      // half of a 210-byte block a row
  return 256 * (lo_bits_of(qtype) + hi_bits_of(qtype)) + (has_min_of(qtype) ? 256 : 128);
}

RowsPlan rows_plan(int M, int N, int K, int qtype, bool pair, bool may_split) {
  const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  const int mblocks = (M + 16 * mt - 1) / (16 * mt);
  const int tiles = (N + 15) / 16, KT = (K + 127) / 128;
  const int cus = gemv_cu_count();
  const double wrow = (double)tile_bytes(qtype) * KT * (pair ? 2 : 1);
  const double xall = (double)(M < 16 * mt ? M : 16 * mt) * K * 2;
  RowsPlan best = {mt, 0, 1, KT, 1};
  double best_us = 0.0;
  for (int nt = 1; nt <= 4; ++nt) {
    if (!rows_has(mt, nt, pair)) continue;
    for (int sk = 1; sk <= (may_split ? 4 : 1); ++sk) {
      if (sk > 1 && KT / sk < 2 * ROWS_NW) break;
      const int per = (KT + sk - 1) / sk;
      if ((KT + per - 1) / per != sk) continue;
      const int blocks = (tiles + nt - 1) / nt * sk * mblocks;
      const int turns = (blocks + cus - 1) / cus;
      // (what compares the tilings with each other; the time itself is rows_us of gemm_lowbit.hip)
      const double us = turns * (xall / sk / 57e3 + nt * wrow / sk / 20e3) + (sk > 1 ? 6.0 : 0.0);
      if (best.nt == 0 || us < best_us) {
        best = {mt, nt, sk, per, turns};
        best_us = us;
      }
    }
  }
  return best;
}

int rows_launch(const RowsArgs& a, const RowsPlan& p, int qtype, hipStream_t st) {
  switch (qtype) {
#define ROWS_CASE(id, name) case id: return gemm_rows_launch_##name(a, p.mt, p.nt, st);
    ROWS_FORMATS(ROWS_CASE)
    default: return -2;
  }
}
}  // namespace bigdl

using namespace bigdl;

// (q6_k: w holds the file's blocks row by row, K % 256 == 0, 4-byte aligned, no w2.)
// y = act(norm?(x) W^T + bias) [* (x W2^T + bias2)] [+ residual] on an explicit tiling (nt weight tiles per workgroup, K
// split over splitk workgroups); nt = 0: the planner's, unsplit.  workspace: fp32, splitk * M * N (twice that with w2) when split: the partial
// sums stay there, nothing is written to out.  For tests and measurements; the public products choose by themselves.
extern "C" int bigdl_gemm_rows(const void* x, const void* w, const void* w2, void* out, const void* bias, const void* bias2,
                               const void* residual, const void* gamma, float gamma_offset, float eps, float* workspace,
                               int64_t workspace_floats, int M, int N, int K, int ldx, int ldo, int qtype, int act, int out_type,
                               int nt, int splitk, hipStream_t stream) {
  qtype = t16_kernel_qtype(qtype);
  const bool raw = qtype == Q_Q6_K;
  if (raw && ((K & 255) || w2 != nullptr)) return -1;
  if (M <= 0 || N <= 0 || K <= 0 || (K & 31) || !rows_ok(x, ldx) || ((uintptr_t)w & (raw ? 3 : 15)) || (w2 && ((uintptr_t)w2 & 15)) || splitk < 1) return -1;
  if (gamma != nullptr && (((uintptr_t)gamma & 15) || M > 16 || splitk > 1)) return -7;
  if (out_type < 0 || out_type > 2) return -3;
  RowsPlan p = rows_plan(M, N, K, qtype, w2 != nullptr, false);
  if (nt > 0) {
    const int KT = (K + 127) / 128;
    p.nt = nt;
    p.kt_per_split = (KT + splitk - 1) / splitk;
    p.splitk = (KT + p.kt_per_split - 1) / p.kt_per_split;
  }
  if (p.splitk > 1 && (workspace == nullptr || workspace_floats < (w2 ? 2 : 1) * (int64_t)p.splitk * M * N)) return -5;
  RowsArgs a = {};
  a.x = (const _Float16*)x; a.w = w; a.w2 = w2; a.out = out; a.partial = workspace; a.bias = bias; a.bias2 = bias2;
  a.residual = residual; a.gamma = (const _Float16*)gamma; a.gamma_offset = gamma_offset; a.eps = eps;
  a.M = M; a.N = N; a.K = K; a.ldx = ldx; a.ldo = ldo; a.act = act; a.out_type = out_type;
  a.splitk = p.splitk; a.kt_per_split = p.kt_per_split;
  if (raw && nt <= 0 && gemv_q6k_takes(a)) return gemv_q6k_launch(a, stream);
  return rows_launch(a, p, qtype, stream);
}
