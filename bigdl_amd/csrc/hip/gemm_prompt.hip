// Host entry of the prompt-sized dequant-fused MFMA GEMM (kernel: gemm_prompt_kernel.h; one instantiation unit per weight
// format: gemm_prompt_inst_*.hip): tile configuration / K-split planning and the C ABI.
#include "gemm_prompt_kernel.h"
#include <stdlib.h>

namespace bigdl {

int gemm_launch_reduce(const GemmArgs& a, hipStream_t stream);      // gemm_lowbit.hip: split-K reduce / epilogue

#define PROMPT_DECL(name) int gemm_prompt_launch_##name(const GemmArgs& a, int cfg, hipStream_t st);
PROMPT_DECL(sym_int4) PROMPT_DECL(asym_int4) PROMPT_DECL(woq_int4) PROMPT_DECL(fp4) PROMPT_DECL(nf4) PROMPT_DECL(sym_int5)
PROMPT_DECL(asym_int5) PROMPT_DECL(fp6) PROMPT_DECL(sym_int8) PROMPT_DECL(fp8_e4m3) PROMPT_DECL(fp8_e5m2)
#undef PROMPT_DECL

static int prompt_dispatch(const GemmArgs& a, int qtype, int cfg, hipStream_t st) {
  switch (qtype) {
    case Q_SYM_INT4: return gemm_prompt_launch_sym_int4(a, cfg, st);
    case Q_ASYM_INT4: return gemm_prompt_launch_asym_int4(a, cfg, st);
    case Q_WOQ_INT4: return gemm_prompt_launch_woq_int4(a, cfg, st);
    case Q_FP4: return gemm_prompt_launch_fp4(a, cfg, st);
    case Q_NF4: return gemm_prompt_launch_nf4(a, cfg, st);
    case Q_SYM_INT5: return gemm_prompt_launch_sym_int5(a, cfg, st);
    case Q_ASYM_INT5: return gemm_prompt_launch_asym_int5(a, cfg, st);
    case Q_FP6: return gemm_prompt_launch_fp6(a, cfg, st);
    case Q_SYM_INT8: return gemm_prompt_launch_sym_int8(a, cfg, st);
    case Q_FP8_E4M3: return gemm_prompt_launch_fp8_e4m3(a, cfg, st);
    case Q_FP8_E5M2: return gemm_prompt_launch_fp8_e5m2(a, cfg, st);
    default: return -2;
  }
}

// Tile configurations (gemm_prompt_launch<QT> instantiates them in this order).  us per 128-deep k tile and us around the loop (first
// requests, epilogue) of 256 tiles at once, one a CU, fitted with the constants below to 2500 launches of 310 random products (M 257 -
// 8000, N 1024 - 14336, K 512 - 14336, pairs among them, weights out of the caches) in 10 formats: off by 4 % on average for one launch
// by itself.  Launches in a row, as a prompt runs them, are slower (power): of 332 other random products in 6 formats the estimate is 5 %
// low in the middle, 16 % above 2000 rows (1024 x 12288 x 4096 71 for 90 us); the plan taken is then 0.5 % slower than the fastest of all
// on average, 11 % at most.  With the first three configurations alone the fastest is 4 % slower: 1024 x 8192 x 8192 is 119 us in
// 256 x 128 tiles, 124 in 256 x 256 with 2 K splits; 1696 x 6544 x 4736 87 in 192 x 256, 96 in 256 x 192.  128 x 256, 192 x 192 and
// 128 x 192 tiles were measured too: 0.1 % on average.
struct PromptCfg { int bm, bn; float kt_us, tile_us; };
static const PromptCfg kPromptCfgs[PROMPT_NCFG] = {{256, 256, 2.285f, 6.80f}, {256, 192, 1.986f, 5.78f}, {128, 128, 0.806f, 2.46f},
                                                   {256, 128, 1.407f, 4.53f}, {192, 256, 1.853f, 5.72f}, {192, 128, 1.210f, 3.86f}};
// time of a k tile against the mean of the formats that plans are made with (the size of their slabs is asked for without a format; with
// the format's own the plan of the 332 products is 0.6 % slower than the fastest)
constexpr double PLAN_FMT = 1.1;

struct PromptPlan { int cfg, splitk, kt_per_split; double us; };
static int g_force_cfg = -1, g_force_sk = 0;         // bigdl_gemm_prompt_force (tests / sweeps)

// Turns of 256 tiles, each its k tiles and its first requests and epilogue; K splits add the fp32 slabs' traffic and the reduce launch.
// 128 x 128 tiles run two to a CU where there are more than 256 (a lone one is 1.24 times as long, not half as long, as two).
static double plan_us(int M, int N, bool pair, int cfg, int splitk, int kt_per_split, double fmt) {
  const PromptCfg& pc = kPromptCfgs[cfg];
  const int bno = pair ? pc.bn / 2 : pc.bn;
  const int64_t tiles = (int64_t)((M + pc.bm - 1) / pc.bm) * ((N + bno - 1) / bno), turns = (tiles * splitk + 255) / 256;
  const double lone = pc.bm == 128 && turns == 1 ? 1.24 : 1.0;
  double us = 1.3 + (double)turns * (pc.kt_us * (pair ? 1.02 : 1.0) * fmt * lone * kt_per_split + pc.tile_us * (pair ? 1.15 : 1.0));
  if (splitk > 1) us += 5.2 + 1.07e-6 * splitk * (double)M * N;
  return us;
}

// The fastest plan by its estimated time.
// pair: the gate / up form (two products per output column: blocks cover bn / 2 output columns, no K split)
// forced_cfg >= 0, forced_sk > 0: only plans of these
static PromptPlan prompt_plan_of(int M, int N, int K, bool pair, int forced_cfg, int forced_sk) {
  const int KT = K >> 7;
  PromptPlan best = {0, 1, KT, 1e300};
  for (int c = 0; c < PROMPT_NCFG; ++c) {
    if (forced_cfg >= 0 && c != forced_cfg) continue;
    for (int sk = 1; sk <= (pair ? 1 : 8); ++sk) {
      if (forced_sk ? sk != forced_sk : (sk > 1 && KT / sk < 6)) continue;
      if (sk > KT) continue;
      const int per = (KT + sk - 1) / sk, rsk = (KT + per - 1) / per;
      const double us = plan_us(M, N, pair, c, rsk, per, PLAN_FMT);
      // (equal within the estimate: the earlier configuration, the larger tile)
      if (us < (best.cfg == c ? 1.0 : 0.985) * best.us) best = {c, rsk, per, us};
    }
  }
  return best;
}
static PromptPlan prompt_plan(int M, int N, int K, bool pair = false) {
  static const int env_cfg = getenv("BIGDL_PROMPT_CFG") ? atoi(getenv("BIGDL_PROMPT_CFG")) : -1;
  static const int env_sk = getenv("BIGDL_PROMPT_SPLITK") ? atoi(getenv("BIGDL_PROMPT_SPLITK")) : 0;
  return prompt_plan_of(M, N, K, pair, g_force_cfg >= 0 ? g_force_cfg : env_cfg, g_force_sk > 0 ? g_force_sk : env_sk);
}

// The time in us, in this format, of the plan that is launched where nothing forces another (callers remember the choice by the product's
// sizes), for the choice between this kernel and others at 257 - 512 rows.  Large tiles of many splits are 10 - 15 % over the estimate: that
// is counted here, but not in the choice of the plan (of the 332 products above it would be 0.8 % behind the fastest instead of 0.5:
// 512 x 4096 x 11008 59.3 us in four splits of 256 x 128, 63.6 in those of 128 x 128 that it would take).
double prompt_us(int M, int N, int K, int qtype, bool pair) {
  double fmt = 1.0;                                    // sym_int4
  switch (qtype) {
    case Q_ASYM_INT4: case Q_WOQ_INT4: fmt = 1.08; break;
    case Q_FP4: fmt = 1.12; break;
    case Q_NF4: fmt = 1.26; break;
    case Q_SYM_INT5: fmt = 1.26; break;
    case Q_ASYM_INT5: fmt = 1.30; break;
    case Q_FP6: fmt = 1.39; break;
    case Q_SYM_INT8: fmt = 1.12; break;
    case Q_FP8_E4M3: fmt = 1.16; break;
    case Q_FP8_E5M2: fmt = 1.08; break;
    default: break;
  }
  const PromptPlan p = prompt_plan_of(M, N, K, pair, -1, 0);
  return (p.splitk >= 4 && p.cfg != 2 ? 1.12 : 1.0) * plan_us(M, N, pair, p.cfg, p.splitk, p.kt_per_split, fmt);
}

// Splits of K whose sums are left to the norm that follows (1: none), and the product that writes them, [splits][M][N] fp32.  The plan is the
// one without a norm: what is split there saves its reduce launch and a pass over the result, with its norm 7 % on average, 2 to 18 (150 random
// products of 257 - 8000 rows, four formats; 1024 x 4096 x 11008 sym_int4 109.1 -> 102.5 us).  What is whole there stays whole: 90 random products of 513 - 8000 rows
// that a price of left sums (0.5 us + 0.9 ps an element and split) would split were 1.2 % slower on average, 39 of them by 2 - 17 % (844 x
// 5120 x 4096 sym_int8 57.4 -> 63.3), and took slabs of up to 150 MB.
int prompt_parts(int M, int N, int K) { return prompt_plan(M, N, K).splitk; }
int prompt_parts_launch(const void* x, const void* w, float* partial, int M, int N, int K, int ldx, int qtype, hipStream_t st) {
  GemmArgs a = {};
  const PromptPlan pl = prompt_plan(M, N, K);
  a.x = (const _Float16*)x; a.w = w; a.partial = partial; a.M = M; a.N = N; a.K = K; a.ldx = ldx; a.ldo = N; a.out_type = OUT_F16;
  a.splitk = pl.splitk; a.kt_per_split = pl.kt_per_split;
  return prompt_dispatch(a, qtype, pl.cfg, st);
}

// the staged 16-bit epilogue covers this output; otherwise one fp32 slab + the reduce kernel
static bool prompt_staged_ok(int N, int ldo, int out_type, const void* out, const void* residual) {
  return out_type != OUT_F32 && (N & 7) == 0 && (ldo & 7) == 0 && (((uintptr_t)out | (uintptr_t)residual) & 15) == 0;
}

}  // namespace bigdl

using namespace bigdl;

extern "C" int bigdl_gemm_prompt_supported(int qtype, int K) {
  qtype = t16_kernel_qtype(qtype);
  return is_t16(qtype) && K >= 256 && (K & 127) == 0;
}

// fp32 slabs of M x N floats the call below needs as workspace (0: none)
extern "C" int bigdl_gemm_prompt_slabs(int M, int N, int K, int ldo, int out_type, int out_aligned16) {
  const PromptPlan pl = prompt_plan(M, N, K);
  if (pl.splitk > 1) return pl.splitk;
  const bool staged = out_type != OUT_F32 && (N & 7) == 0 && (ldo & 7) == 0 && out_aligned16;
  return staged ? 0 : 1;
}

// cfg >= 0 / splitk > 0 pin the tile configuration / K splits of the following calls (-1 / 0: planned)
extern "C" void bigdl_gemm_prompt_force(int cfg, int splitk) {
  g_force_cfg = cfg < PROMPT_NCFG ? cfg : -1;
  g_force_sk = splitk;
}

extern "C" int bigdl_gemm_prompt_plan(int M, int N, int K, int* cfg, int* splitk) {
  const PromptPlan pl = prompt_plan(M, N, K);
  if (cfg) *cfg = pl.cfg;
  if (splitk) *splitk = pl.splitk;
  return 0;
}

// the estimate that the choice of the kernel goes by, for its tests
extern "C" double bigdl_gemm_prompt_us(int M, int N, int K, int qtype, int pair) {
  return prompt_us(M, N, K, t16_kernel_qtype(qtype), pair != 0);
}

// Gate / up pair in one launch: out[M, N] = act(x W^T + bias) * (x W2^T + bias2), both weights [N, K] of one format,
// N % 16 == 0; 16-bit output with N % 8 == 0, ldo % 8 == 0 and a 16-byte aligned out (the staged epilogue; -7 otherwise).
extern "C" int bigdl_gemm_prompt_pair(const void* x, const void* w, const void* w2, void* out, const void* bias,
                                      const void* bias2, int M, int N, int K, int ldx, int ldo, int qtype, int act,
                                      int out_type, hipStream_t stream) {
  qtype = t16_kernel_qtype(qtype);
  if (M <= 0 || N <= 0 || (N & 15) || K < 256 || (K & 127) || (ldx & 7) || ((uintptr_t)x & 15) || ((uintptr_t)w & 15) ||
      w2 == nullptr || ((uintptr_t)w2 & 15))
    return -1;
  if ((bias != nullptr && ((uintptr_t)bias & 7)) || (bias2 != nullptr && ((uintptr_t)bias2 & 7))) return -1;
  if (out_type != OUT_F16 && out_type != OUT_BF16) return -3;
  if (!prompt_staged_ok(N, ldo, out_type, out, nullptr)) return -7;
  if ((int64_t)M * ldx >= (1ll << 31)) return -6;
  GemmArgs a = {};
  a.x = (const _Float16*)x; a.w = w; a.w2 = w2; a.out = out; a.bias = bias; a.bias2 = bias2;
  a.M = M; a.N = N; a.K = K; a.ldx = ldx; a.ldo = ldo; a.act = act; a.out_type = out_type;
  const PromptPlan pl = prompt_plan(M, N, K, true);
  a.splitk = 1; a.kt_per_split = K >> 7;
  return prompt_dispatch(a, qtype, pl.cfg, stream);
}

// x fp16 [M, ldx] (ldx % 8 == 0, 16-byte aligned), K % 128 == 0.  workspace: fp32, >= slabs * M * N floats.
extern "C" int bigdl_gemm_prompt(const void* x, const void* w, void* out, const void* bias, const void* residual,
                                 float* workspace, int64_t workspace_floats, int M, int N, int K, int ldx, int ldo,
                                 int qtype, int act, int out_type, hipStream_t stream) {
  qtype = t16_kernel_qtype(qtype);
  if (M <= 0 || N <= 0 || K < 256 || (K & 127) || (ldx & 7) || ((uintptr_t)x & 15) || ((uintptr_t)w & 15)) return -1;
  if (bias != nullptr && ((uintptr_t)bias & 7)) return -1;
  if (out_type < 0 || out_type > 2) return -3;
  if ((int64_t)M * ldx >= (1ll << 31)) return -6;
  GemmArgs a = {};
  a.x = (const _Float16*)x; a.w = w; a.out = out; a.bias = bias; a.residual = residual; a.partial = workspace;
  a.M = M; a.N = N; a.K = K; a.ldx = ldx; a.ldo = ldo; a.act = act; a.out_type = out_type;
  const PromptPlan pl = prompt_plan(M, N, K);
  a.splitk = pl.splitk; a.kt_per_split = pl.kt_per_split;
  a.force_partial = (a.splitk == 1 && !prompt_staged_ok(N, ldo, out_type, out, residual)) ? 1 : 0;
  const bool partial = a.splitk > 1 || a.force_partial;
  if (partial && (workspace == nullptr || workspace_floats < (int64_t)a.splitk * M * N)) return -5;
  const int rc = prompt_dispatch(a, qtype, pl.cfg, stream);
  if (rc != 0 || !partial) return rc;
  return gemm_launch_reduce(a, stream);
}
