// Host entry points of the dequant-fused MFMA GEMM (kernel: gemm_kernel.h; one instantiation unit per weight
// format: gemm_inst_*.hip), its split-K reduce/epilogue kernel and the device-side block table of the grouped
// (mixture-of-experts) form.
#include "gemm_kernel.h"
#include "gemm_rows_kernel.h"
#include "gemm_rows.h"
#include "gemm_frag_kernel.h"
#include "gemm_frag.h"
#include <math.h>
#include <stdlib.h>

namespace bigdl {
int gemm_launch_sym_int4(const GemmArgs& a, int bm, int bn, int mblocks, hipStream_t st);
int gemm_launch_asym_int4(const GemmArgs& a, int bm, int bn, int mblocks, hipStream_t st);
int gemm_launch_woq_int4(const GemmArgs& a, int bm, int bn, int mblocks, hipStream_t st);
int gemm_launch_fp4(const GemmArgs& a, int bm, int bn, int mblocks, hipStream_t st);
int gemm_launch_nf4(const GemmArgs& a, int bm, int bn, int mblocks, hipStream_t st);
int gemm_launch_sym_int5(const GemmArgs& a, int bm, int bn, int mblocks, hipStream_t st);
int gemm_launch_asym_int5(const GemmArgs& a, int bm, int bn, int mblocks, hipStream_t st);
int gemm_launch_fp6(const GemmArgs& a, int bm, int bn, int mblocks, hipStream_t st);
int gemm_launch_sym_int8(const GemmArgs& a, int bm, int bn, int mblocks, hipStream_t st);
int gemm_launch_fp8_e4m3(const GemmArgs& a, int bm, int bn, int mblocks, hipStream_t st);
int gemm_launch_fp8_e5m2(const GemmArgs& a, int bm, int bn, int mblocks, hipStream_t st);
double prompt_us(int M, int N, int K, int qtype, bool pair);        // gemm_prompt.hip
int prompt_parts(int M, int N, int K);
int prompt_parts_launch(const void* x, const void* w, float* partial, int M, int N, int K, int ldx, int qtype, hipStream_t st);

// out[m][n] = epilogue(sum_s partial[s][m][n]); pair form: act(first) * second; optional folded RMSNorm factor of the
// row (row_ssq) and sum of squares of the rows written (ssq_out, for the norm folded into the next product).
// V = elements per thread (4: N % 4 == 0, rows of out / residual 8-byte aligned; else 1).  A workgroup covers 256 * V
// consecutive elements; with ssq_out it adds ONE value per row it touches (LDS reduction first: same-address atomics
// from every wavefront of a row cost more than the rest of the kernel).
template <int V>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(GemmArgs a) {
  const int64_t total = (int64_t)a.M * a.N;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
  const bool in = i < total;
  const int64_t ic = in ? i : total - V;
  const int m = (int)(ic / a.N);
  const int n = (int)(ic - (int64_t)m * a.N);
  typedef float fvec __attribute__((ext_vector_type(V)));
  float v[V], u[V];
#pragma unroll
  for (int e = 0; e < V; ++e) v[e] = u[e] = 0.0f;
  // the slabs of up to four splits are requested together: one at a time, every split costs its own memory round
  // trip (8 splits: 8 dependent trips, most of this kernel's time)
  auto gather = [&](float (&acc)[V], const float* base) {
    int s = 0;
    for (; s + 4 <= a.splitk; s += 4) {
      const fvec p0 = *(const fvec*)(base + (int64_t)s * total + ic);
      const fvec p1 = *(const fvec*)(base + (int64_t)(s + 1) * total + ic);
      const fvec p2 = *(const fvec*)(base + (int64_t)(s + 2) * total + ic);
      const fvec p3 = *(const fvec*)(base + (int64_t)(s + 3) * total + ic);
#pragma unroll
      for (int e = 0; e < V; ++e) acc[e] += (p0[e] + p1[e]) + (p2[e] + p3[e]);
    }
    for (; s < a.splitk; ++s) {
      const fvec p = *(const fvec*)(base + (int64_t)s * total + ic);
#pragma unroll
      for (int e = 0; e < V; ++e) acc[e] += p[e];
    }
  };
  gather(v, a.partial);
  if (a.w2 != nullptr) gather(u, a.partial + a.pair_stride);
  const float rs = a.row_ssq != nullptr ? rsqrtf(a.row_ssq[m] / (float)a.K + a.eps) : 1.0f;
  const float rsc = a.row_scale != nullptr ? a.row_scale[m] : 1.0f;
  const int64_t oi = (int64_t)m * a.ldo + n;
  float q = 0.0f;
#pragma unroll
  for (int e = 0; e < V; ++e) {
    float x = v[e] * rs;
    if (a.bias != nullptr) x += (float)((const _Float16*)a.bias)[n + e];
    x = act_apply(a.act, x);
    if (a.w2 != nullptr) {
      float y = u[e] * rs;
      if (a.bias2 != nullptr) y += (float)((const _Float16*)a.bias2)[n + e];
      x *= y;
    }
    x *= rsc;
    if (a.residual) {
      if (a.out_type == OUT_F16) x += load_out<OUT_F16>(a.residual, oi + e);
      else if (a.out_type == OUT_BF16) x += load_out<OUT_BF16>(a.residual, oi + e);
      else x += load_out<OUT_F32>(a.residual, oi + e);
    }
    // what is stored, rounded (the next norm sees the rounded values)
    if (a.out_type == OUT_F16) x = (float)(_Float16)x;
    else if (a.out_type == OUT_BF16) x = bf16_bits_to_f32(f32_to_bf16_bits(x));
    v[e] = x;
    q += x * x;
  }
  if (in) {
    if (a.out_type == OUT_F16) {
      _Float16 h[V];
#pragma unroll
      for (int e = 0; e < V; ++e) h[e] = (_Float16)v[e];
      if constexpr (V == 4) *(uint2v*)((_Float16*)a.out + oi) = *(const uint2v*)h;
      else ((_Float16*)a.out)[oi] = h[0];
    } else if (a.out_type == OUT_BF16) {
#pragma unroll
      for (int e = 0; e < V; ++e) store_out<OUT_BF16>(a.out, oi + e, v[e]);
    } else {
#pragma unroll
      for (int e = 0; e < V; ++e) store_out<OUT_F32>(a.out, oi + e, v[e]);
    }
  }
  if (a.ssq_out != nullptr) {
    __shared__ float part[4];
    __shared__ int rowof[4];
    if (!in) q = 0.0f;
    const int wave = threadIdx.x >> 6;
    const int m_first = __shfl(m, 0), m_last = __shfl(m, 63);
    const bool uniform = m_first == m_last;            // (N % (64 V) == 0 makes every wavefront single-row)
    if (uniform) {
      q = wave_sum(q);
      if ((threadIdx.x & 63) == 0) { part[wave] = q; rowof[wave] = m; }
    } else {
      if (in) unsafeAtomicAdd(a.ssq_out + m, q);
      if ((threadIdx.x & 63) == 0) { part[wave] = 0.0f; rowof[wave] = -1; }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      // merge the wavefronts that share a row: at most one add per row and workgroup
      for (int w = 0; w < 4; ++w) {
        if (rowof[w] < 0) continue;
        float t = part[w];
        for (int y = w + 1; y < 4; ++y)
          if (rowof[y] == rowof[w]) { t += part[y]; rowof[y] = -1; }
        // hardware fp32 add (plain atomicAdd compiles to a compare-and-swap loop)
        unsafeAtomicAdd(a.ssq_out + rowof[w], t);
      }
    }
  }
}

static int launch_reduce(const GemmArgs& a, hipStream_t stream) {
  const int64_t total = (int64_t)a.M * a.N;
  const bool vec = (a.N % 4 == 0) && (a.ldo % 4 == 0) && (((uintptr_t)a.out & 7) == 0) &&
                   (a.residual == nullptr || ((uintptr_t)a.residual & 7) == 0) && (a.pair_stride % 4 == 0) &&
                   (((uintptr_t)a.partial & 15) == 0);
  if (vec) hipLaunchKernelGGL(gemm_splitk_reduce_kernel<4>, dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0, stream, a);
  else hipLaunchKernelGGL(gemm_splitk_reduce_kernel<1>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, stream, a);
  return HIP_CHECK_LAUNCH();
}

int gemm_launch_reduce(const GemmArgs& a, hipStream_t stream) { return launch_reduce(a, stream); }   // gemm_big.hip

// counts[e] rows of expert e, rows sorted by expert -> table of m-blocks of at most bm rows; unused entries get
// expert -1.  One wavefront: E is at most a few hundred.
__global__ void moe_block_table_kernel(const int64_t* counts, int n_experts, int bm, int max_blocks, int* blk_expert,
                                       int* blk_row0, int* blk_rows) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  int b = 0;
  int64_t row = 0;
  for (int e = 0; e < n_experts; ++e) {
    int64_t c = counts[e];
    for (int64_t o = 0; o < c && b < max_blocks; o += bm, ++b) {
      blk_expert[b] = e;
      blk_row0[b] = (int)(row + o);
      blk_rows[b] = (int)min((int64_t)bm, c - o);
    }
    row += c;
  }
  for (; b < max_blocks; ++b) { blk_expert[b] = -1; blk_row0[b] = 0; blk_rows[b] = 0; }
}
}  // namespace bigdl

using namespace bigdl;

static int dispatch(const GemmArgs& a, int qtype, int bm, int bn, int mblocks, hipStream_t st) {
  switch (qtype) {
    case Q_SYM_INT4: return gemm_launch_sym_int4(a, bm, bn, mblocks, st);
    case Q_ASYM_INT4: return gemm_launch_asym_int4(a, bm, bn, mblocks, st);
    case Q_WOQ_INT4: return gemm_launch_woq_int4(a, bm, bn, mblocks, st);
    case Q_FP4: return gemm_launch_fp4(a, bm, bn, mblocks, st);
    case Q_NF4: return gemm_launch_nf4(a, bm, bn, mblocks, st);
    case Q_SYM_INT5: return gemm_launch_sym_int5(a, bm, bn, mblocks, st);
    case Q_ASYM_INT5: return gemm_launch_asym_int5(a, bm, bn, mblocks, st);
    case Q_FP6: return gemm_launch_fp6(a, bm, bn, mblocks, st);
    case Q_SYM_INT8: return gemm_launch_sym_int8(a, bm, bn, mblocks, st);
    case Q_FP8_E4M3: return gemm_launch_fp8_e4m3(a, bm, bn, mblocks, st);
    case Q_FP8_E5M2: return gemm_launch_fp8_e5m2(a, bm, bn, mblocks, st);
    default: return -2;
  }
}

// K splits of the tile kernel.  mblocks: number of row blocks (dense: ceil(M / bm))
static void plan(int mblocks, int bn, int N, int K, int* splitk, int* kt_per_split) {
  const int KT = (K + 127) / 128;
  const int blocks = ((N + bn - 1) / bn) * mblocks;
  int sk = 1;
  static const int target = getenv("BIGDL_GEMM_TARGET") ? atoi(getenv("BIGDL_GEMM_TARGET")) : 256;
  if (blocks < target * 3 / 4) sk = (target + blocks - 1) / blocks;
  sk = sk < 1 ? 1 : sk;
  if (sk > KT / 2) sk = KT / 2 > 0 ? KT / 2 : 1;   // at least two k tiles per split
  const int per = (KT + sk - 1) / sk;
  *kt_per_split = per;
  *splitk = (KT + per - 1) / per;
}

static int pick_bn(int M) {
  (void)M;
  return 128;
}

extern "C" int bigdl_gemm_lowbit_bm(int M) {
  (void)M;
  static const int forced = getenv("BIGDL_GEMM_BM") ? atoi(getenv("BIGDL_GEMM_BM")) : 0;
  if (forced == 64 || forced == 128) return forced;
  // 64-row blocks keep two or more wavefronts per SIMD (170 VGPRs): measured 10-40 % faster than 128-row blocks at
  // every M between 64 and 1024 on the Llama-2-7B projection shapes
  return 64;
}

// What a product of 33 to 256 rows takes on the tile kernel and on the few-row kernel (gemm_rows_kernel.h), in us: the chooser
// below compares the two.  Both models were fitted to 3300 products on one MI355X: 11 formats, 18 shapes from 512 x 2048 to
// 8192 x 28672 and 10 gate / up pairs, 33 to 256 rows, weights from memory.  They are exact to 8 %, worst cases 25 %.
struct DenseCost {
  float kt;                 // tile kernel: us per k-tile of a workgroup with a CU of its own
  float two, three;         // ... times this with 2 / 3 workgroups a CU (asym_int4 and nearly all wider formats: one after the other)
  float rows_kt;            // few-row kernel: us per k-tile and 16-column weight tile of a workgroup
};
static DenseCost dense_cost(int qtype) {
  switch (qtype) {
    case Q_SYM_INT4: return {0.65f, 1.36f, 2.65f, 0.067f};
    case Q_ASYM_INT4: case Q_WOQ_INT4: return {0.90f, 2.0f, 3.3f, 0.072f};
    case Q_FP4: return {0.77f, 1.4f, 2.5f, 0.075f};
    case Q_NF4: return {1.21f, 1.2f, 2.1f, 0.085f};
    case Q_SYM_INT5: return {0.97f, 1.45f, 2.4f, 0.091f};
    case Q_ASYM_INT5: return {1.54f, 1.95f, 3.15f, 0.097f};
    case Q_FP6: return {1.23f, 1.85f, 2.9f, 0.12f};
    case Q_SYM_INT8: return {0.78f, 1.85f, 3.2f, 0.095f};
    case Q_FP8_E4M3: return {0.93f, 1.85f, 3.05f, 0.103f};
    default: return {0.73f, 1.85f, 3.3f, 0.092f};        // fp8_e5m2
  }
}
static double tile_us(const DenseCost& c, int M, int N, int K, bool pair) {
  const int bm = bigdl_gemm_lowbit_bm(M), bn = pick_bn(M), mblocks = (M + bm - 1) / bm * (pair ? 2 : 1);
  int sk, per;
  plan(mblocks, bn, N, K, &sk, &per);
  const double load = (double)((N + bn - 1) / bn) * mblocks * sk / gemv_cu_count();       // workgroups a CU
  double turns = 1.0;
  // (a second workgroup on a few CUs only is hardly felt)
  if (load > 3.0) turns = c.three + 0.25 + 1.13 * (load - 3.0);
  else if (load > 2.0) turns = c.three + 0.25 * (load - 2.0);
  else if (load > 1.0) turns = 1.0 + (c.two - 1.0) * fmin(1.0, 8.0 * (load - 1.0)) + 0.25 * (load - 1.0);
  double us = 12.3 + per * c.kt * turns;
  if (sk > 1 || pair) us += 3.2e-6 * sk * M * N * (pair ? 2 : 1) - 4.2;     // slabs and the reduce launch; the kernel's epilogue shrinks
  return us;
}
static double rows_us(const DenseCost& c, const RowsPlan& p, int K, int qtype, bool pair) {
  const double ktiles = (double)((K + 127) / 128) / p.splitk;
  // (fp6: the pair's kernel spills)
  const double tiles_us = p.nt * (pair ? 2 : 1) * c.rows_kt * (pair && qtype == Q_FP6 ? 1.15 : 1.0);
  return (lo_bits_of(qtype) == 8 ? 5.0 : 6.2) + p.turns * ktiles * (0.112 + tiles_us) + 4.2 * (p.turns - 1) + (p.splitk > 1 ? 3.5 : 0.0);
}

// Which products the few-row kernel takes from the tile kernel: above 64 rows those where it is expected to be ahead by what the
// estimates may be off in its favour.  Measured alone, tile -> few-row kernel, us.  Taken: 64 rows sym_int4
// 12288 x 4096 25.3 -> 16.9, 4096 x 4096 16.3 -> 11.9, pair of 11008 x 4096 33.4 -> 23.1, 4096 x 11008 22.0 -> 20.9 (two K splits);
// 128 rows asym_int4 6144 x 4096 35.6 -> 16.5, pair of 14336 x 4096 77.5 -> 68.2.  Left: a grid of many turns (sym_int4 14336 x 4096:
// 128 rows 32.0 -> 42.7, 256 rows 45.9 -> 72.1; 152064 x 3584, 64 rows 106 -> 172), and a long K that x crosses whole in every
// workgroup (1024 x 14336: 65 rows 16.2 -> 26.9; 4096 x 11008, 192 rows 40.4 -> 54.3).
// Up to 64 rows a pass runs nearly all of its products on the few-row kernel, and a lone product on the tile kernel between them is
// slower than alone (its code is out of the caches by then): in decode steps of 64 sequences the head of 32000 x 4096 (three
// turns) took 38 us alone on the tile kernel, 42 among other tile products and 47 among few-row products, where the few-row
// kernel takes 43; 4 steps of 3 layers 2802 and 2783 us.  So up to three turns stay there.  Up to 32 rows it was never behind.
static bool takes_rows_kernel(int ldx, int M, int N, int K, int qtype, bool pair, RowsPlan* plan) {
  if (M > 256 || !is_t16(qtype) || !rows_ok(nullptr, ldx)) return false;
  *plan = rows_plan(M, N, K, qtype, pair, !pair && M <= 64);
  if (M <= 32 || (M <= 64 && plan->turns <= 3)) return true;
  const DenseCost c = dense_cost(qtype);
  return rows_us(c, *plan, K, qtype, pair) < tile_us(c, M, N, K, pair) * (pair ? 0.90 : 0.94);
}
static int launch_rows(const GemmArgs& a, int qtype, const RowsPlan& p, hipStream_t stream) {
  RowsArgs b = {};
  b.x = a.x; b.w = a.w; b.w2 = a.w2; b.out = a.out; b.partial = a.partial; b.bias = a.bias; b.bias2 = a.bias2; b.residual = a.residual;
  b.M = a.M; b.N = a.N; b.K = a.K; b.ldx = a.ldx; b.ldo = a.ldo; b.act = a.act; b.out_type = a.out_type;
  b.splitk = p.splitk; b.kt_per_split = p.kt_per_split;
  const int rc = rows_launch(b, p, qtype, stream);
  return rc != 0 || p.splitk == 1 ? rc : launch_reduce(a, stream);
}

// The kernel a call runs on and the fp32 scratch it needs: one place for the launches and for the size that callers ask for
struct DensePlan {
  bool rows;                // few-row kernel; otherwise the tile kernel
  RowsPlan r;
  int bm, mblocks, splitk, kt_per_split;
  bool partial;             // the results pass through scratch and the reduce kernel
  int64_t floats;
};
// fold_norm, ssq_out: the tile kernel's forms of gemm_lowbit_ex
static DensePlan dense_plan(int M, int N, int K, int ldx, int qtype, bool pair, bool fold_norm, bool ssq_out) {
  DensePlan p = {};
  p.rows = !fold_norm && !ssq_out && takes_rows_kernel(ldx, M, N, K, qtype, pair, &p.r);
  if (p.rows) {
    p.splitk = p.r.splitk;
    p.kt_per_split = p.r.kt_per_split;
    p.partial = p.splitk > 1;
  } else {
    p.bm = bigdl_gemm_lowbit_bm(M);
    p.mblocks = (M + p.bm - 1) / p.bm;
    plan(p.mblocks * (pair ? 2 : 1), pick_bn(M), N, K, &p.splitk, &p.kt_per_split);
    p.partial = p.splitk > 1 || pair || ssq_out;
  }
  p.floats = p.partial ? (pair ? 2 : 1) * (int64_t)p.splitk * M * N : 0;
  return p;
}
static int launch_dense(GemmArgs& a, const DensePlan& p, int qtype, int64_t workspace_floats, hipStream_t stream) {
  if (p.floats > 0 && (a.partial == nullptr || workspace_floats < p.floats)) return -5;
  a.splitk = p.splitk;
  a.kt_per_split = p.kt_per_split;
  if (p.rows) return launch_rows(a, qtype, p.r, stream);
  a.force_partial = p.partial && p.splitk == 1 ? 1 : 0;
  a.pair_stride = (int64_t)a.splitk * a.M * a.N;
  const int rc = dispatch(a, qtype, p.bm, pick_bn(a.M), p.mblocks, stream);
  return rc != 0 || !p.partial ? rc : launch_reduce(a, stream);
}

// fp32 scratch, in floats, that bigdl_gemm_lowbit (pair, fold_norm, ssq_out = 0) and bigdl_gemm_lowbit_ex need for this call;
// 0: none.  qtype: the format as the caller knows it.
extern "C" int64_t bigdl_gemm_lowbit_workspace(int M, int N, int K, int ldx, int qtype, int pair, int fold_norm, int ssq_out) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  return dense_plan(M, N, K, ldx, t16_kernel_qtype(qtype), pair != 0, fold_norm != 0, ssq_out != 0).floats;
}

// Dense form.  x fp16 [M, ldx] (ldx % 8 == 0, 16-byte aligned), K % 32 == 0.  workspace: see bigdl_gemm_lowbit_workspace.
extern "C" int bigdl_gemm_lowbit(const void* x, const void* w, void* out, const void* bias, const void* residual,
                                 float* workspace, int64_t workspace_floats, int M, int N, int K, int ldx, int ldo,
                                 int qtype, int act, int out_type, hipStream_t stream) {
  qtype = t16_kernel_qtype(qtype);
  if (M <= 0 || N <= 0 || K <= 0 || (K & 31) || (ldx & 7) || ((uintptr_t)x & 15) || ((uintptr_t)w & 15)) return -1;
  if (out_type < 0 || out_type > 2) return -3;
  if ((int64_t)M * ldx >= (1ll << 31)) return -6;
  GemmArgs a = {};
  a.x = (const _Float16*)x; a.w = w; a.out = out; a.bias = bias; a.residual = residual; a.partial = workspace;
  a.M = M; a.N = N; a.K = K; a.ldx = ldx; a.ldo = ldo; a.act = act; a.out_type = out_type;
  return launch_dense(a, dense_plan(M, N, K, ldx, qtype, false, false, false), qtype, workspace_floats, stream);
}

// Which products the kernel on x in fragment order takes: those where it is expected to be ahead of the faster of the others.
//  * Rows: with the pass that orders them, by 5 % for what the estimates may be off.  Up to 64 rows, where little is gained, and below
//    16 us by 3 us more: a call takes the host 13 us, and the second launch up to 3.  Of 6000 random products of 33 to 512 rows, pairs
//    among them, it takes 37 %, and 0.6 % of all are slower by more than 2 % for it (5.6 % by estimates without their tile and mem
//    terms); the mean speed is 1.15 times the former.  Measured, us, before -> with the pass -> x in fragment order already: sym_int4
//    4096 x 4096 at 160 / 256 rows 22.7 -> 16.6 -> 12.7, 23.7 -> 19.1 -> 14.6; sym_int8 4672 x 4544 at 203 rows 37.6 -> 24.1 -> 20.7.  Left:
//    sym_int4 4096 x 4096 at 77 rows 14.6 -> 12.2 -> 9.1, 12288 x 4096 at 64 rows 16.5 -> 18.3 -> 15.4, 14336 x 4096 at 256 rows 45.6 -> 55.1 -> 50.5.
//  * Rows in bf16 need a pass in any case, their conversion: by 5 %.  At 257 - 512 rows too: the prompt way's conversion, 3 - 5 us, is not in
//    its estimate.  Of 158 random products in a row this choice is 0.6 % behind the faster way on average, 20 % at most (all on the prompt
//    kernel: 12 and 72).
//  * x whose producer writes it in that order: in a whole step, against the others with x in rows, it is ahead where both are
//    alike alone (their split sums take a launch more, and they come back to cold code), so up to 256 rows unless it is expected
//    to be 15 % behind.  Steps of 8 layers, us, without it / with 3 % ahead asked for / as here: llama3-8b nf4 33 rows 988 / 896 / 857,
//    q4_k 64 rows 970 / 915 / 871, llama2-7b sym_int4 64 rows 1157 / 1121 / 1074.
//  * Against the prompt kernel (257 - 512 rows) this kernel's estimate is a tenth too high: at 1.08 of its time for rows the choice among
//    90 random products loses 0.4 % on average, 9 % at most (at 0.95 1.6 and 22), of 158 in a row 1.2 and 18; at 1.14 for produced x prompts of 3 layers take, us, at
//    0.95 / 1.14 / 1.3: llama2-7b sym_int4 300 tokens 699 / 699 / 733, 400 809 / 799 / 831, llama3-8b nf4 300 778 / 765 / 779, q4_k 450 887 /
//    893 / 910, tinyllama nf4 300 399 / 370 / 376.
enum XKind { X_ROWS = 0, X_ROWS_BF16 = 1, X_FRAGMENTS = 2, X_PRODUCED = 3 };
static bool takes_frag_kernel(int ldx, int M, int N, int K, int qtype, bool pair, int x_kind, bool out_frags, FragPlan* plan) {
  if (M <= 32 || !is_t16(qtype)) return false;
  // (rows that bigdl_gemm_frag_dense refuses: the callers' other ways take them as they are, or 256 at a time)
  if (x_kind < X_FRAGMENTS && ((ldx & 7) || (int64_t)M * ldx >= (1ll << 31))) return false;
  *plan = frag_plan(M, N, K, qtype, pair, !pair);
  if (plan->ns == 0) return false;
  if (x_kind == X_FRAGMENTS) return true;
  if (M > FRAG_MAX_ROWS) return false;
  double other;
  const bool prompt = M > 256 && K >= 256 && (K & 127) == 0;
  if (prompt) {
    if (M > 512) return false;                         // (what the estimates cover)
    other = prompt_us(M, N, K, qtype, pair);
  } else {
    const DenseCost c = dense_cost(qtype);
    const int rows = M < 256 ? M : 256;                // (callers pass more rows 256 at a time)
    RowsPlan r;
    other = takes_rows_kernel(ldx, rows, N, K, qtype, pair, &r) ? rows_us(c, r, K, qtype, pair) : tile_us(c, rows, N, K, pair);
    other *= (M + 255) / 256;
  }
  if (x_kind == X_ROWS) return plan->us + frag_pack_us(M, K) + (M <= 64 || other < 16.0 ? 3.0 : 0.0) < (prompt ? 1.08 : 0.95) * other;
  if (x_kind == X_ROWS_BF16) return plan->us < 0.95 * other;
  return plan->us - (out_frags ? frag_pack_us(M, N) : 0.0) < other * (prompt ? 1.14 : 1.15);
}

// Whether the kernel on x in fragment order is the one for this product.  x_kind 0: fp16 rows; 1: bf16 rows; 2: x in that order already
// (whether it can be multiplied at all); 3: x that its producer writes in that order if so.  out_frags (with 3): the result of a pair
// goes out in that order too, to a product that saves its pass.
extern "C" int bigdl_gemm_lowbit_frag(int M, int N, int K, int ldx, int qtype, int pair, int x_kind, int out_frags) {
  if (M <= 0 || N <= 0 || K <= 0 || (K & 31) || x_kind < 0 || x_kind > X_PRODUCED) return 0;
  FragPlan p;
  return takes_frag_kernel(ldx, M, N, K, t16_kernel_qtype(qtype), pair != 0, x_kind, out_frags != 0, &p) ? 1 : 0;
}

// fp32 scratch, in floats, of the call below: x in fragment order (unless it comes so) and the partial sums of a split K
extern "C" int64_t bigdl_gemm_frag_workspace(int M, int N, int K, int qtype, int pair, int x_kind) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const FragPlan p = frag_plan(M, N, K, t16_kernel_qtype(qtype), pair != 0, !pair);
  return (x_kind == X_FRAGMENTS ? 0 : frag_halves(M, K) / 2) + (p.splitk > 1 ? (int64_t)p.splitk * M * N : 0);
}

// y = act(x W^T + bias) [* (x W2^T + bias2)] [+ residual] on the kernel on x in fragment order.  x_kind 0: x fp16 [M, ldx] (ldx % 8 == 0,
// 16-byte aligned); 1: bf16 rows, rounded to fp16; 2: fp16 in fragment order (ldx is not looked at).  K % 32 == 0.  out_type 3 (pairs,
// N % 128 == 0, no residual): fp16 in fragment order; rows past M of its last row tile are left as they are, they reach only rows of
// a product that are not stored.
extern "C" int bigdl_gemm_frag_dense(const void* x, const void* w, const void* w2, void* out, const void* bias, const void* bias2,
                                     const void* residual, float* workspace, int64_t workspace_floats, int M, int N, int K, int ldx,
                                     int ldo, int qtype, int act, int out_type, int x_kind, hipStream_t stream) {
  qtype = t16_kernel_qtype(qtype);
  if (M <= 0 || N <= 0 || K <= 0 || (K & 31) || ((uintptr_t)x & 15) || ((uintptr_t)w & 15) || !is_t16(qtype)) return -1;
  if (x_kind != X_FRAGMENTS && (ldx & 7)) return -1;
  if (x_kind != X_FRAGMENTS && (int64_t)M * ldx >= (1ll << 31)) return -6;
  if (w2 != nullptr && ((uintptr_t)w2 & 15)) return -1;
  if (out_type == OUT_FRAG && (w2 == nullptr || residual != nullptr || (N & 127) || ((uintptr_t)out & 15))) return -1;
  if (out_type < 0 || out_type > OUT_FRAG || x_kind < 0 || x_kind > X_FRAGMENTS) return -3;
  const FragPlan p = frag_plan(M, N, K, qtype, w2 != nullptr, w2 == nullptr);
  if (p.ns == 0) return -6;
  const int64_t xfloats = x_kind == X_FRAGMENTS ? 0 : frag_halves(M, K) / 2;
  const int64_t floats = xfloats + (p.splitk > 1 ? (int64_t)p.splitk * M * N : 0);
  if (floats > 0 && (workspace == nullptr || workspace_floats < floats)) return -5;
  if ((uintptr_t)workspace & 15) return -1;
  FragArgs b = {};
  b.xp = (const _Float16*)x;
  if (xfloats > 0) {
    const int rc = frag_pack(x, workspace, M, K, ldx, x_kind == X_ROWS_BF16, stream);
    if (rc != 0) return rc;
    b.xp = (const _Float16*)workspace;
  }
  b.w = w; b.w2 = w2; b.out = out; b.partial = workspace + xfloats; b.bias = bias; b.bias2 = bias2; b.residual = residual;
  b.M = M; b.N = N; b.K = K; b.mt_all = (M + 15) / 16; b.ldo = ldo; b.act = act; b.out_type = out_type;
  b.splitk = p.splitk; b.kt_per_split = p.kt_per_split;
  const int rc = frag_launch(b, p, qtype, stream);
  if (rc != 0 || p.splitk == 1) return rc;
  GemmArgs a = {};
  a.out = out; a.bias = bias; a.residual = residual; a.partial = workspace + xfloats;
  a.M = M; a.N = N; a.K = K; a.ldo = ldo; a.act = act; a.out_type = out_type; a.splitk = p.splitk;
  return launch_reduce(a, stream);
}

// A product in front of a norm: with K split over workgroups its sums can stay in their slabs, and the norm, which reads every element
// anyway, adds them up (bigdl_rms_norm_parts).  Returns the splits (0: the product is better off whole).  x_kind 2: x in fragment order;
// 0: fp16 rows, more than 256 of them, where the prompt kernel runs.
extern "C" int bigdl_gemm_parts(int M, int N, int K, int ldx, int qtype, int x_kind) {
  qtype = t16_kernel_qtype(qtype);
  if (M <= 32 || N <= 0 || K <= 0 || (K & 31) || (N & 7) || !is_t16(qtype)) return 0;
  int splits = 0;
  if (x_kind == X_FRAGMENTS) {
    const FragPlan p = frag_plan(M, N, K, qtype, false, true, true);
    splits = p.ns == 0 ? 0 : p.splitk;
  } else if (x_kind == X_ROWS && M > 256 && K >= 256 && (K & 127) == 0 && (ldx & 7) == 0 && (int64_t)M * ldx < (1ll << 31)) {
    splits = prompt_parts(M, N, K);
  }
  return splits > 1 ? splits : 0;
}

// that product: partial [bigdl_gemm_parts][M][N] fp32, 16-byte aligned, `floats` of them.  x as there, 16-byte aligned.  (A scratch of any
// other size is refused, a larger one too: the norm adds up all the slabs that it is given.)
extern "C" int bigdl_gemm_parts_run(const void* x, const void* w, float* partial, int64_t floats, int M, int N, int K, int ldx, int qtype,
                                    int x_kind, hipStream_t stream) {
  const int splits = bigdl_gemm_parts(M, N, K, ldx, qtype, x_kind);
  if (splits < 2) return -4;
  if (partial == nullptr || floats != (int64_t)splits * M * N) return -5;
  if (((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)partial & 15)) return -1;
  qtype = t16_kernel_qtype(qtype);
  if (x_kind != X_FRAGMENTS) return prompt_parts_launch(x, w, partial, M, N, K, ldx, qtype, stream);
  const FragPlan p = frag_plan(M, N, K, qtype, false, true, true);
  FragArgs b = {};
  b.xp = (const _Float16*)x; b.w = w; b.partial = partial;
  b.M = M; b.N = N; b.K = K; b.mt_all = (M + 15) / 16; b.ldo = N; b.act = ACT_NONE; b.out_type = OUT_F16;
  b.splitk = p.splitk; b.kt_per_split = p.kt_per_split;
  return frag_launch(b, p, qtype, stream);
}

// Extended dense form for batched decode: RMSNorm folded in (gamma + row_ssq of x, see GemmArgs), gate / up pair in one
// launch (w2: out = act(x W^T + bias) * (x W2^T + bias2)), and the sums of squares of the output rows (ssq_out, after
// the residual add) for the norm folded into the next product.  workspace: see bigdl_gemm_lowbit_workspace.
extern "C" int bigdl_gemm_lowbit_ex(const void* x, const void* w, const void* w2, void* out, const void* bias, const void* bias2,
                                    const void* residual, const void* gamma, float gamma_offset, float eps,
                                    const float* row_ssq, float* ssq_out, float* workspace, int64_t workspace_floats, int M,
                                    int N, int K, int ldx, int ldo, int qtype, int act, int out_type, hipStream_t stream) {
  qtype = t16_kernel_qtype(qtype);
  if (M <= 0 || N <= 0 || K <= 0 || (K & 31) || (ldx & 7) || ((uintptr_t)x & 15) || ((uintptr_t)w & 15)) return -1;
  if (w2 != nullptr && ((uintptr_t)w2 & 15)) return -1;
  if (gamma != nullptr && (((uintptr_t)gamma & 15) || row_ssq == nullptr)) return -1;
  if (out_type < 0 || out_type > 2) return -3;
  if ((int64_t)M * ldx >= (1ll << 31)) return -6;
  GemmArgs a = {};
  a.x = (const _Float16*)x; a.w = w; a.out = out; a.bias = bias; a.residual = residual; a.partial = workspace;
  a.M = M; a.N = N; a.K = K; a.ldx = ldx; a.ldo = ldo; a.act = act; a.out_type = out_type;
  a.gamma = (const _Float16*)gamma; a.gamma_offset = gamma_offset; a.eps = eps; a.row_ssq = gamma != nullptr ? row_ssq : nullptr;
  a.ssq_out = ssq_out; a.w2 = w2; a.bias2 = bias2;
  return launch_dense(a, dense_plan(M, N, K, ldx, qtype, w2 != nullptr, gamma != nullptr, ssq_out != nullptr), qtype, workspace_floats,
                      stream);
}

// Grouped form: `rows` sorted rows in total; row i uses the weights of the expert that the block table assigns
// to its block, reads x row x_rows[i] (null: i) and writes out row i (scaled by row_scale[i] if given).
// The experts' [N, K] matrices are stacked by rows in w (N % 16 == 0).  bm is 64 or 128 and must be the value the
// block table was built with; max_blocks >= ceil(rows / bm) + n_experts.
extern "C" int bigdl_gemm_lowbit_grouped(const void* x, const void* w, void* out, const int* blk_expert,
                                         const int* blk_row0, const int* blk_rows, const int* x_rows,
                                         const float* row_scale, int rows, int max_blocks, int bm, int n_experts,
                                         int N, int K, int ldx, int ldo, int qtype, int act, int out_type,
                                         int x_row_count, hipStream_t stream) {
  qtype = t16_kernel_qtype(qtype);
  if (x_row_count <= 0 || (int64_t)x_row_count * ldx >= (1ll << 31)) return -6;
  if (rows <= 0 || N <= 0 || K <= 0 || (K & 31) || (N & 15) || (ldx & 7) || ((uintptr_t)x & 15) || ((uintptr_t)w & 15) ||
      blk_expert == nullptr || blk_row0 == nullptr || blk_rows == nullptr || (bm != 64 && bm != 128) || max_blocks <= 0 ||
      max_blocks > 65535 || n_experts <= 0)
    return -1;
  if (out_type < 0 || out_type > 2) return -3;
  GemmArgs a = {};
  a.x = (const _Float16*)x; a.w = w; a.out = out; a.M = rows; a.N = N; a.K = K; a.ldx = ldx; a.ldo = ldo; a.act = act;
  a.out_type = out_type; a.splitk = 1; a.kt_per_split = (K + 127) / 128;
  a.blk_expert = blk_expert; a.blk_row0 = blk_row0; a.blk_rows = blk_rows; a.x_rows = x_rows; a.row_scale = row_scale;
  a.n_total = n_experts * N;
  return dispatch(a, qtype, bm, 128, max_blocks, stream);
}

extern "C" int bigdl_moe_block_table(const int64_t* counts, int n_experts, int bm, int max_blocks, int* blk_expert,
                                     int* blk_row0, int* blk_rows, hipStream_t stream) {
  if (counts == nullptr || n_experts <= 0 || bm <= 0 || max_blocks <= 0) return -1;
  hipLaunchKernelGGL(moe_block_table_kernel, dim3(1), dim3(64), 0, stream, counts, n_experts, bm, max_blocks, blk_expert,
                     blk_row0, blk_rows);
  return HIP_CHECK_LAUNCH();
}
