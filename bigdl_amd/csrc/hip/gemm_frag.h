// Interface of the product on x in fragment order (gemm_frag.hip) for the entry points that share it.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bigdl {
// Rows of a call that the rule (gemm_lowbit.hip) gives to this product: above 512 only where K is no multiple of 128 and the
// alternative is the tile kernel, 256 rows at a time.  Measured at 200 such products of 513 to 2500 rows, 10 formats, pairs among them:
// 1.06 to 3.4 times the former speed (4672 x 4544, 1024 rows, sym_int4 141 -> 75 us, sym_int8 153 -> 80; 14336 x 4128, 1500 rows,
// sym_int4 310 -> 293).  One call of 4096 rows of 14336 x 4128 lost (asym_int4 926 -> 1143 us, sym_int8 999 -> 1155), so more rows go in
// pieces, which also bounds the copy of x.
constexpr int FRAG_MAX_ROWS = 2048;
struct FragArgs;
struct FragPlan {
  int mt, ns;               // 16-row tiles of x and 16-column weight tiles of a workgroup (pair form: ns / 2 of each weight); ns 0: none
  int splitk, kt_per_split;
  double us;                // what it is expected to take with its reduce launch, without the pass that orders x
};
static inline double frag_pack_us(int M, int K) { return 3.4 + 1e-6 * M * K; }
// sums_left: the sums of a split K stay in their slabs, for the norm that follows to add up
FragPlan frag_plan(int M, int N, int K, int qtype, bool pair, bool may_split, bool sums_left = false);
// halves of x in fragment order
static inline int64_t frag_halves(int M, int K) { return (int64_t)((K + 127) / 128) * 4 * ((M + 15) / 16) * 512; }
int frag_pack(const void* x, void* xp, int M, int K, int ldx, bool bf16, hipStream_t st);
int frag_launch(const FragArgs& a, const FragPlan& p, int qtype, hipStream_t st);
}  // namespace bigdl
