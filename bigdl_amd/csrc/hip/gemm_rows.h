// Interface of the few-row low-bit product (gemm_rows.hip) for the entry points that share it.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bigdl {
struct RowsArgs;
struct RowsPlan {
  int mt, nt;               // 16-row tiles of x and 16-column weight tiles of a workgroup
  int splitk, kt_per_split;
  int turns;                // of the grid over the CUs, one workgroup each
};
RowsPlan rows_plan(int M, int N, int K, int qtype, bool pair, bool may_split);
// x the kernel can address: 16-byte rows, a row block within a gigabyte (its offsets are 32 bits)
static inline bool rows_ok(const void* x, int ldx) {
  return (ldx & 7) == 0 && ((uintptr_t)x & 15) == 0 && ldx > 0 && (int64_t)ldx * 128 < 0x40000000;
}
int rows_launch(const RowsArgs& a, const RowsPlan& p, int qtype, hipStream_t st);
// gemv_q6k.hip: q6_k blocks, 1 - 4 rows
bool gemv_q6k_takes(const RowsArgs& a);
int gemv_q6k_launch(const RowsArgs& a, hipStream_t st);
}  // namespace bigdl
