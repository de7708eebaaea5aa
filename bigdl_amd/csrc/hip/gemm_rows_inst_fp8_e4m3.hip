// Instantiation unit of the few-row low-bit product for one weight format.
#include "gemm_rows_kernel.h"
namespace bigdl {
int gemm_rows_launch_fp8_e4m3(const RowsArgs& a, int mt, int nt, hipStream_t st) { return gemm_rows_launch_qt<Q_FP8_E4M3>(a, mt, nt, st); }
}  // namespace bigdl
