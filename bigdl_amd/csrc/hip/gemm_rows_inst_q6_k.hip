// Instantiation unit of the few-row low-bit product for one weight format.
#include "gemm_rows_kernel.h"
namespace bigdl {
int gemm_rows_launch_q6_k(const RowsArgs& a, int mt, int nt, hipStream_t st) { return gemm_rows_launch_qt<Q_Q6_K>(a, mt, nt, st); }
}  // namespace bigdl
