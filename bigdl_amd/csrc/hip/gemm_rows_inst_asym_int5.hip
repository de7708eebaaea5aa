// Instantiation unit of the few-row low-bit product for one weight format.
#include "gemm_rows_kernel.h"
namespace bigdl {
int gemm_rows_launch_asym_int5(const RowsArgs& a, int mt, int nt, hipStream_t st) { return gemm_rows_launch_qt<Q_ASYM_INT5>(a, mt, nt, st); }
}  // namespace bigdl
