// Instantiation unit of the product on x in fragment order for one weight format.
#include "gemm_frag_kernel.h"
namespace bigdl {
int gemm_frag_launch_sym_int8(const FragArgs& a, int mt, int ns, hipStream_t st) { return gemm_frag_launch_qt<Q_SYM_INT8>(a, mt, ns, st); }
}  // namespace bigdl
