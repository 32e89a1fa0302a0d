// GEMM kernels for _Float16 operands (one translation unit per element type so the
// instantiations compile in parallel).
#include "bi_gemm_kernel.h"

bi_gemm_dev::KernelFn bi_gemm_kernel_f16(int g, bool trans_b, bool ragged) {
  return bi_gemm_dev::kernel_for<_Float16>(g, trans_b, ragged);
}
