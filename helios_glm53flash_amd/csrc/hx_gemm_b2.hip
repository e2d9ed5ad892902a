// Instantiation of the MFMA linear kernels for 2-bit trellis.
#include "hx_gemm_impl.hpp"

namespace hx {
template hipError_t launch_mfma_b<2>(int, const MfmaGemmArgs&, hipStream_t);
}  // namespace hx
