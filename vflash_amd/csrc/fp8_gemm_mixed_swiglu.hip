// The mixed-tile E4M3 GEMM with the SwiGLU epilogue (fp8_gemm_mixed.h).
#include "fp8_gemm_mixed.h"

namespace vfa {
template hipError_t launch_mixed<EPI_SWIGLU>(const GemmParams&, int64_t, int, hipStream_t);
}
