// The few-row E4M3 GEMM with each epilogue that it serves (fp8_gemm_skinny.h).
#include "fp8_gemm_skinny.h"

namespace vfa {
template hipError_t launch_skinny<EPI_BIAS>(const GemmParams&, int, hipStream_t);
template hipError_t launch_skinny<EPI_GATE>(const GemmParams&, int, hipStream_t);
template hipError_t launch_skinny<EPI_LORA>(const GemmParams&, int, hipStream_t);
template hipError_t launch_skinny<EPI_LORA_GATE>(const GemmParams&, int, hipStream_t);
}  // namespace vfa
