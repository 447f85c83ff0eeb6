// gn_gemm_dma_glu.hip — LDS-DMA GEMM launches with the GLU epilogue (down projection dA = dY Wd: both
// operands untransposed, the only orientation gemm_dma_launch passes on), instantiated in a compilation
// unit of their own (gn_gemm_dma_core.h).
#include "gn_gemm_dma_core.h"

namespace gn {

int gemm_dma_glu(const GemmDesc& g, hipStream_t s) { return launch_shape<false, false, bf16_t, 1>(g, s); }

}  // namespace gn
