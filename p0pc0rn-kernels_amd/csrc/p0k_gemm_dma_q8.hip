// p0k_gemm_dma_q8.hip — the load-to-LDS GEMM (p0k_gemm_dma.h) for q8 weights: one translation unit per encoding, so
// that they compile side by side.
#include "p0k_gemm_dma.h"

namespace p0k {

hipError_t launch_dma_q8(const Params &p, int xg, unsigned bm, unsigned bn, unsigned wv, hipStream_t s) {
  switch (xg) {
  case X_F16: return launch_dma_we<W_Q8, X_F16>(p, bm, bn, wv, s);
  case X_CONV: return launch_dma_we<W_Q8, X_CONV>(p, bm, bn, wv, s);
  case X_CONV3: return launch_dma_we<W_Q8, X_CONV3>(p, bm, bn, wv, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace p0k
