// p0k_gemm_dma_f16.hip — the load-to-LDS GEMM (p0k_gemm_dma.h) for f16 weights: one translation unit per encoding, so
// that they compile side by side.
#include "p0k_gemm_dma.h"

namespace p0k {

hipError_t launch_dma_f16(const Params &p, int xg, unsigned bm, unsigned bn, unsigned wv, hipStream_t s) {
  switch (xg) {
  case X_F16: return launch_dma_we<W_F16, X_F16>(p, bm, bn, wv, s);
  case X_CONV: return launch_dma_we<W_F16, X_CONV>(p, bm, bn, wv, s);
  case X_CONV3:
    return p.Ci % 64 == 0 ? launch_dma_we<W_F16, X_CONV3>(p, bm, bn, wv, s) : launch_dma_we<W_F16, X_CONV3H>(p, bm, bn, wv, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace p0k
