// gemm_tile.h instantiated for a k-contiguous A and a K-major B: the input gradients dX = dY W, also with
// the operands in pieces along k (several projections of one input) and with the SwiGLU backward.
#include "gemm_tile.h"

namespace q3gemm {

template <typename T, int EPI, bool KP> static int nn(int cfg, const Args& a, hipStream_t s) {
  switch (cfg) {
    case 0: return launch_tile<T, 256, 256, 4, 2, 2, false, true, EPI, KP>(a, s);
    case 1: return launch_tile<T, 128, 256, 2, 4, 2, false, true, EPI, KP>(a, s);
    case 2: return launch_tile<T, 128, 128, 2, 2, 3, false, true, EPI, KP>(a, s);
    case 3: return launch_tile<T, 64, 128, 2, 4, 4, false, true, EPI, KP>(a, s);
    case 6: return launch_tile<T, 192, 256, 4, 2, 2, false, true, EPI, KP>(a, s);
    case 7: return launch_tile<T, 192, 128, 4, 2, 3, false, true, EPI, KP>(a, s);
    default: return launch_tile<T, 64, 64, 2, 2, 4, false, true, EPI, KP>(a, s);
  }
}

int launch_tile_nn(int dtype, int cfg, int epi, const Args& a, hipStream_t s) {
  if (epi == 5) return dtype == Q3_BF16 ? nn<BF16, 5, false>(cfg, a, s) : nn<F16, 5, false>(cfg, a, s);
  if (a.axis == 1) return dtype == Q3_BF16 ? nn<BF16, 0, true>(cfg, a, s) : nn<F16, 0, true>(cfg, a, s);
  return dtype == Q3_BF16 ? nn<BF16, 0, false>(cfg, a, s) : nn<F16, 0, false>(cfg, a, s);
}

}  // namespace q3gemm
