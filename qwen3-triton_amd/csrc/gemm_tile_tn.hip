// gemm_tile.h instantiated for two K-major operands: the weight gradients dW = dY^T X.
#include "gemm_tile.h"

namespace q3gemm {

template <typename T> static int tn(int cfg, const Args& a, hipStream_t s) {
  switch (cfg) {
    case 0: return launch_tile<T, 256, 256, 4, 2, 2, true, true, 0>(a, s);
    case 1: return launch_tile<T, 128, 256, 2, 4, 2, true, true, 0>(a, s);
    case 2: return launch_tile<T, 128, 128, 2, 2, 3, true, true, 0>(a, s);
    case 3: return launch_tile<T, 64, 128, 2, 4, 4, true, true, 0>(a, s);
    default: return launch_tile<T, 64, 64, 2, 2, 4, true, true, 0>(a, s);
  }
}

int launch_tile_tn(int dtype, int cfg, const Args& a, hipStream_t s) {
  return dtype == Q3_BF16 ? tn<BF16>(cfg, a, s) : tn<F16>(cfg, a, s);
}

}  // namespace q3gemm
