// gemm_tile.h instantiated for two k-contiguous operands (Y = X W^T, its gate/up form, the LM head's statistics).
#include "gemm_tile.h"

namespace q3gemm {

template <typename T, int EPI> static int nt(int cfg, const Args& a, hipStream_t s) {
  switch (cfg) {
    case 0: return launch_tile<T, 256, 256, 4, 2, 2, false, false, EPI>(a, s);
    case 1: return launch_tile<T, 128, 256, 2, 4, 2, false, false, EPI>(a, s);
    case 2: return launch_tile<T, 128, 128, 2, 2, 3, false, false, EPI>(a, s);
    case 3: return launch_tile<T, 64, 128, 2, 4, 4, false, false, EPI>(a, s);
    case 4: return launch_tile<T, 64, 64, 2, 2, 4, false, false, EPI>(a, s);
    case 6: return launch_tile<T, 192, 256, 4, 2, 2, false, false, EPI>(a, s);
    case 7: return launch_tile<T, 192, 128, 4, 2, 3, false, false, EPI>(a, s);
    default: return launch_tile<T, 32, 64, 2, 2, 4, false, false, EPI>(a, s);
  }
}

template <typename T> static int stats(int cfg, const Args& a, hipStream_t s) {
  if (cfg == 0) return launch_tile<T, 256, 256, 4, 2, 2, false, false, 2>(a, s);
  return launch_tile<T, 128, 256, 4, 2, 2, false, false, 2>(a, s);
}

int launch_tile_nt(int dtype, int cfg, int epi, const Args& a, hipStream_t s) {
  if (epi == 2) return dtype == Q3_BF16 ? stats<BF16>(cfg, a, s) : stats<F16>(cfg, a, s);
  if (epi == 3) return dtype == Q3_BF16 ? nt<BF16, 3>(cfg, a, s) : nt<F16, 3>(cfg, a, s);
  return dtype == Q3_BF16 ? nt<BF16, 0>(cfg, a, s) : nt<F16, 0>(cfg, a, s);
}

}  // namespace q3gemm
