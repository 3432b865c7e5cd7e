// fp8 (e4m3fn / e5m2) instantiations of the ring kernel (gemm_ring.h), both operands K-major.
#include "gemm_ring.h"

namespace mi355 {

namespace {
template <typename E>
int launch(const GemmArgs& p, int shape, int splits, int chunk_bytes, hipStream_t stream) {
  switch (shape) {
    case 0: return launch_gemm_ring<E, 128, 128, 2, true, 4>(p, splits, chunk_bytes, stream);
    case 4: return launch_gemm_ring<E, 128, 128, 2, true, 2>(p, splits, chunk_bytes, stream);
    case 1: return launch_gemm_ring<E, 128, 64, 2, true, 4>(p, splits, chunk_bytes, stream);
    case 3: return launch_gemm_ring<E, 64, 32, 2, true, 8>(p, splits, chunk_bytes, stream);
    default: return launch_gemm_ring<E, 64, 64, 2, true, 4>(p, splits, chunk_bytes, stream);
  }
}
}  // namespace

int gemm_ring8_launch(const GemmArgs& p, bool e5m2, int shape, int splits, int chunk_bytes, hipStream_t stream) {
  return e5m2 ? launch<Ring8<1>>(p, shape, splits, chunk_bytes, stream) : launch<Ring8<0>>(p, shape, splits, chunk_bytes, stream);
}

}  // namespace mi355
