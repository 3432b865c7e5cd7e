// Block-scaled (MXFP4 / MXFP8) instantiations of the ring kernel (gemm_ring.h), both operands K-major: products that give the
// CUs too few 256-column tiles, or tiles whose K or rows the four-wave kernels have no pipelined form for.
#include "gemm_ring.h"

namespace mi355 {

namespace {
template <typename E>
int launch(const GemmArgs& p, int shape, int splits, int chunk_bytes, hipStream_t stream) {
  switch (shape) {
    case 0: return launch_gemm_ring<E, 128, 128, 2, true, 4>(p, splits, chunk_bytes, stream);
    case 4: return launch_gemm_ring<E, 128, 128, 2, true, 2>(p, splits, chunk_bytes, stream);
    case 1: return launch_gemm_ring<E, 128, 64, 2, true, 4>(p, splits, chunk_bytes, stream);
    default: return launch_gemm_ring<E, 64, 64, 2, true, 4>(p, splits, chunk_bytes, stream);
  }
}
}  // namespace

int gemm_ring_mx_launch(const GemmArgs& p, bool fp4, int shape, int splits, int chunk_bytes, hipStream_t stream) {
  return fp4 ? launch<RingMx4>(p, shape, splits, chunk_bytes, stream) : launch<RingMx8>(p, shape, splits, chunk_bytes, stream);
}

}  // namespace mi355
