// fp16 / bf16 instantiations of the ring kernel (gemm_ring.h), row-major or K-major B.
#include "gemm_ring.h"

namespace mi355 {

namespace {
template <typename E, bool KM>
int launch(const GemmArgs& p, int shape, int splits, int chunk_bytes, hipStream_t stream) {
  switch (shape) {
    case 0: return launch_gemm_ring<E, 128, 128, 2, KM, 4>(p, splits, chunk_bytes, stream);
    case 1: return launch_gemm_ring<E, 128, 64, 2, KM, 4>(p, splits, chunk_bytes, stream);
    default: return launch_gemm_ring<E, 64, 64, 2, KM, 4>(p, splits, chunk_bytes, stream);
  }
}
}  // namespace

int gemm_ring16_launch(const GemmArgs& p, bool bf16, bool b_kmajor, int shape, int splits, int chunk_bytes, hipStream_t stream) {
  if (bf16) return b_kmajor ? launch<Ring16<bf16x8>, true>(p, shape, splits, chunk_bytes, stream) : launch<Ring16<bf16x8>, false>(p, shape, splits, chunk_bytes, stream);
  return b_kmajor ? launch<Ring16<f16x8>, true>(p, shape, splits, chunk_bytes, stream) : launch<Ring16<f16x8>, false>(p, shape, splits, chunk_bytes, stream);
}

}  // namespace mi355
