// fp16 / bf16 instantiations of the ring kernel (gemm_ring.h), row-major or K-major B.
#include "gemm_ring.h"

namespace mi355 {

namespace {
template <typename E, bool KM>
int launch(const GemmArgs& p, int shape, int splits, int chunk_bytes, hipStream_t stream) {
  switch (shape) {
    case 0: return launch_gemm_ring<E, 128, 128, 2, KM, 4>(p, splits, chunk_bytes, stream);
    case 4: return launch_gemm_ring<E, 128, 128, 2, KM, 2>(p, splits, chunk_bytes, stream);
    case 1: return launch_gemm_ring<E, 128, 64, 2, KM, 4>(p, splits, chunk_bytes, stream);
    case 3:
      if constexpr (KM) return launch_gemm_ring<E, 64, 32, 2, true, 8>(p, splits, chunk_bytes, stream);
      return (int)hipErrorInvalidValue;
    default: return launch_gemm_ring<E, 64, 64, 2, KM, 4>(p, splits, chunk_bytes, stream);
  }
}

// Grouped GEMM (python/tutorials/08-grouped-gemm.py:64-140: row-major A, B and C of one type) with the problem table as a
// kernel argument: program b takes the tiles b, b + gridDim.x, ... of all problems, numbered problem after problem, each
// problem on tiles of 128x128 or of 64x64 as the host chose for it.  Problems have rows of whole 16-byte chunks (A and B).
// Bound by the launch for small groups: with the tables copied to the device (five copies) and three launches of which one
// works, the group 1024^3, 512^3, 256^3, 128^3 took 112 us a call, 25 of them on 85 tiles of 128x128; now 11 us, one launch of
// 340 tiles of 64x64.  Experts 2440 -> 600 with 20 .. 334 rows each, four of them: 126 -> 14 us; 1664 -> 3712 with 30 .. 1758 rows,
// three: 156 -> 50.
template <typename E>
__global__ __launch_bounds__(256, 1) void gemm_ring_grouped_kernel(GroupedTable ga) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const unsigned lds0 = lds_addr((LDS_PTR(char))smem);
  const int nprog = gridDim.x;
  // one table entry per lane: the problem of a tile is a comparison away, whatever the number of problems
  const int first = ga.first_tile[threadIdx.x & 63];
  for (int t = xcd_remap(blockIdx.x, nprog); t < ga.total_tiles; t += nprog) {
    const int gi = __builtin_amdgcn_readfirstlane((int)__popcll(__ballot(first <= t)) - 1);
    const int tile = t - ga.first_tile[gi];
    GemmArgs p{};
    p.A = (const char*)ga.a_ptrs[gi]; p.B = (const char*)ga.b_ptrs[gi]; p.C = (char*)ga.c_ptrs[gi];
    p.M = ga.sizes[gi * 3]; p.N = ga.sizes[gi * 3 + 1]; p.K = ga.sizes[gi * 3 + 2];
    p.k_bytes = p.K * 2;
    p.lda = (int64_t)ga.lds[gi * 3] * 2; p.ldb = (int64_t)ga.lds[gi * 3 + 1] * 2; p.ldc = ga.lds[gi * 3 + 2];
    p.scn = 1; p.out_dtype = ga.out_dtype;
    p.c_vec_ok = p.ldc % 4 == 0 && (uintptr_t)p.C % 16 == 0;
    const int edge = (ga.small_tiles >> gi) & 1 ? 64 : 128;
    int pm, pn;
    grouped_tile(tile, (p.M + edge - 1) / edge, (p.N + edge - 1) / edge, 8, pm, pn);
    if (edge == 64) gemm_ring_tile<E, 64, 64, 2, false, 4>(p, pm, pn, lds0);
    else gemm_ring_tile<E, 128, 128, 2, false, 4>(p, pm, pn, lds0);
    wait_vmcnt<0>();   // (the stores: the next tile counts its loads)
    block_barrier();   // the next tile's loads overwrite the stages
  }
}

template <typename E>
int launch_grouped(const GroupedTable& ga, int nprog, hipStream_t stream) {
  constexpr int most = 4 * (128 + 128) * RING_ROW;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_ring_grouped_kernel<E>, hipFuncAttributeMaxDynamicSharedMemorySize, most);
    if (e != hipSuccess) return (int)e;
    attr_set = true;
  }
  const uint64_t all = ga.group_size == 64 ? ~0ull : (1ull << ga.group_size) - 1;
  gemm_ring_grouped_kernel<E><<<dim3(nprog), dim3(256), ga.small_tiles == all ? most / 2 : most, stream>>>(ga);
  return (int)hipGetLastError();
}
}  // namespace

int gemm_ring_grouped_launch(const GroupedTable& ga, bool bf16, int nprog, hipStream_t stream) {
  return bf16 ? launch_grouped<Ring16<bf16x8>>(ga, nprog, stream) : launch_grouped<Ring16<f16x8>>(ga, nprog, stream);
}

int gemm_ring16_launch(const GemmArgs& p, bool bf16, bool b_kmajor, int shape, int splits, int chunk_bytes, hipStream_t stream) {
  if (bf16) return b_kmajor ? launch<Ring16<bf16x8>, true>(p, shape, splits, chunk_bytes, stream) : launch<Ring16<bf16x8>, false>(p, shape, splits, chunk_bytes, stream);
  return b_kmajor ? launch<Ring16<f16x8>, true>(p, shape, splits, chunk_bytes, stream) : launch<Ring16<f16x8>, false>(p, shape, splits, chunk_bytes, stream);
}

}  // namespace mi355
