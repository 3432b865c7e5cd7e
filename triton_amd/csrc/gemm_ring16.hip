// fp16 / bf16 instantiations of the ring kernel (gemm_ring.h), row-major or K-major B.
#include "gemm_ring.h"

namespace mi355 {

namespace {
template <typename E, bool KM, bool DWORDS>
int launch(const GemmArgs& p, int shape, int splits, int chunk_bytes, hipStream_t stream) {
  switch (shape) {
    case 0: return launch_gemm_ring<E, 128, 128, 2, KM, 4, DWORDS>(p, splits, chunk_bytes, stream);
    case 4: return launch_gemm_ring<E, 128, 128, 2, KM, 2, DWORDS>(p, splits, chunk_bytes, stream);
    case 1: return launch_gemm_ring<E, 128, 64, 2, KM, 4, DWORDS>(p, splits, chunk_bytes, stream);
    case 3:
      if constexpr (KM) return launch_gemm_ring<E, 64, 32, 2, true, 8, DWORDS>(p, splits, chunk_bytes, stream);
      return (int)hipErrorInvalidValue;
    default: return launch_gemm_ring<E, 64, 64, 2, KM, 4, DWORDS>(p, splits, chunk_bytes, stream);
  }
}

// Rows on dwords have kernels of their own: what the ends of their rows take in the prologue made the launches of whole chunks next to a
// row-major B 1 to 2 % longer.  us, one kernel for both / two: fp16 256^3 4.09 / 4.00, 512^3 4.59 / 4.52, 768 x 2944 x 384 7.95 / 7.75, 2048 x 512 x 4096 16.9 / 16.7.
template <typename E, bool KM>
int launch(const GemmArgs& p, int shape, int splits, int chunk_bytes, hipStream_t stream) {
  const bool chunks = ((p.k_bytes | p.lda | p.ldb | (int64_t)(uintptr_t)p.A | (int64_t)(uintptr_t)p.B) & 15) == 0;
  return chunks ? launch<E, KM, false>(p, shape, splits, chunk_bytes, stream) : launch<E, KM, true>(p, shape, splits, chunk_bytes, stream);
}

// Grouped GEMM (python/tutorials/08-grouped-gemm.py:64-140: row-major A, B and C of one type) with the problem table as a
// kernel argument: program b takes the tiles b, b + gridDim.x, ... of all problems, numbered problem after problem, in the
// order that group_plan chose.
// Problems have rows of whole 16-byte chunks (A and B).
// Bound by the launch for small groups: with the tables copied to the device (five copies) and three launches of which one
// works, the group 1024^3, 512^3, 256^3, 128^3 took 112 us a call, 25 of them on 85 tiles of 128x128; now 8, one launch of
// 340 tiles of 64x64.  Larger ones run on 128x128 tiles, in four stages or, more of them than CUs, in two with two
// workgroups on a CU (group_plan): us on 64x64 / 128x128 / those pairs, eleven experts 2304 -> 256 of 35 .. 1464 rows 35.0 / 33.4 / 24.5,
// 272 -> 3248 18.0 / 28.7 / 39.9, 1024 -> 1280 19.4 / 14.5 / 18.2.  EDGE 0: both sizes in one launch, each problem on what costs it less, the 64x64
// tiles with the LDS of 128x128 ones and a CU to themselves: six problems of 64 .. 1984 x 72 .. 1448 and K of 96 .. 1552 17.3 / 16.1 / 20.7 / 13.4.
template <typename E, int EDGE, int NS>
__global__ __launch_bounds__(256, 1) void gemm_ring_grouped_kernel(GroupedTable ga) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const unsigned lds0 = lds_addr((LDS_PTR(char))smem);
  const int nprog = gridDim.x;
  // one table entry per lane: the problem of a tile is a comparison away, whatever the number of problems
  const int first = ga.first_tile[threadIdx.x & 63];
  // chunk: the tiles in runs of so many, dealt to the XCDs in turn; 0: an XCD takes an eighth of them, one after the other
  const int c = ga.chunk;
  for (int u = c > 0 ? (int)blockIdx.x : xcd_remap(blockIdx.x, nprog); u < ga.padded_tiles; u += nprog) {
    const int t = c > 0 ? (u / 8 / c * 8 + u % 8) * c + u / 8 % c : u;
    if (t >= ga.total_tiles) continue;
    const int gi = __builtin_amdgcn_readfirstlane((int)__popcll(__ballot(first <= t)) - 1);
    const int tile = t - ga.first_tile[gi];
    GemmArgs p{};
    p.A = (const char*)ga.a_ptrs[gi]; p.B = (const char*)ga.b_ptrs[gi]; p.C = (char*)ga.c_ptrs[gi];
    p.M = ga.sizes[gi * 3]; p.N = ga.sizes[gi * 3 + 1]; p.K = ga.sizes[gi * 3 + 2];
    p.k_bytes = p.K * 2;
    p.lda = (int64_t)ga.lds[gi * 3] * 2; p.ldb = (int64_t)ga.lds[gi * 3 + 1] * 2; p.ldc = ga.lds[gi * 3 + 2];
    p.scn = 1; p.out_dtype = ga.out_dtype;
    p.c_vec_ok = p.ldc % 4 == 0 && (uintptr_t)p.C % 16 == 0;
    int pm, pn;
    const int edge = EDGE > 0 ? EDGE : (ga.small_tiles >> gi) & 1 ? 64 : 128;
    grouped_tile(tile, (p.M + edge - 1) / edge, (p.N + edge - 1) / edge, 8, pm, pn);
    if constexpr (EDGE > 0) gemm_ring_tile<E, EDGE, EDGE, 2, false, NS>(p, pm, pn, lds0);
    else if (edge == 64) gemm_ring_tile<E, 64, 64, 2, false, NS>(p, pm, pn, lds0);
    else gemm_ring_tile<E, 128, 128, 2, false, NS>(p, pm, pn, lds0);
    wait_vmcnt<0>();   // (the stores: the next tile counts its loads)
    block_barrier();   // the next tile's loads overwrite the stages
  }
}

template <typename E, int EDGE, int NS>
int launch_grouped(const GroupedTable& ga, int nprog, hipStream_t stream) {
  constexpr int smem = NS * 2 * (EDGE > 0 ? EDGE : 128) * RING_ROW;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_ring_grouped_kernel<E, EDGE, NS>, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) return (int)e;
    attr_set = true;
  }
  gemm_ring_grouped_kernel<E, EDGE, NS><<<dim3(nprog), dim3(256), smem, stream>>>(ga);
  return (int)hipGetLastError();
}

template <typename E>
int launch_grouped(const GroupedTable& ga, int shape, int nprog, hipStream_t stream) {
  if (shape == 2) return launch_grouped<E, 64, 4>(ga, nprog, stream);
  if (shape == 5) return launch_grouped<E, 0, 4>(ga, nprog, stream);
  return shape == 4 ? launch_grouped<E, 128, 2>(ga, nprog, stream) : launch_grouped<E, 128, 4>(ga, nprog, stream);
}
}  // namespace

int gemm_ring_grouped_launch(const GroupedTable& ga, bool bf16, int shape, int nprog, hipStream_t stream) {
  return bf16 ? launch_grouped<Ring16<bf16x8>>(ga, shape, nprog, stream) : launch_grouped<Ring16<f16x8>>(ga, shape, nprog, stream);
}

int gemm_ring16_launch(const GemmArgs& p, bool bf16, bool b_kmajor, int shape, int splits, int chunk_bytes, hipStream_t stream) {
  if (bf16) return b_kmajor ? launch<Ring16<bf16x8>, true>(p, shape, splits, chunk_bytes, stream) : launch<Ring16<bf16x8>, false>(p, shape, splits, chunk_bytes, stream);
  return b_kmajor ? launch<Ring16<f16x8>, true>(p, shape, splits, chunk_bytes, stream) : launch<Ring16<f16x8>, false>(p, shape, splits, chunk_bytes, stream);
}

}  // namespace mi355
