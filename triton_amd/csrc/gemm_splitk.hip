// Second launch of a split-K product: C = act(alpha * (sum over the splits of the fp32 partial tiles) + addend), one
// rounding to the output type - the epilogue of the reference's kernel (python/tutorials/03-matrix-multiplication.py:
// 304-316) on sums that gemm_splitk_kernel left in the workspace as [splits][M][N] floats.  The slices are added in
// split order, so the result does not depend on how the workgroups of the first launch were scheduled.
#include "common.h"
#include "launch.h"
#include "formats.h"

namespace mi355 {

namespace {

// A thread per four consecutive columns of a row, a 16-byte load per slice (N not a multiple of four: of any alignment, columns
// beyond N left out), four slices under way, one 8-byte store of a 16-bit C.  A launch's latency more than bandwidth, 3.4 .. 4.4
// us.  Whole calls against 64-bit index arithmetic, a slice at a time and single elements stored, us: 41 x 1408 x 7680 fp16 11.7 ->
// 9.3, 256 x 1024 x 6656 13.9 -> 13.1, 48 x 4096 x 8192 bf16 18.3 -> 17.4, 64 x 8192 x 8192 28.0 -> 27.5 (weights in the last-level cache).
__global__ __launch_bounds__(256) void splitk_reduce_kernel(GemmStridedArgs p, const float* __restrict__ ws, int splits, unsigned groups, unsigned total) {
  const unsigned id = blockIdx.x * 256u + threadIdx.x;
  if (id >= total) return;
  const int m = (int)(id / groups), n = (int)(id % groups) * 4;
  const int64_t slice = (int64_t)p.M * p.N;
  const float* src = ws + (int64_t)m * p.N + n;
  const int count = min(p.N - n, 4);
  typedef float Four __attribute__((ext_vector_type(4), aligned(4)));
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (count == 4) {
    int z = 0;
    for (; z + 4 <= splits; z += 4) {
      const Four t0 = *(const Four*)(src + z * slice), t1 = *(const Four*)(src + (z + 1) * slice);
      const Four t2 = *(const Four*)(src + (z + 2) * slice), t3 = *(const Four*)(src + (z + 3) * slice);
      v += t0; v += t1; v += t2; v += t3;   // (in split order)
    }
    if (splits - z >= 2) {
      const Four t0 = *(const Four*)(src + z * slice), t1 = *(const Four*)(src + (z + 1) * slice);
      v += t0; v += t1;
      z += 2;
    }
    if (z < splits) v += *(const Four*)(src + z * slice);
  } else {
    for (int z = 0; z < splits; z++)
#pragma unroll
      for (int e = 0; e < 3; e++)
        if (e < count) v[e] += src[z * slice + e];
  }
  if (p.a_scale || p.b_scale) {
    float alpha = 1.f;
    if (p.a_scale) alpha *= *p.a_scale;
    if (p.b_scale) alpha *= *p.b_scale;
    v *= alpha;
  }
  if (p.aux) {
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (e < count) v[e] += load_aux(p.aux, (int64_t)m * p.aux_sm + (int64_t)(n + e) * p.aux_sn, p.aux_dtype);
  }
  if (p.activation == 1) {
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = v[e] >= 0.f ? v[e] : 0.01f * v[e];
  }
  const int64_t at = (int64_t)m * p.scm + (int64_t)n * p.scn;
  if (count == 4 && p.scn == 1 && (p.out_dtype == 0 || p.out_dtype == 1)) {
    auto store = [&](auto* c0) {
      using OutT = std::remove_pointer_t<decltype(c0)>;
      typedef OutT Out4 __attribute__((ext_vector_type(4), aligned(2)));
      *(Out4*)(c0 + at) = Out4{(OutT)v[0], (OutT)v[1], (OutT)v[2], (OutT)v[3]};
    };
    if (p.out_dtype == 1) store((__bf16*)p.C);
    else store((_Float16*)p.C);
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; e++) {
    if (e >= count) break;
    const float x = v[e];
    const int64_t idx = at + e * p.scn;
    switch (p.out_dtype) {
      case 0: ((_Float16*)p.C)[idx] = (_Float16)x; break;
      case 1: ((__bf16*)p.C)[idx] = (__bf16)x; break;
      case 2: ((uint8_t*)p.C)[idx] = f32_to_e4m3(x); break;
      case 3: ((uint8_t*)p.C)[idx] = f32_to_e5m2(x); break;
      default: ((float*)p.C)[idx] = x; break;
    }
  }
}

}  // namespace

int splitk_reduce_launch(const GemmStridedArgs& out, const float* workspace, int splits, hipStream_t stream) {
  const int64_t groups = ((int64_t)out.N + 3) / 4, threads = (int64_t)out.M * groups;
  if (threads <= 0 || threads > 0xffffff00ll) return -1;   // (the launch's own limit, and the index's: 128 GiB of a caller's slices; the library's are 64 MiB at most)
  splitk_reduce_kernel<<<dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream>>>(out, workspace, splits, (unsigned)groups, (unsigned)threads);
  return (int)hipGetLastError();
}

}  // namespace mi355
