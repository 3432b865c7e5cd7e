// Rows copied into a pitch that the MFMA kernels' 16-byte loads can use, zeros behind them: what a product with rows that do
// not start on 16-byte boundaries needs before it can run on those kernels (the reference masks the K tail instead,
// python/tutorials/03-matrix-multiplication.py:297-298, on loads of any alignment).  Both operands in one launch.
//
// Bound by memory: every byte is read and written once.  A thread moves 16-byte chunks of the destination; the source's are
// read at whatever alignment they have (2-byte aligned 16-byte global loads are split by the memory pipeline, not by code).
// bf16 4095 x 4100 and 4100 x 4100: 134 MB in 28 us, 4.8 TB/s - the rate of a plain copy -, where three fills and three
// copies of a library took 82.
#include "common.h"
#include "launch.h"

namespace mi355 {

namespace {

struct RepackArgs { RepackRows op[2]; unsigned blocks0; };
constexpr int kChunksPerThread = 4;

__global__ __launch_bounds__(256) void repack_kernel(RepackArgs args) {
  const bool second = blockIdx.x >= args.blocks0;
  const RepackRows o = args.op[second ? 1 : 0];
  const unsigned block = second ? blockIdx.x - args.blocks0 : blockIdx.x;
  const unsigned per_row = (unsigned)(o.dst_bytes / 16);
  const uint64_t chunks = (uint64_t)per_row * (unsigned)o.dst_rows;
  const uint64_t first = (uint64_t)block * (256 * kChunksPerThread) + threadIdx.x;
  i32x4 v[kChunksPerThread];
  int64_t to[kChunksPerThread];
#pragma unroll
  for (int j = 0; j < kChunksPerThread; j++) {
    const uint64_t id = first + 256 * j;
    v[j] = i32x4{0, 0, 0, 0};
    to[j] = -1;
    if (id < chunks) {
      const unsigned row = (unsigned)(id / per_row), c = (unsigned)(id - (uint64_t)row * per_row) * 16;
      to[j] = (int64_t)row * o.dst_pitch + c;
      if (row < (unsigned)o.rows && c < (unsigned)o.bytes) {
        const char* src = o.src + (int64_t)row * o.pitch + c;
        if (c + 16 <= (unsigned)o.bytes) {
          __builtin_memcpy(&v[j], src, 16);
        } else if (o.bytes >= 16) {   // the row's last 16 bytes, shifted down over what the chunk before has of them
          unsigned __int128 w;
          __builtin_memcpy(&w, src - (c + 16 - (unsigned)o.bytes), 16);
          w >>= 8 * (c + 16 - (unsigned)o.bytes);
          __builtin_memcpy(&v[j], &w, 16);
        } else {
          unsigned __int128 w = 0;
          for (int e = o.bytes - 1; e >= 0; e--) w = (w << 8) | (unsigned char)src[e];
          __builtin_memcpy(&v[j], &w, 16);
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < kChunksPerThread; j++)
    if (to[j] >= 0) *(i32x4*)(o.dst + to[j]) = v[j];
}

}  // namespace

int repack_launch(const RepackRows* op, int count, hipStream_t stream) {
  RepackArgs args{};
  uint64_t blocks[2] = {0, 0};
  for (int i = 0; i < count; i++) {
    args.op[i] = op[i];
    const uint64_t chunks = (uint64_t)(op[i].dst_bytes / 16) * op[i].dst_rows;
    blocks[i] = (chunks + 256 * kChunksPerThread - 1) / (256 * kChunksPerThread);
  }
  if (blocks[0] + blocks[1] == 0 || blocks[0] + blocks[1] > 0x7fffffffull) return -1;
  args.blocks0 = (unsigned)blocks[0];
  repack_kernel<<<dim3((unsigned)(blocks[0] + blocks[1])), dim3(256), 0, stream>>>(args);
  return (int)hipGetLastError();
}

}  // namespace mi355
