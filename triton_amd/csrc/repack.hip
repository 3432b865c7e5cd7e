// Rows copied into a pitch that the MFMA kernels' 16-byte loads can use, zeros behind them: what a product with rows that do
// not start on 16-byte boundaries needs before it can run on those kernels (the reference masks the K tail instead,
// python/tutorials/03-matrix-multiplication.py:297-298, on loads of any alignment).  Both operands in one launch.
//
// Bound by memory where the operands are large, by latency where they are not.  A wave moves up to 256 consecutive 16-byte chunks of
// one row of the destination, four loads a lane under way, its row found by one scalar division; the source's chunks are read
// at whatever alignment they have (2-byte aligned 16-byte global loads are split by the memory pipeline, not by code).
// bf16 4095 x 4100 and 4100 x 4100: 134 MB in 21.6 us, 6.2 TB/s; 1025 x 1029 and 1029 x 1027: 8.1 -> 6.9 us, fp16 300 x 3003 and 2001 x
// 3003 10.3 -> 9.3 (before: a 64-bit division for every chunk, and a fifth as many wavefronts).
#include "common.h"
#include "launch.h"

namespace mi355 {

namespace {

constexpr int kLoads = 4;                    // per lane
constexpr unsigned kSegment = 64 * kLoads;   // chunks per wave
struct RepackArgs { RepackRows op[2]; unsigned segments[2]; unsigned blocks0; };   // segments per row

__global__ __launch_bounds__(256) void repack_kernel(RepackArgs args) {
  const bool second = blockIdx.x >= args.blocks0;
  const RepackRows o = args.op[second ? 1 : 0];
  const unsigned wave = (second ? blockIdx.x - args.blocks0 : blockIdx.x) * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const unsigned segments = args.segments[second ? 1 : 0], row = wave / segments;
  if (row >= (unsigned)o.dst_rows) return;
  const unsigned at = ((wave - row * segments) * kSegment + lane) * 16, bytes = row < (unsigned)o.rows ? (unsigned)o.bytes : 0u;
  const char* const src = o.src + (int64_t)row * o.pitch;
  char* const dst = o.dst + (int64_t)row * o.dst_pitch;
  i32x4 v[kLoads];
#pragma unroll
  for (int j = 0; j < kLoads; j++) {
    const unsigned c = at + j * 1024;
    v[j] = i32x4{0, 0, 0, 0};
    if (c + 16 <= bytes) __builtin_memcpy(&v[j], src + c, 16);
  }
#pragma unroll
  for (int j = 0; j < kLoads; j++) {
    const unsigned c = at + j * 1024;
    if (c < bytes && c + 16 > bytes) {   // the row ends inside the chunk
      unsigned __int128 w = 0;
      if (bytes >= 16) {   // the row's last 16 bytes, shifted down over what the chunk before has of them
        __builtin_memcpy(&w, src + bytes - 16, 16);
        w >>= 8 * (c + 16 - bytes);
      } else {
        for (int e = (int)bytes - 1; e >= 0; e--) w = (w << 8) | (unsigned char)src[e];
      }
      __builtin_memcpy(&v[j], &w, 16);
    }
    if (c < (unsigned)o.dst_bytes) *(i32x4*)(dst + c) = v[j];
  }
}

}  // namespace

int repack_launch(const RepackRows* op, int count, hipStream_t stream) {
  RepackArgs args{};
  args.segments[1] = 1;
  uint64_t blocks[2] = {0, 0};
  for (int i = 0; i < count; i++) {
    args.op[i] = op[i];
    args.segments[i] = ((unsigned)(op[i].dst_bytes / 16) + kSegment - 1) / kSegment;
    blocks[i] = ((uint64_t)args.segments[i] * (unsigned)op[i].dst_rows + 3) / 4;   // (a wave each, four to a block)
  }
  if (blocks[0] + blocks[1] == 0 || blocks[0] + blocks[1] > 0x3fffffffull) return -1;
  args.blocks0 = (unsigned)blocks[0];
  repack_kernel<<<dim3((unsigned)(blocks[0] + blocks[1])), dim3(256), 0, stream>>>(args);
  return (int)hipGetLastError();
}

}  // namespace mi355
