// Pieces shared by the four-wave GEMM kernels (gemm_wave128.hip: 16-bit and fp8; gemm_wave128_mx.hip: the
// block-scaled forms): the wait for the last MFMAs, the grid size, and the epilogue of 16x16 accumulator tiles.
#pragma once

// L2 touches ahead of the direct loads in the four-wave kernels (see gemm_wave128_tiles): on / off and the number of
// K steps they run ahead of the loads, as build-time switches for A/B measurements.
#ifndef MI355_W128_PREFETCH
#define MI355_W128_PREFETCH 1
#endif
#ifndef MI355_W128_PREFETCH_DISTANCE
#define MI355_W128_PREFETCH_DISTANCE 2
#endif
#include "gemm_core.h"

namespace mi355 {

// Epilogue for 16x16 tiles computed with the operands swapped (D[n][m]): lane l owns C row
// `mrow0 + 16 i + l%16` and, of tile (i, j), the four consecutive columns `ncol0 + 16 j + 4 (l/16) ..`.
// The MFMAs of these kernels are inline assembly, so the compiler neither knows that they are MFMAs nor waits
// for the last ones before it reads their results.  Waiting alone is not enough: nothing ties a plain
// `s_nop` statement to the accumulators, and the compiler has moved accumulator reads (spills and moves of the
// epilogue's register shuffle) in front of it, where they see registers that the last MFMAs have yet to write.
// So every accumulator passes through an (empty) assembly statement behind the wait: volatile statements keep
// their order, and a value read after its statement is read after the wait.
//
// The wait itself (mfma_retire) stands INSIDE the K loop, at the end of the body of a tile's last iteration:
// whatever the register allocator does with the accumulators on the edge that leaves the loop (its register
// shuffle for the epilogue, spills), it does behind the loop's last basic block, hence behind the wait.  A
// wait placed behind the loop can end up behind those moves (a block-scaled fp8 product once came out wrong
// that way, in one run of many).  A read of an MFMA result has to come (passes + 3) issue slots behind the
// MFMA - 7 for the 4-pass 16x16x32 16-bit and 16x16x128 fp4 forms, 11 for the 8-pass 16x16x128 fp8 form -;
// `s_nop 15` is 16 slots of 4 cycles, once per tile.
// The loop compares with a copy of the step count that went through an empty assembly statement: told that
// the test equals the loop's own exit test, the compiler sinks the wait out of the loop again.
__device__ __forceinline__ void mfma_retire() {
#if MI355_DEVICE_PASS
  asm volatile("s_nop 15" ::: "memory");
#endif
}
__device__ __forceinline__ void mfma_drain_row(f32x4 (&r)[8]) {
#if MI355_DEVICE_PASS
  asm volatile("" : "+a"(r[0]), "+a"(r[1]), "+a"(r[2]), "+a"(r[3]), "+a"(r[4]), "+a"(r[5]), "+a"(r[6]), "+a"(r[7]));
#endif
}
template <int MT>
__device__ __forceinline__ void mfma_drain(f32x4 (&acc)[MT][8]) {
#if MI355_DEVICE_PASS
  asm volatile("s_nop 15" ::: "memory");
#endif
#pragma unroll
  for (int i = 0; i < MT; i++) mfma_drain_row(acc[i]);
}

// Rows that are no whole number of 128-byte K steps (the ANYK forms): what is left of them, `rest` bytes, is multiplied FIRST, as
// step 0, from registers through LDS with zeros beyond K - its loads are the oldest of the prologue, so the second stage
// fills behind them and the step runs like any other.  Those forms take one tile per workgroup, and an odd number of
// steps ends with one more step behind the loop.  (A tail multiplied behind the loop, without overlap, cost three to seven steps, a
// group of scales more than a step: us, with that / so: bf16 8192 x 8192 x 8176 K-major 893 / 794, e4m3 8192 x 8192 x 1664 120 / 110; against the
// eight-wave kernel: 4096 x 4096 x 1088 fp16 with a bias row 75 / 38, MXFP8 6400 x 7936 x 8064 915 / 377, MXFP4 5376 x 5376 x 6912 212 / 112.)
// L loads of 8 rows each, 16 bytes a lane, in the order of the direct loads (PERM: chunks of MXFP4 rows, see there).
template <bool PERM>
__device__ __forceinline__ int head_chunk(int q, int lane) {
  const int s = (lane & 7) ^ (((q & 1) * 4 + (lane >> 4)) & 7);
  return PERM ? 2 * (s & 3) + (s >> 2) : s;
}
// BYTES: `rest` need not be whole chunks.  The chunk that a row ends inside is read as the row's last 16 bytes and moved down, so
// that nothing behind the row is read (the rows have 16 bytes at least).
template <int L, bool PERM = false>
__device__ __forceinline__ void head_load(i32x4 (&t)[L], const char* src, unsigned pitch, int lane, int rest) {
#pragma unroll   // (16 taken off the base: no lane offset is negative)
  for (int q = 0; q < L; q++) load16_sbase<0>(t[q], src - 16, ((lane >> 3) + 8 * q) * pitch + min(head_chunk<PERM>(q, lane) * 16 + 16, rest));
}
template <int L, bool PERM = false, bool BYTES = false>
__device__ __forceinline__ void head_store(i32x4 (&t)[L], unsigned dst, int lane, int rest) {
  const i32x4 zero = {0, 0, 0, 0};
#pragma unroll
  for (int q = 0; q < L; q++) {
    const int at = head_chunk<PERM>(q, lane) * 16;
    lds_use(t[q]);
    const i32x4 whole = !BYTES || at + 16 <= rest ? t[q] : bytes_down(t[q], -rest & 15);
    *(LDS_PTR(i32x4))(uintptr_t)(dst + q * 1024 + lane * 16) = at < rest ? whole : zero;
  }
}

// The e8m0 scales of the block-scaled kernels lie in LDS as 16 bytes a row - a group of G K steps -, A's row r at 16 r and B's
// behind 256 of those, in two slots.  Scale rows that begin on 16 bytes and a K of whole groups are fetched 16 bytes a lane; the
// ANYK forms, whose rows begin on dwords, fetch a dword a lane, 16 rows an instruction: a quarter of the wave's rows in
// each of four steps (G = 2: two quarters in each of two), in the G steps between the last read of the slot and the first of the
// next.  (A dword of 64 rows an instruction, one for each operand and step, made the loop 12 to 19 % longer: 64 lines to look
// up instead of 16.)  `bytes`: what a row holds, in whole dwords; the lanes behind it fetch the last one again.
template <int ROWS, int Q0, int QN, bool SETTLE>
__device__ __forceinline__ void scale_quarters(const char* sa, const char* sb, unsigned pitch_a, unsigned pitch_b, int q, int at, int bytes, unsigned slot, int wave, int lane) {
#pragma unroll
  for (int i = Q0; i < Q0 + QN; i++) {
    const int row = 16 * (q + i) + (lane >> 2);
    const unsigned in_row = min(at + 4 * (lane & 3), bytes - 4);
    if (ROWS == 64 || row < ROWS) async_copy4_sbase<SETTLE>(sa, (unsigned)min(row, ROWS - 1) * pitch_a + in_row, slot + (wave * ROWS + 16 * (q + i)) * 16);
    async_copy4_sbase<SETTLE>(sb, (unsigned)row * pitch_b + in_row, slot + 4096 + (wave * 64 + 16 * (q + i)) * 16);
  }
}
// The first step of `blocks` scale blocks (see head_load), through registers: dword d of the wave's rows, 2^0 behind the last block.
template <int SD>
__device__ __forceinline__ void head_scale_load(int (&t)[2][SD], const char* sa, const char* sb, unsigned off_a, unsigned off_b, int blocks) {
#pragma unroll
  for (int d = 0; d < SD; d++) {   // (no dword without a block of the row)
    const unsigned at = 4 * min(d, (blocks - 1) / 4);
    load4_sbase(t[0][d], sa, off_a + at);
    load4_sbase(t[1][d], sb, off_b + at);
  }
}
template <int SD>
__device__ __forceinline__ void head_scale_store(int (&t)[2][SD], unsigned slot, int wave, int lane, int blocks) {
#pragma unroll
  for (int d = 0; d < SD; d++) {
    const int n = blocks - 4 * d;
    const unsigned mask = n >= 4 ? ~0u : n <= 0 ? 0u : (1u << (8 * n)) - 1u;
#pragma unroll
    for (int o = 0; o < 2; o++) {
      lds_use(t[o][d]);
      *(LDS_PTR(int))(uintptr_t)(slot + o * 4096 + (wave * 64 + lane) * 16 + 4 * d) = (int)(((unsigned)t[o][d] & mask) | (0x7f7f7f7fu & ~mask));
    }
  }
}

// Workgroups for `tiles` tiles on at most `cap` CUs.  More tiles than CUs need r = ceil(tiles / cap) rounds
// however they are dealt: ceil(tiles / r) programs walk r tiles each (the last ones r - 1) as one stream of K
// steps, without the restart that a fresh workgroup per tile pays, and the CUs left without a program leave
// their share of the board's power to the others.  Against one workgroup per tile wherever the tiles do not
// divide by the CU count, same call, bf16 / fp8 TFLOP/s: 6144^3 (576 tiles -> 192 programs) 1240 vs 1180 and
// 2380 vs 2200; 7168^3 (784 -> 196) 1270 vs 1200 and 2450 vs 2307; 4352 x 4352 x 4096 (289 -> 145) 973 vs 892
// and 1692 vs 1603; 5120^3 (400 -> 200) 1233 vs 1229 and 2323 vs 2248; 4096 x 11008 x 4096 (688 -> 230, ragged)
// 1315 vs 1307 and 2408 vs 2330.
static inline int wave128_grid(int tiles, int cap) {
  if (cap <= 0 || tiles <= cap) return tiles;
  const int rounds = (tiles + cap - 1) / cap;
  return (tiles + rounds - 1) / rounds;
}

// Exchange between the lane pairs (kg, kg ^ 1): see gemm_epilogue16_lean.
__device__ __forceinline__ void swap16(int& a, int& b) {
#if MI355_DEVICE_PASS
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
#endif
}

// Scales, addend, activation and any N, one row of 16x16 tiles at a time, every option behind one uniform branch per row.
// ANY = false: C in a 16-bit type with unit column stride, the addend (if any) a row of N consecutive values - a bias, read
// once for all rows of the lane (rows_epilogue).  C leaves as 16 bytes per lane (gemm_epilogue16_lean) whatever its alignment:
// the memory pipeline splits what it has to.  ANY = true: every output type, strides and addend that the C ABI takes.
// Columns from p.N on are left out; they can only be the last seven (16-bit operands) or fifteen (fp8) of the wave's 128, the
// padding of a 16-byte chunk that a tile of a row-major B may end in, so that only the last 16 columns are looked at.
template <int MT, int NT, bool ANY>
__device__ __forceinline__ void gemm_epilogue16(f32x4 (&acc)[MT][NT], const GemmArgs& p, int mrow0, int ncol0, int l16, int kg) {
  static_assert(NT % 2 == 0, "pairs of 16-column tiles");
  float alpha = 1.f;
  if (p.a_scale) alpha *= *p.a_scale;
  if (p.b_scale) alpha *= *p.b_scale;
  // columns of the lane's four that exist, for tile j
  auto columns = [&](auto J_) { return decltype(J_)::value == NT - 1 ? min(p.N - (ncol0 + decltype(J_)::value * 16 + kg * 4), 4) : 4; };
  // r += the addend at `off` (its row's first element)
  auto add_row = [&](f32x4 (&r)[NT], int64_t off) {
    auto typed = [&](auto* aux) {
      using AuxT = std::remove_const_t<std::remove_pointer_t<decltype(aux)>>;
      typedef AuxT Aux4 __attribute__((ext_vector_type(4), aligned(sizeof(AuxT))));
      auto* const at = aux + off + (int64_t)(ncol0 + kg * 4) * p.aux_sn;
      if (!ANY || p.aux_sn == 1) {
        static_for<NT>([&](auto J_) {
          constexpr int j = decltype(J_)::value;
          const int count = columns(J_);
          if (j < NT - 1 || count == 4) {
            const Aux4 t = *(const Aux4*)(at + j * 16);
#pragma unroll
            for (int e = 0; e < 4; e++) r[j][e] += (float)t[e];
          } else {
#pragma unroll
            for (int e = 0; e < 3; e++)
              if (e < count) r[j][e] += (float)at[j * 16 + e];
          }
        });
      } else {
        static_for<NT>([&](auto J_) {
          constexpr int j = decltype(J_)::value;
          const int count = columns(J_);
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (j < NT - 1 || e < count) r[j][e] += (float)at[(j * 16 + e) * p.aux_sn];
        });
      }
    };
    if (p.aux_dtype == 4) typed((const float*)p.aux);
    else if (p.aux_dtype == 1) typed((const __bf16*)p.aux);
    else typed((const _Float16*)p.aux);
  };
  f32x4 bias[ANY ? 1 : NT];
  if constexpr (!ANY) {
    static_for<NT>([&](auto J_) { bias[decltype(J_)::value] = f32x4{0.f, 0.f, 0.f, 0.f}; });
    if (p.aux) add_row(bias, 0);
  }
  static_for<MT>([&](auto I_) {
    constexpr int i = decltype(I_)::value;
    const int m = mrow0 + i * 16 + l16;
    f32x4 r[NT];
    static_for<NT>([&](auto J_) { r[decltype(J_)::value] = acc[i][decltype(J_)::value] * alpha; });
    if (p.aux) {
      if constexpr (ANY) add_row(r, (int64_t)m * p.aux_sm);
      else static_for<NT>([&](auto J_) { r[decltype(J_)::value] += bias[decltype(J_)::value]; });
    }
    if (p.activation == 1)
      static_for<NT>([&](auto J_) {
        f32x4& v = r[decltype(J_)::value];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = v[e] >= 0.f ? v[e] : 0.01f * v[e];
      });
    if (!ANY || ((p.out_dtype == 0 || p.out_dtype == 1) && p.scn == 1)) {
      int h[NT][2];   // the row in C's type, two columns a register
      auto round = [&](auto x) {
        using OutT = decltype(x);
        typedef OutT Out2 __attribute__((ext_vector_type(2)));
        static_for<NT>([&](auto J_) {
          constexpr int j = decltype(J_)::value;
          h[j][0] = __builtin_bit_cast(int, Out2{(OutT)r[j][0], (OutT)r[j][1]});
          h[j][1] = __builtin_bit_cast(int, Out2{(OutT)r[j][2], (OutT)r[j][3]});
        });
      };
      if (p.out_dtype == 1) round((__bf16)0.f);
      else round((_Float16)0.f);
      typedef int Chunk __attribute__((ext_vector_type(4), aligned(2)));
      const int col = ncol0 + 4 * (kg & 2) + 16 * (kg & 1);
      short* const row = (short*)p.C + (int64_t)m * p.ldc + col;
      static_for<NT / 2>([&](auto J_) {
        constexpr int j = 2 * decltype(J_)::value;
        swap16(h[j][0], h[j + 1][0]);
        swap16(h[j][1], h[j + 1][1]);
        const int w[4] = {h[j][0], h[j][1], h[j + 1][0], h[j + 1][1]};
        const int count = p.N - (col + j * 16);
        if (j < NT - 2 || count >= 8) {
          *(Chunk*)(row + j * 16) = Chunk{w[0], w[1], w[2], w[3]};
        } else {
#pragma unroll
          for (int e = 0; e < 7; e++)
            if (e < count) row[j * 16 + e] = (short)(w[e / 2] >> (16 * (e & 1)));
        }
      });
      return;
    }
    if constexpr (ANY)
      static_for<NT>([&](auto J_) {
        constexpr int j = decltype(J_)::value;
        const int n = ncol0 + j * 16 + kg * 4, count = columns(J_);
        const int64_t at = (int64_t)m * p.ldc + (int64_t)n * p.scn;
        const float v[4] = {r[j][0], r[j][1], r[j][2], r[j][3]};
        if (p.out_dtype == 2 || p.out_dtype == 3) {
          if (count > 0) store4_fp8(p.C, at, p.scn, p.out_dtype, v, p.c_vec_ok && n % 4 == 0, count);
        } else if (p.out_dtype == 4) {
          typedef float Four __attribute__((ext_vector_type(4), aligned(4)));
          if (p.scn == 1 && count == 4) *(Four*)((float*)p.C + at) = r[j];
          else {
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (e < count) ((float*)p.C)[at + e * p.scn] = v[e];
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; e++)
            if (e < count) ((short*)p.C)[at + e * p.scn] = p.out_dtype == 1 ? __builtin_bit_cast(short, (__bf16)v[e]) : __builtin_bit_cast(short, (_Float16)v[e]);
        }
      });
  });
}

// Whether the problem is one for gemm_epilogue16<ANY = false>.
static inline bool rows_epilogue(const GemmArgs& p) {
  return (p.out_dtype == 0 || p.out_dtype == 1) && p.scn == 1 && (!p.aux || (p.aux_sm == 0 && p.aux_sn == 1));
}

// The same for a plain C = A @ B in the operands' own 16-bit type with unit column stride (the grouped GEMM).
template <int MT, int NT, typename OutT>
__device__ __forceinline__ void gemm_epilogue16_plain(f32x4 (&acc)[MT][NT], const GemmArgs& p, int mrow0, int ncol0, int l16, int kg) {
  typedef OutT Out4 __attribute__((ext_vector_type(4)));
  static_for<MT>([&](auto I_) {
    constexpr int i = decltype(I_)::value;
    OutT* row = (OutT*)p.C + (int64_t)(mrow0 + i * 16 + l16) * p.ldc + ncol0 + kg * 4;
    static_for<NT>([&](auto J_) {
      constexpr int j = decltype(J_)::value;
      const f32x4 v = acc[i][j];
      if (p.c_vec_ok) *(Out4*)(row + j * 16) = Out4{(OutT)v[0], (OutT)v[1], (OutT)v[2], (OutT)v[3]};
      else {
#pragma unroll
        for (int e = 0; e < 4; e++) row[j * 16 + e] = (OutT)v[e];
      }
    });
  });
}

// The common case as an epilogue of its own: C in a 16-bit type with unit column stride and aligned rows, the
// product scaled by the per-tensor scales (1 without), no activation, no addend.  The general epilogue above decides
// output type, activation and store form at run time inside its 64 unrolled tiles: kernels of 132 - 140 KB with it (70 KiB of 81 when
// the figures here were taken) against 22 - 27 without, more than the instruction cache holds, fetched anew at the end of every tile (and from memory when the kernel
// starts on cold caches): same call, 8192^3 bf16 1425 -> 1457 TFLOP/s back to back and 1352 -> 1397 with flushed
// caches, 4096^3 1201 -> 1301 and 1011 -> 1205.  Kernels take it as a separate instantiation, chosen on the host.
// A lane holds 4 consecutive columns of a 16-column tile (8 bytes of C), so stores straight from the registers are 64
// pieces of 8 bytes per instruction and the memory pipeline takes a request per piece: 16384 of them per 256 x 256
// tile.  Two neighbouring tiles are therefore exchanged between the lane pairs (kg, kg ^ 1) first
// (v_permlane16_swap: the odd 16-lane rows of its first register with the even rows of its second): the even lane
// then holds 8 consecutive columns of the first tile and the odd lane 8 of the second - 16 bytes per lane, half the
// requests and half the store instructions (rows need 16-byte alignment: lean_epilogue_type).
template <int MT, int NT, typename OutT>
__device__ __forceinline__ void gemm_epilogue16_lean(f32x4 (&acc)[MT][NT], const GemmArgs& p, int mrow0, int ncol0, int l16, int kg) {
  static_assert(NT % 2 == 0 && sizeof(OutT) == 2, "pairs of 16-column tiles of a 16-bit type");
  typedef OutT Out2 __attribute__((ext_vector_type(2)));
  float alpha = 1.f;
  if (p.a_scale) alpha *= *p.a_scale;
  if (p.b_scale) alpha *= *p.b_scale;
  // even kg: columns 4 kg .. 4 kg + 7 of the pair's first tile; odd kg: 4 (kg - 1) .. 4 (kg - 1) + 7 of its second
  const int col = ncol0 + 4 * (kg & 2) + 16 * (kg & 1);
  static_for<MT>([&](auto I_) {
    constexpr int i = decltype(I_)::value;
    OutT* row = (OutT*)p.C + (int64_t)(mrow0 + i * 16 + l16) * p.ldc + col;
    static_for<NT / 2>([&](auto J_) {
      constexpr int j = 2 * decltype(J_)::value;
      const f32x4 u = acc[i][j], v = acc[i][j + 1];
      int a0 = __builtin_bit_cast(int, Out2{(OutT)(u[0] * alpha), (OutT)(u[1] * alpha)});
      int a1 = __builtin_bit_cast(int, Out2{(OutT)(u[2] * alpha), (OutT)(u[3] * alpha)});
      int b0 = __builtin_bit_cast(int, Out2{(OutT)(v[0] * alpha), (OutT)(v[1] * alpha)});
      int b1 = __builtin_bit_cast(int, Out2{(OutT)(v[2] * alpha), (OutT)(v[3] * alpha)});
      swap16(a0, b0);
      swap16(a1, b1);
      *(i32x4*)(row + j * 16) = i32x4{a0, a1, b0, b1};
    });
  });
}
// 0 = the problem needs the general epilogue; else the C ABI code + 1 of the 16-bit output type the lean one writes
static inline int lean_epilogue_type(const GemmArgs& p) {
  if (!p.lean_ok || p.aux || p.activation != 0 || p.scn != 1 || !p.c_vec_ok || p.ldc % 8 != 0 || p.N % 8 != 0) return 0;
  return p.out_dtype == 0 ? 1 : p.out_dtype == 1 ? 2 : 0;
}

}  // namespace mi355
