// GEMM tiles of 64 .. 128 rows and columns for products that do not give every CU a 256 x 256 tile: a workgroup of
// four waves per tile, each wave a quarter of it from 16x16 MFMAs, K in steps of 128 bytes of every operand row through
// a ring of NS LDS stages.
//
// What bounds it: at one workgroup per CU a K step is too short to hide its own loads - a 128 x 128 step is 512 cycles of
// MFMAs, a first touch in memory takes about 2500 - so the design is about bytes in flight.  A stage is refilled with the
// K step NS further on as soon as every wave holds that stage's fragments in registers, which keeps NS whole steps
// (128 KiB for the 128 x 128 tile) requested at any time; a load instruction moves whole 128-byte lines.  The fragments of the
// next stage are read between the MFMAs of the current one, so that a step has one barrier and no exposed LDS latency.
// (The kernel it replaces here - 64-byte K steps, three of them in flight, half-line loads, fragments read behind the
// barrier - took 0.33 us for 32 elements of K where this one takes 0.44 for 64.  us by tile shape 128x128 / 128x64 / 64x64, and
// before: bf16 1024 x 4096 x 4096 31.6 / 40.3 / 47.6, 45.6; 2048^3 18.9 / 23.6 / 26.6, 24.7; 1024^3 9.9 / 7.7 / 6.2, 13.5; fp16
// 512^3 6.8 / 5.1 / 4.3, 8.3; e4m3 1024 x 4096 x 4096 18.3 / 23.8 / 25.6, 24.3; 384 x 256 x 6784 fp16 39.0 / 31.3 / 21.4, 66.1.)
//
// Tiles of 64x32 are for up to 64 rows next to a K-major B, where the loads of one workgroup per CU are all there is: 12 KB
// a step, eight steps deep, 96 KB requested.  Against the better of 64x64 tiles, those split along K and the streaming kernel,
// us, weights from memory: e4m3 33 x 8192 x 8192 18.2 -> 13.7, fp16 33 x 6016 x 5376 22.0 -> 15.5.
//
// What is left at one 128 x 128 tile per CU (bf16, 1024 x 4096 x 4096, copies of the kernel with parts taken out): MFMAs and
// barriers alone 20.3 us, with the fragment reads 25.5, with the loads 26.6, all 31.6 - the tiles' 537 MB from L2 at 19 TB/s
// are the longest part; eight waves of half a tile each, or a ring twice as deep, change nothing.
//
// K tail (K bytes not a multiple of 128, or a last step that B's rows end inside): multiplied FIRST, as step 0, from registers through LDS with zeros beyond K -
// its loads are the oldest of the prologue, so the ring fills behind them and the tail costs one ordinary step.
#pragma once
#include "common.h"
#include "launch.h"

namespace mi355 {

// One element family: KS MFMAs per fragment pair and K step, two 16-byte chunks of a row per lane and step.  The MFMAs are
// inline assembly with the accumulator tied to the accumulation registers: left to the register allocator, the loop
// copied all of them once per pair of steps.
template <typename V8>
struct Ring16 {
  static constexpr int kElemBytes = 2, kSubSteps = 2, kScaleDwords = 0;
  using Operand = V8;
  __device__ static void mma(const bf16x8& a, const bf16x8& b, f32x4& c) {
#if MI355_DEVICE_PASS
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
#endif
  }
  __device__ static void mma(const f16x8& a, const f16x8& b, f32x4& c) {
#if MI355_DEVICE_PASS
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
#endif
  }
};
template <int FMT>   // 0 = e4m3fn, 1 = e5m2
struct Ring8 {
  static constexpr int kElemBytes = 1, kSubSteps = 1, kScaleDwords = 0;
  using Operand = i32x8;
  __device__ static void mma(const i32x8& a, const i32x8& b, f32x4& c) {
#if MI355_DEVICE_PASS
    if constexpr (FMT == 0) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 cbsz:1 blgp:1" : "+a"(c) : "v"(a), "v"(b));
#endif
  }
};

// Block-scaled elements (OCP MX: one e8m0 scale for every 32 of K): kScaleDwords dwords of scales per row and K step travel
// through the stages behind the operands.  MXFP8: a lane's two chunks, kg and 4 + kg, are halves of the blocks that the
// instruction takes them for, and the lane supplies the scale of block kg (see gemm_wave128_mx.hip).  MXFP4: a chunk is a
// block; lane kg takes block 2 kg in the first sub-step and 2 kg + 1 in the second, so that one 16-bit read fetches both
// scales and the sub-step's instruction names its byte.
struct RingMx8 {
  static constexpr int kElemBytes = 1, kSubSteps = 1, kScaleDwords = 1, kBlockBytes = 32;
  using Operand = i32x8;
  template <int KS>
  __device__ static void mma(const i32x8& a, const i32x8& b, f32x4& c, int sa, int sb) {
#if MI355_DEVICE_PASS
    asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0]" : "+a"(c) : "v"(a), "v"(b), "v"(sa), "v"(sb));
#endif
  }
};
struct RingMx4 {
  static constexpr int kElemBytes = 1, kSubSteps = 2, kScaleDwords = 2, kBlockBytes = 16;
  using Operand = i32x4;
  template <int KS>
  __device__ static void mma(const i32x4& a, const i32x4& b, f32x4& c, int sa, int sb) {
#if MI355_DEVICE_PASS
    if constexpr (KS == 0)
      asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0] cbsz:4 blgp:4" : "+a"(c) : "v"(a), "v"(b), "v"(sa), "v"(sb));
    else
      asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel:[1,1,0] op_sel_hi:[0,0,0] cbsz:4 blgp:4" : "+a"(c) : "v"(a), "v"(b), "v"(sa), "v"(sb));
#endif
  }
};

// Epilogue of 16x16 tiles computed with the operands swapped (D[n][m]): lane (l16, kg) owns C row mrow0 + 16 i + l16 and, of
// tile (i, j), the four consecutive columns ncol0 + 16 j + 4 kg ...  Scale, addend, activation and store are passes of
// their own over the accumulators, each behind one uniform branch, so that a plain product runs only the last one.
// Rows of C that start on 2-byte boundaries only (an odd N) still take 8-byte stores, which the memory pipeline splits;
// columns beyond N are stored one by one.
template <int MT, int NT>
__device__ __forceinline__ void ring_epilogue(f32x4 (&acc)[MT][NT], const GemmArgs& p, const int mrow0, const int ncol0, const int l16, const int kg) {
  if (p.a_scale || p.b_scale) {
    float alpha = 1.f;
    if (p.a_scale) alpha *= *p.a_scale;
    if (p.b_scale) alpha *= *p.b_scale;
    static_for<MT>([&](auto I_) { static_for<NT>([&](auto J_) { acc[decltype(I_)::value][decltype(J_)::value] *= alpha; }); });
  }
  if (p.aux) {
    auto add = [&](auto* aux0) {
      using AuxT = std::remove_const_t<std::remove_pointer_t<decltype(aux0)>>;
      typedef AuxT Aux4 __attribute__((ext_vector_type(4), aligned(sizeof(AuxT))));
      static_for<NT>([&](auto J_) {
        constexpr int j = decltype(J_)::value;
        const int n = ncol0 + j * 16 + kg * 4;
        const bool vec = p.aux_sn == 1 && n + 4 <= p.N;
        auto four = [&](int64_t row_off) {
          f32x4 v = {0.f, 0.f, 0.f, 0.f};
          if (vec) {
            const Aux4 t = *(const Aux4*)(aux0 + row_off + n);
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = (float)t[e];
          } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (n + e < p.N) v[e] = (float)aux0[row_off + (int64_t)(n + e) * p.aux_sn];
          }
          return v;
        };
        if (p.aux_sm == 0) {   // a row of N values: the same four for all rows of the lane
          const f32x4 v = four(0);
          static_for<MT>([&](auto I_) { acc[decltype(I_)::value][j] += v; });
        } else {
          static_for<MT>([&](auto I_) {
            constexpr int i = decltype(I_)::value;
            const int m = mrow0 + i * 16 + l16;
            if (m < p.M) acc[i][j] += four((int64_t)m * p.aux_sm);
          });
        }
      });
    };
    if (p.aux_dtype == 4) add((const float*)p.aux);
    else if (p.aux_dtype == 1) add((const __bf16*)p.aux);
    else add((const _Float16*)p.aux);
  }
  if (p.activation == 1)
    static_for<MT>([&](auto I_) {
      static_for<NT>([&](auto J_) {
        f32x4& v = acc[decltype(I_)::value][decltype(J_)::value];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] = v[e] >= 0.f ? v[e] : 0.01f * v[e];
      });
    });
  const bool inside = mrow0 + MT * 16 <= p.M && ncol0 + NT * 16 <= p.N;
  auto store16 = [&](auto* c0) {
    using OutT = std::remove_pointer_t<decltype(c0)>;
    (void)inside;
    typedef OutT Out2 __attribute__((ext_vector_type(2)));
    typedef OutT Out4 __attribute__((ext_vector_type(4), aligned(2)));
    if constexpr (NT % 2 == 0) if (inside && p.c_vec_ok && p.ldc % 8 == 0) {
      // two neighbouring tiles exchanged between lane pairs (kg, kg ^ 1): 16 bytes per lane (see gemm_epilogue16_lean)
      const int col = ncol0 + 4 * (kg & 2) + 16 * (kg & 1);
      static_for<MT>([&](auto I_) {
        constexpr int i = decltype(I_)::value;
        OutT* row = c0 + (int64_t)(mrow0 + i * 16 + l16) * p.ldc + col;
        static_for<NT / 2>([&](auto J_) {
          constexpr int j = 2 * decltype(J_)::value;
          const f32x4 u = acc[i][j], v = acc[i][j + 1];
          int a0 = __builtin_bit_cast(int, Out2{(OutT)u[0], (OutT)u[1]}), a1 = __builtin_bit_cast(int, Out2{(OutT)u[2], (OutT)u[3]});
          int b0 = __builtin_bit_cast(int, Out2{(OutT)v[0], (OutT)v[1]}), b1 = __builtin_bit_cast(int, Out2{(OutT)v[2], (OutT)v[3]});
#if MI355_DEVICE_PASS
          asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a0), "+v"(b0));
          asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a1), "+v"(b1));
#endif
          *(i32x4*)(row + j * 16) = i32x4{a0, a1, b0, b1};
        });
      });
      return;
    }
    static_for<MT>([&](auto I_) {
      constexpr int i = decltype(I_)::value;
      const int m = mrow0 + i * 16 + l16;
      if (m < p.M) {
        static_for<NT>([&](auto J_) {
          constexpr int j = decltype(J_)::value;
          const int n = ncol0 + j * 16 + kg * 4;
          const f32x4 v = acc[i][j];
          OutT* c = c0 + (int64_t)m * p.ldc + (int64_t)n * p.scn;
          if (p.scn == 1 && n + 4 <= p.N) {
            *(Out4*)c = Out4{(OutT)v[0], (OutT)v[1], (OutT)v[2], (OutT)v[3]};
          } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (n + e < p.N) c[e * p.scn] = (OutT)v[e];
          }
        });
      }
    });
  };
  if (p.out_dtype == 1) { store16((__bf16*)p.C); return; }
  if (p.out_dtype == 0) { store16((_Float16*)p.C); return; }
  static_for<MT>([&](auto I_) {
    constexpr int i = decltype(I_)::value;
    const int m = mrow0 + i * 16 + l16;
    if (m < p.M) {
      static_for<NT>([&](auto J_) {
        constexpr int j = decltype(J_)::value;
        const int n = ncol0 + j * 16 + kg * 4;
        const f32x4 x = acc[i][j];
        if (p.out_dtype == 4) {
          float* c = (float*)p.C + (int64_t)m * p.ldc + (int64_t)n * p.scn;
          if (p.c_vec_ok && n + 4 <= p.N) {
            *(f32x4*)c = x;
          } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (n + e < p.N) c[e * p.scn] = x[e];
          }
        } else {
          const float v[4] = {x[0], x[1], x[2], x[3]};
          const int count = p.N - n < 4 ? p.N - n : 4;
          if (count > 0) store4_fp8(p.C, (int64_t)m * p.ldc + (int64_t)n * p.scn, p.scn, p.out_dtype, v, p.c_vec_ok, count);
        }
      });
    }
  });
}

__device__ __forceinline__ void ring_pin(f32x4& c) {
#if MI355_DEVICE_PASS
  asm volatile("" : "+a"(c));
#endif
}

// The wait of a step of the ring's last NS steps, `left` of them to go (this one included): all but the loads of the
// steps behind the next one.  The branches stand inside the statement: as branches of the compiler's own they made the
// accumulators change registers at the loop's edges.
template <int NS, int L>
__device__ __forceinline__ void ring_drain_wait(int left) {
#if MI355_DEVICE_PASS
  static_assert(NS == 2 || NS == 4 || NS == 8, "the ladders of these depths");
  if constexpr (NS == 2)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  else if constexpr (NS == 4)
    asm volatile("s_cmp_lt_i32 %0, 4\n\ts_cbranch_scc1 ring_three_%=\n\ts_waitcnt vmcnt(%1)\n\ts_branch ring_done_%=\n"
                 "ring_three_%=:\n\ts_cmp_lt_i32 %0, 3\n\ts_cbranch_scc1 ring_all_%=\n\ts_waitcnt vmcnt(%2)\n\ts_branch ring_done_%=\n"
                 "ring_all_%=:\n\ts_waitcnt vmcnt(0)\nring_done_%=:" :: "s"(left), "i"(2 * L), "i"(L) : "memory", "scc");
  else   // (seven and five steps to go wait for one step more than they have to)
    asm volatile("s_cmp_lt_i32 %0, 6\n\ts_cbranch_scc1 ring_five_%=\n\ts_waitcnt vmcnt(%3)\n\ts_branch ring_done_%=\n"
                 "ring_five_%=:\n\ts_cmp_lt_i32 %0, 4\n\ts_cbranch_scc1 ring_three_%=\n\ts_waitcnt vmcnt(%1)\n\ts_branch ring_done_%=\n"
                 "ring_three_%=:\n\ts_cmp_lt_i32 %0, 3\n\ts_cbranch_scc1 ring_all_%=\n\ts_waitcnt vmcnt(%2)\n\ts_branch ring_done_%=\n"
                 "ring_all_%=:\n\ts_waitcnt vmcnt(0)\nring_done_%=:" :: "s"(left), "i"(2 * L), "i"(L), "i"(4 * L) : "memory", "scc");
#endif
}

constexpr int RING_ROW = 128;   // bytes of an operand row per K step
template <typename E, int BM, int BN>
constexpr int ring_stage_bytes() { return (BM + BN) * (RING_ROW + 4 * E::kScaleDwords); }

// Tile (pm, pn) of the product p with the ring of NS stages at LDS address lds0 (NS * (BM + BN) * 128 bytes).  A has whole
// 16-byte chunks along K (k_bytes in all) and a K-major B too; a row-major B (16-bit types) has p.K rows of whole 16-byte chunks: in
// the last chunk's place of A's rows there may be zeros beyond K.  DWORDS (16-bit types): dwords instead of chunks will do (8 elements at
// least), for the rows' begin as for their length - a direct load moves 16 bytes from any dword on, as fast as from rows of 16-byte but not 128-byte
// pitch (bf16 2048^3, rows of 2048 / 2056 / 2050 elements 18.6 / 24.5 / 24.4 us, 1024^3 8.1 / 8.2 / 8.3).  Block-scaled: both operands K-major, K a
// multiple of 128 elements, scale rows that begin on dwords.  Every wave's
// fragments are in registers when the last step's MFMAs begin, so a caller that runs another tile needs one barrier first.
template <typename E, int BM, int BN, int WN, bool B_KMAJOR, int NS, bool DWORDS = false>
__device__ __forceinline__ void gemm_ring_tile(const GemmArgs& p, const int pm, const int pn, const unsigned lds0) {
#if MI355_DEVICE_PASS
  using Op = typename E::Operand;
  constexpr bool WIDE = sizeof(Op) == 32;                  // a fragment is two chunks of a row, else one for each sub-step
  constexpr int SD = E::kScaleDwords;
  constexpr bool MX = SD > 0;
  static_assert(B_KMAJOR || (E::kElemBytes == 2 && BN >= 64), "row-major B: 16-bit types, pieces of 128 bytes and more");
  static_assert(!DWORDS || E::kElemBytes == 2, "rows on dwords: 16-bit types");
  static_assert((BM == 64 || BM == 128) && (BN == 32 || BN == 64 || BN == 128), "tile sizes");
  constexpr int NW = 2 * WN, TM = BM / 2, TN = BN / WN, MT = TM / 16, NT = TN / 16;
  constexpr int A_BYTES = BM * RING_ROW, S_BYTES = (BM + BN) * RING_ROW, STAGE = ring_stage_bytes<E, BM, BN>();
  constexpr int BLOCKS = (BM + BN) / 64, LS = (BLOCKS * SD + NW - 1) / NW;   // scales: loads of one dword of 64 rows
  constexpr int LA = BM / 8 / NW, LB = BN / 8 / NW, L = LA + LB + LS;   // direct loads per wave and step: 1 KiB each, then the scales
  constexpr int KS = E::kSubSteps, NMFMA = KS * MT * NT;
  static_assert(NS * L < 64, "vmcnt has six bits");

  const int lane = threadIdx.x & 63, l16 = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int m0 = pm * BM, n0 = pn * BN;
  // (a step that a row-major B ends inside is a tail too, a whole one where A's padding fills it: B has no rows to load there)
  // (and so is one that holds the last row of a row-major B whose rows end inside a chunk: nothing may be read behind that row)
  const int rest = p.k_bytes % RING_ROW;
  const bool open_rows = DWORDS && !B_KMAJOR && p.N % 8 != 0 && ((p.ldb | (int64_t)(uintptr_t)p.B) & 15) != 0;
  const int tail = !B_KMAJOR && rest == 0 && (open_rows || p.K * E::kElemBytes < p.k_bytes) ? RING_ROW : rest;
  const int steps = (p.k_bytes + RING_ROW - 1) / RING_ROW;
  constexpr int KROWS = RING_ROW / 2;                        // k rows of a row-major B per step

  auto scalar_ptr = [](const char* x) {   // (wave-uniform, but possibly read from device tables)
    const uint64_t v = (uint64_t)x;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const char*)(((uint64_t)hi << 32) | lo);
  };

  // ---- direct loads.  K-major operand: an instruction moves 8 rows of 128 bytes; LDS row r keeps chunk c in slot
  // c ^ ((r >> 1) & 7), so the 16 lanes of a fragment read (16 rows, one chunk) cover all banks once.  Row-major B: k rows of
  // BN * 2 bytes; the 32-byte column group g of row k sits at g ^ x(k), which spreads the 8 pieces that a transpose read
  // fetches at a time (k & 3 and (k >> 3) & 1 vary, same columns) over all banks.  Rows and columns past the matrix are
  // clamped onto the last valid ones.  The lane offsets carry 4096 (taken off the base) so that none is negative once
  // the instruction offset, which moves the LDS side, is taken back out of the global side.
  auto xor_of = [](int k) { return BN == 128 ? ((k & 3) << 1) ^ ((k >> 3) & 1) : (((k >> 1) & 1) << 1) ^ ((k >> 3) & 1); };
  auto chunk_of = [](int c) { return MX && KS == 2 ? 2 * (c & 3) + (c >> 2) : c; };   // the chunk of the row in the place of chunk c
  unsigned voffA[LA], voffB[LB];
  int chunkA[LA], rowB[LB];   // for the tail: the lane's chunk of A (and of a K-major B), the lane's k row of a row-major B
#pragma unroll
  for (int q = 0; q < LA; q++) {
    const int r = (wave * LA + q) * 8 + (lane >> 3);
    chunkA[q] = chunk_of((lane & 7) ^ ((r >> 1) & 7));
    voffA[q] = (unsigned)min(r, p.M - 1 - m0) * (unsigned)p.lda + chunkA[q] * 16 + 4096u - q * 1024;
  }
#pragma unroll
  for (int q = 0; q < LB; q++) {
    if constexpr (B_KMAJOR) {
      const int r = (wave * LB + q) * 8 + (lane >> 3);
      rowB[q] = chunk_of((lane & 7) ^ ((r >> 1) & 7));
      voffB[q] = (unsigned)min(r, p.N - 1 - n0) * (unsigned)p.ldb + rowB[q] * 16 + 4096u - q * 1024;
    } else {
      constexpr int CPR = BN / 8, RPI = 64 / CPR;   // 16-byte chunks per k row, k rows per instruction
      const int k = (wave * LB + q) * RPI + lane / CPR, pc = lane % CPR;
      const int chunk = (((pc >> 1) ^ xor_of(k)) << 1) | (pc & 1);
      const int last = (p.N + 7) / 8 - 1 - n0 / 8;
      rowB[q] = k;
      voffB[q] = (unsigned)k * (unsigned)p.ldb + min(chunk, last) * 16 + 4096u - q * 1024;
    }
  }
  const int64_t stepB = B_KMAJOR ? (int64_t)RING_ROW : KROWS * p.ldb;
  const char* tileA = scalar_ptr(p.A + (int64_t)m0 * p.lda - 4096);
  const char* tileB = scalar_ptr((B_KMAJOR ? p.B + (int64_t)n0 * p.ldb : p.B + (int64_t)n0 * 2) - 4096);
  const char* fA = tail ? tileA - RING_ROW : tileA;   // the K step being requested (step s, or s - 1 behind a tail)
  const char* fB = tail ? tileB - stepB : tileB;
  // scales: dword d of the 64 rows of block b (those of A, then those of B) at S_BYTES + 256 (b SD + d); waves without a share of
  // their own repeat another's, so that every wave counts the same loads
  const char* fS[LS > 0 ? LS : 1];
  unsigned voffS[LS > 0 ? LS : 1], slotS[LS > 0 ? LS : 1];
  auto scale_rows = [&](int b) {   // the lane's row of block b: address of the operand's scales, rows, pitch
    const bool a = b < BM / 64;
    const int r = (a ? b : b - BM / 64) * 64 + lane;
    return a ? (unsigned)min(r, p.M - 1 - m0) * (unsigned)p.lds_a : (unsigned)min(r, p.N - 1 - n0) * (unsigned)p.lds_b;
  };
  auto scale_base = [&](int b) {
    return scalar_ptr((const char*)(b < BM / 64 ? p.sA + (int64_t)m0 * p.lds_a : p.sB + (int64_t)n0 * p.lds_b));
  };
  if constexpr (MX) {
#pragma unroll
    for (int l = 0; l < LS; l++) {
      const int at = (wave * LS + l) % (BLOCKS * SD), b = at / SD, d = at % SD;
      fS[l] = scale_base(b) - (tail ? 4 * SD : 0);
      voffS[l] = scale_rows(b) + 4 * d;
      slotS[l] = S_BYTES + at * 256;
    }
  }
  auto advance = [&]() {
    fA += RING_ROW;
    fB += stepB;
#pragma unroll
    for (int l = 0; l < LS; l++) fS[l] += 4 * SD;
  };
  auto issue = [&](auto Q_, unsigned stage_base, auto SETTLE_) {   // (SETTLE in the prologue: scalar registers may just have been restored)
    constexpr int q = decltype(Q_)::value;
    if constexpr (q >= LA + LB) async_copy4_sbase<decltype(SETTLE_)::value>(fS[q - LA - LB], voffS[q - LA - LB], stage_base + slotS[q - LA - LB]);
    else
    if constexpr (q < LA) async_copy16_sbase_off<q * 1024, q == 0, decltype(SETTLE_)::value>(fA, voffA[q], stage_base + wave * (LA * 1024));
    else async_copy16_sbase_off<(q - LA) * 1024, q == LA, decltype(SETTLE_)::value>(fB, voffB[q - LA], stage_base + A_BYTES + wave * (LB * 1024));
  };

  // ---- fragment reads
  unsigned adrA[2], adrB[B_KMAJOR ? 2 : NT];
  {
    const unsigned s = (l16 >> 1) & 7;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const unsigned slot = ((4 * h + kg) ^ s) * 16;
      adrA[h] = lds0 + (wm * TM + l16) * RING_ROW + slot;
      if constexpr (B_KMAJOR) adrB[h] = lds0 + A_BYTES + (wn * TN + l16) * RING_ROW + slot;
    }
    if constexpr (!B_KMAJOR) {
      const int k = 8 * kg + (l16 >> 2);
#pragma unroll
      for (int t = 0; t < NT; t++) adrB[t] = lds0 + A_BYTES + k * (BN * 2) + (((wn * NT + t) ^ xor_of(k)) * 32) + (l16 & 3) * 8;
    }
  }
  // scale byte x of row R at 256 (R / 64 SD + x / 4) + 4 (R % 64) + x % 4 (16 rows of a tile stay in one block of 64)
  auto scale_at = [&](int row) {
    const int x = KS == 2 ? 2 * kg : kg;
    return lds0 + S_BYTES + ((row >> 6) * SD + (x >> 2)) * 256 + (row & 63) * 4 + (x & 3);
  };
  const unsigned adrSA = scale_at(wm * TM + l16), adrSB = scale_at(BM + wn * TN + l16);
  struct Frags { Op a[KS][MT]; Op b[KS][NT]; int sa[MX ? MT : 1]; int sb[MX ? NT : 1]; };
  Frags f[2];
  // read number R of a step: the fragments of A first, then those of B, then the scales
  auto read_frag = [&](auto R_, unsigned so, Frags& dst) {
    constexpr int r = decltype(R_)::value;
    if constexpr (r >= KS * (MT + NT)) {
      constexpr int t = r - KS * (MT + NT);
      auto read = [&](auto T_, unsigned adr) {
        if constexpr (KS == 2) return lds_read_u16<decltype(T_)::value * 64>(adr);
        else return lds_read_u8<decltype(T_)::value * 64>(adr);
      };
      if constexpr (t < MT) dst.sa[t] = read(std::integral_constant<int, t>{}, adrSA + so);
      else dst.sb[t - MT] = read(std::integral_constant<int, t - MT>{}, adrSB + so);
    } else if constexpr (r < KS * MT) {
      constexpr int ks = r / MT, t = r % MT;
      if constexpr (WIDE) {
        const i32x4 lo = lds_read_b128<t * 16 * RING_ROW>(adrA[0] + so), hi = lds_read_b128<t * 16 * RING_ROW>(adrA[1] + so);
        dst.a[0][t] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      } else {
        dst.a[ks][t] = __builtin_bit_cast(Op, lds_read_b128<t * 16 * RING_ROW>(adrA[ks] + so));
      }
    } else {
      constexpr int ks = (r - KS * MT) / NT, t = (r - KS * MT) % NT;
      if constexpr (WIDE) {
        const i32x4 lo = lds_read_b128<t * 16 * RING_ROW>(adrB[0] + so), hi = lds_read_b128<t * 16 * RING_ROW>(adrB[1] + so);
        dst.b[0][t] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      } else if constexpr (B_KMAJOR) {
        dst.b[ks][t] = __builtin_bit_cast(Op, lds_read_b128<t * 16 * RING_ROW>(adrB[ks] + so));
      } else {
        constexpr int imm = ks * 32 * BN * 2;
        const i32x2 lo = lds_read_tr16_b64<imm>(adrB[t] + so), hi = lds_read_tr16_b64<imm + 4 * BN * 2>(adrB[t] + so);
        dst.b[ks][t] = __builtin_bit_cast(Op, __builtin_shufflevector(lo, hi, 0, 1, 2, 3));
      }
    }
  };
  constexpr int NFRAG = KS * (MT + NT) + (MX ? MT + NT : 0);
  auto pin = [&](Frags& x) {
    static_for<KS>([&](auto S_) {
      constexpr int s = decltype(S_)::value;
      static_for<MT>([&](auto T_) { lds_use(x.a[s][decltype(T_)::value]); });
      static_for<NT>([&](auto T_) { lds_use(x.b[s][decltype(T_)::value]); });
    });
    if constexpr (MX) {
      static_for<MT>([&](auto T_) { lds_use(x.sa[decltype(T_)::value]); });
      static_for<NT>([&](auto T_) { lds_use(x.sb[decltype(T_)::value]); });
    }
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      ring_pin(acc[i][j]);   // (cleared here: an assembly MFMA must not follow a register write of the compiler's within two slots)
    }

  // ---- prologue: the tail's loads, the first NS steps of the ring, then the fragments of step 0
  auto fill = [&](bool skip0) {
#pragma unroll
    for (int s = 0; s < NS; s++) {
      if (s < steps && !(s == 0 && skip0)) static_for<L>([&](auto Q_) { issue(Q_, lds0 + s * STAGE, std::true_type{}); });
      advance();
    }
    if (steps >= NS) wait_vmcnt<(NS - 1) * L>(); else wait_vmcnt<0>();   // (all but the youngest NS - 1 steps)
  };
  if (tail) {   // (one block from the loads to their use: at a join the compiler may copy registers still in flight)
    i32x4 ta[LA], tb[LB];
    const int kfull = p.k_bytes - tail;                       // bytes of K before the tail
    const int krows = p.K - kfull / E::kElemBytes;            // (a row-major B may end before the padded rows of A do)
    // The chunk that a row ends inside is read as the row's last 16 bytes and moved down: of K-contiguous rows at k_bytes, of rows of a
    // row-major B at N (past: bytes that the lane's chunk of load q reaches beyond).
    int past[LB];
#pragma unroll
    for (int q = 0; q < LB; q++) past[q] = 0;
    if (open_rows) {
      constexpr int CPR = BN / 8, RPI = 64 / CPR;
#pragma unroll
      for (int q = 0; q < LB; q++) {
        const int pc = lane % CPR, k = (wave * LB + q) * RPI + lane / CPR;
        const int chunk = min((((pc >> 1) ^ xor_of(k)) << 1) | (pc & 1), (p.N + 7) / 8 - 1 - n0 / 8);
        past[q] = max(0, (n0 + chunk * 8 + 8 - p.N) * 2);
      }
    }
    const char* kA = tileA + kfull;
    const char* kB = B_KMAJOR ? tileB + kfull : tileB + (int64_t)(kfull / 2) * p.ldb;
#pragma unroll
    for (int q = 0; q < LA; q++) load16_sbase<0>(ta[q], kA, voffA[q] + q * 1024 - chunkA[q] * 16 + min(chunkA[q] * 16, tail - 16));
#pragma unroll
    for (int q = 0; q < LB; q++) {
      if constexpr (B_KMAJOR) load16_sbase<0>(tb[q], kB, voffB[q] + q * 1024 - rowB[q] * 16 + min(rowB[q] * 16, tail - 16));
      else load16_sbase<0>(tb[q], kB, voffB[q] + q * 1024 - (unsigned)(rowB[q] - min(rowB[q], krows - 1)) * (unsigned)p.ldb - (unsigned)past[q]);
    }
    int ts = 0;   // (block-scaled: K is a multiple of 128 elements, so an MXFP4 tail is four blocks - one dword of scales - and there is no other)
    const int bs = wave % BLOCKS;
    if constexpr (MX) load4_sbase(ts, scale_base(bs) + kfull / RING_ROW * 4 * SD, scale_rows(bs));
    fill(true);
    const i32x4 zero = {0, 0, 0, 0};
    if constexpr (DWORDS) {
      // (landed, all of them: from here on branches may move them)
#pragma unroll
      for (int q = 0; q < LA; q++) lds_use(ta[q]);
#pragma unroll
      for (int q = 0; q < LB; q++) lds_use(tb[q]);
      if (tail & 15) {
#pragma unroll
        for (int q = 0; q < LA; q++) ta[q] = chunkA[q] * 16 + 16 <= tail ? ta[q] : bytes_down(ta[q], -tail & 15);
        if constexpr (B_KMAJOR) {
#pragma unroll
          for (int q = 0; q < LB; q++) tb[q] = rowB[q] * 16 + 16 <= tail ? tb[q] : bytes_down(tb[q], -tail & 15);
        }
      }
      if (open_rows) {
#pragma unroll
        for (int q = 0; q < LB; q++) tb[q] = past[q] > 0 ? bytes_down(tb[q], -2 * p.N & 15) : tb[q];
      }
    }
#pragma unroll
    for (int q = 0; q < LA; q++) {
      lds_use(ta[q]);
      *(LDS_PTR(i32x4))(uintptr_t)(lds0 + (wave * LA + q) * 1024 + lane * 16) = chunkA[q] * 16 < tail ? ta[q] : zero;
    }
#pragma unroll
    for (int q = 0; q < LB; q++) {
      lds_use(tb[q]);
      const bool in = B_KMAJOR ? rowB[q] * 16 < tail : rowB[q] < krows;
      *(LDS_PTR(i32x4))(uintptr_t)(lds0 + A_BYTES + (wave * LB + q) * 1024 + lane * 16) = in ? tb[q] : zero;
    }
    if constexpr (MX) {
      lds_use(ts);
#pragma unroll
      for (int d = 0; d < SD; d++)   // (2^0 beyond K: multiplies zeros)
        *(LDS_PTR(int))(uintptr_t)(lds0 + S_BYTES + (bs * SD + d) * 256 + lane * 4) = d == 0 ? ts : 0x7f7f7f7f;
    }
    lds_wait<0>();
  } else {
    fill(false);
  }
  block_barrier();
  static_for<NFRAG>([&](auto R_) { read_frag(R_, 0u, f[0]); });
  lds_wait<0>();
  pin(f[0]);

  // ---- one K step: every wave holds the step's fragments, so its stage can be refilled behind the barrier; the barrier
  // also says that the next stage has landed.  The next step's fragments and the refill are spread over the MFMAs.  (The last
  // step reads fragments that nobody uses from a stage that holds old data: one path through the code keeps the accumulators
  // and fragments in the same registers everywhere.)
  int s = 0;
  unsigned cur = 0;   // byte offset of step s's stage in the ring
  auto step = [&](auto P_, auto MORE_) {
    constexpr int P = decltype(P_)::value;
    constexpr bool more = decltype(MORE_)::value;
    constexpr int NL = more ? L : 0;
    const unsigned next = cur + STAGE == NS * STAGE ? 0u : cur + STAGE;
    if constexpr (more) wait_vmcnt<(NS - 2) * L>();   // (steps s + 2 .. s + NS - 1 may be under way)
    else ring_drain_wait<NS, L>(steps - s);
    block_barrier();
    static_for<NMFMA>([&](auto N_) {
      constexpr int n = decltype(N_)::value, ks = n / (MT * NT), i = (n / NT) % MT, j = n % NT;
      if constexpr (MX) E::template mma<ks>(f[P].b[ks][j], f[P].a[ks][i], acc[i][j], f[P].sb[j], f[P].sa[i]);
      else E::mma(f[P].b[ks][j], f[P].a[ks][i], acc[i][j]);
      // The reads over the first three quarters of the MFMAs, so that the last ones have returned by the end of the step; the
      // loads over all of them (behind each other they would wait for the memory pipeline, and the MFMAs behind them).
      constexpr int RS = NMFMA * 3 / 4;
      constexpr int r0 = n >= RS ? NFRAG : n * NFRAG / RS, r1 = n + 1 >= RS ? NFRAG : (n + 1) * NFRAG / RS;
      static_for<r1 - r0>([&](auto O_) { read_frag(std::integral_constant<int, r0 + decltype(O_)::value>{}, next, f[P ^ 1]); });
      constexpr int l0 = n * NL / NMFMA, l1 = (n + 1) * NL / NMFMA;
      static_for<l1 - l0>([&](auto O_) { issue(std::integral_constant<int, l0 + decltype(O_)::value>{}, lds0 + cur, std::false_type{}); });
      __builtin_amdgcn_sched_barrier(0);
    });
    lds_wait<0>();
    pin(f[P ^ 1]);
    advance();
    cur = next;
    s++;
  };
  using T = std::true_type; using F = std::false_type;
  using I0 = std::integral_constant<int, 0>; using I1 = std::integral_constant<int, 1>;
  // steps with a refill, then the last NS (all of a short K) without; the loops take two at a time
  const int refills = steps > NS ? steps - NS : 0;
  if (refills & 1) {
    step(I0{}, T{});
    f[0] = f[1];
  }
  while (s < refills) {
    step(I0{}, T{});
    step(I1{}, T{});
  }
  if ((steps - refills) & 1) {
    step(I0{}, F{});
    f[0] = f[1];
  }
  while (s < steps) {
    step(I0{}, F{});
    step(I1{}, F{});
  }
  // (the compiler does not know that the statements above are MFMAs: the last ones must have retired before it reads an
  // accumulator, and no read may move in front of the wait)
  asm volatile("s_nop 15" ::: "memory");
  static_for<MT>([&](auto I_) { static_for<NT>([&](auto J_) { ring_pin(acc[decltype(I_)::value][decltype(J_)::value]); }); });
  ring_epilogue<MT, NT>(acc, p, m0 + wm * TM, n0 + wn * TN, l16, kg);
#endif
}

// Splits of K: workgroup z * tiles + t multiplies the K bytes [z * chunk, z * chunk + chunk) of tile t into slice z of the
// workspace (chunk: whole K steps; 0 = no split).
template <typename E, int BM, int BN, int WN, bool B_KMAJOR, int NS, bool DWORDS>
__global__ __launch_bounds__(128 * WN, 1) void gemm_ring_kernel(GemmArgs p, int chunk_bytes) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int num_m = (p.M + BM - 1) / BM, num_n = (p.N + BN - 1) / BN, tiles = num_m * num_n;
  int t = blockIdx.x;
  if (chunk_bytes > 0) {
    const int z = t / tiles, k0 = z * chunk_bytes;
    t -= z * tiles;
    p.k_bytes = min(p.k_bytes - k0, chunk_bytes);   // (the host leaves no split empty)
    p.K -= k0 / E::kElemBytes;
    p.A += k0;
    p.B += B_KMAJOR ? (int64_t)k0 : (int64_t)(k0 / E::kElemBytes) * p.ldb;
    if constexpr (E::kScaleDwords > 0) { p.sA += k0 / E::kBlockBytes; p.sB += k0 / E::kBlockBytes; }
    p.C = (char*)(p.workspace + (int64_t)z * p.M * p.N);
    p.ldc = p.N; p.scn = 1; p.out_dtype = 4;        // fp32 partial sums, dense rows (the workspace is 16-byte aligned)
    p.c_vec_ok = p.N % 4 == 0;
    p.a_scale = nullptr; p.b_scale = nullptr; p.activation = 0; p.aux = nullptr;
  }
  int pm, pn;
  grouped_tile(xcd_remap(t, tiles), num_m, num_n, p.group_m, pm, pn);
  gemm_ring_tile<E, BM, BN, WN, B_KMAJOR, NS, DWORDS>(p, pm, pn, lds_addr((LDS_PTR(char))smem));
}

template <typename E, int BM, int BN, int WN, bool B_KMAJOR, int NS, bool DWORDS = false>
static int launch_gemm_ring(const GemmArgs& p, int splits, int chunk_bytes, hipStream_t stream) {
  constexpr int smem = NS * ring_stage_bytes<E, BM, BN>();
  static_assert(smem <= 160 * 1024, "LDS ring does not fit");
  static bool attr_set = false;  // benign race: setting the attribute twice is harmless
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_ring_kernel<E, BM, BN, WN, B_KMAJOR, NS, DWORDS>, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) return (int)e;
    attr_set = true;
  }
  const int tiles = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
  gemm_ring_kernel<E, BM, BN, WN, B_KMAJOR, NS, DWORDS><<<dim3(tiles * splits), dim3(128 * WN), smem, stream>>>(p, splits > 1 ? chunk_bytes : 0);
  return (int)hipGetLastError();
}

}  // namespace mi355
