// extern "C" entry points declared in include/mi355_kernels.h: argument validation, kernel
// family / tile selection, launch.  Plays the role of the generated launcher of the reference
// (third_party/amd/backend/driver.py:326-377): pointers and scalars in, one asynchronous
// launch on the caller's stream out, an integer status back.
#include <algorithm>
#include <cmath>
#include <utility>
#include <hip/hip_runtime.h>
#include <stdlib.h>
#include <string.h>
#include <atomic>
#include <climits>
#include <mutex>
#include "../../include/mi355_kernels.h"
#include "launch.h"

using namespace mi355;

namespace {

struct DeviceInfo {
  int ok = 0, cus = 0, gfx950 = 0, lds = 0, clock_khz = 0, wall_clock_khz = 0;
};

// properties of the CURRENT device, read once per device (a process may hold several)
const DeviceInfo& device_info() {
  constexpr int kMax = 64;
  static DeviceInfo infos[kMax];
  static std::atomic<int> ready[kMax];
  static std::mutex mutex;
  static const DeviceInfo none;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMax) return none;
  if (ready[dev].load(std::memory_order_acquire)) return infos[dev];
  std::lock_guard<std::mutex> lock(mutex);
  if (ready[dev].load(std::memory_order_relaxed)) return infos[dev];
  DeviceInfo& info = infos[dev];
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return none;
  info.cus = prop.multiProcessorCount;
  info.gfx950 = strncmp(prop.gcnArchName, "gfx950", 6) == 0;
  info.lds = (int)prop.sharedMemPerBlock;
  info.clock_khz = prop.clockRate;
  if (hipDeviceGetAttribute(&info.wall_clock_khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess) info.wall_clock_khz = 0;
  info.ok = 1;
  ready[dev].store(1, std::memory_order_release);
  return info;
}

// Tuning knobs from the environment (the reference's third configuration mechanism: environment
// variables read by the runtime, python/triton/runtime/jit.py:717, :848).  Read ONCE per process, at the
// first call that needs them, and again only when mi355_refresh_env() is called: a launch costs no getenv.
// UNSET = the variable is absent or empty and the call site's own default applies.
constexpr int UNSET = INT_MIN;
struct Knobs {
  int force_strided, group_m, tile, programs, skinny, grouped_big_min, grouped_wave128_min_k, grouped_chunk, grouped_shape, grouped_run,
      attn_fwd_variant, attn_bwd_groups, attn_programs, lean_epilogue, tile_m, rowfused_max_mk, mixed_rows, splitk;
};
Knobs g_knobs;
std::atomic<int> g_knobs_ready{0};
std::mutex g_knobs_mutex;

int read_env(const char* name, int lo) {
  const char* s = getenv(name);
  if (!s || !*s) return UNSET;
  const int v = atoi(s);
  return v < lo ? lo : v;   // (out-of-range values are clamped, never passed on to a kernel)
}

void load_knobs() {
  std::lock_guard<std::mutex> lock(g_knobs_mutex);
  Knobs k;
  k.force_strided = read_env("MI355_GEMM_FORCE_STRIDED", 0);
  k.group_m = read_env("MI355_GEMM_GROUP_M", 1);
  k.tile = read_env("MI355_GEMM_TILE", -1);   // (-1: the block-scaled products' one-thread-per-output kernel)
  k.programs = read_env("MI355_GEMM_PROGRAMS", 1);
  k.skinny = read_env("MI355_GEMM_SKINNY", 0);
  k.grouped_big_min = read_env("MI355_GROUPED_BIG_MIN", 1);
  k.grouped_wave128_min_k = read_env("MI355_GROUPED_WAVE128_MIN_K", 0);
  k.grouped_chunk = read_env("MI355_GROUPED_CHUNK", 1);
  k.grouped_shape = read_env("MI355_GROUPED_SHAPE", 0);   // of group_plan: 0, 2, 4 or 5 (others: its choice)
  k.grouped_run = read_env("MI355_GROUPED_RUN", 0);       // tiles that an XCD takes at a time (0: an eighth of all)
  k.attn_fwd_variant = read_env("MI355_ATTN_FWD_VARIANT", 0);
  k.attn_bwd_groups = read_env("MI355_ATTN_BWD_GROUPS", 0);   // dQ groups + 16 * dK/dV groups
  k.attn_programs = read_env("MI355_ATTN_PROGRAMS", 1);
  k.lean_epilogue = read_env("MI355_GEMM_LEAN_EPILOGUE", 0);
  k.tile_m = read_env("MI355_GEMM_TILE_M", 0);
  k.rowfused_max_mk = read_env("MI355_ROWFUSED_MAX_MK", 0);
  k.mixed_rows = read_env("MI355_GEMM_MIXED_ROWS", 0);
  k.splitk = read_env("MI355_GEMM_SPLITK", 0);   // 0: matmul's own route never splits K
  g_knobs = k;
  g_knobs_ready.store(1, std::memory_order_release);
}

const Knobs& knobs() {
  if (!g_knobs_ready.load(std::memory_order_acquire)) load_knobs();
  return g_knobs;
}

int knob(int value, int dflt) { return value == UNSET ? dflt : value; }

// Two tile heights in one launch (gemm_wave128_mixed_kernel and its fp8 / block-scaled forms): the rows of C to give to
// the 256-row tiles, the rest going to 192-row tiles, for a product of M rows and nn tile columns on P programs - or 0
// when no split is rated 5 % better than one tile height.  A split is rated by its busiest program (tiles b, b + P, ...
// of the first part and P - 1 - b, ... of the second; a 192-row tile counted as 0.78 of a 256-row one: 3072^3 on 192
// of them against 4096^3 on 256 tiles, per tile and K step); among the splits within 7 % of the best, the one whose two
// parts are closest in work is taken (measured: 5120^3 bf16 1164 / 1280 / 1325 TFLOP/s for 100 + 400 / 160 + 320 / 220 +
// 240 tiles, which the count rates the same).
int mixed_split(int M, int nn, int P) {
  if (M % 256 != 0 || nn <= 0 || P <= 0) return 0;
  auto count = [&](long tiles, int b) { return b < tiles ? (tiles - b + P - 1) / P : 0; };
  const long tiles256 = (long)(M / 256) * nn;
  double one_height = (double)((tiles256 + P - 1) / P), best = 1e30;   // in units of a 256-row tile's time
  if (M % 192 == 0) one_height = std::min(one_height, 0.78 * (double)(((long)(M / 192) * nn + P - 1) / P));
  auto busiest = [&](int a) {
    const long n256 = (long)a * nn, n192 = (long)((M - a * 256) / 192) * nn;
    double worst = 0;
    for (int b = 0; b < P; b++) worst = std::max(worst, (double)count(n256, b) + 0.78 * (double)count(n192, P - 1 - b));
    return worst;
  };
  for (int a = 1; a * 256 < M; a++)
    if ((M - a * 256) % 192 == 0) best = std::min(best, busiest(a));
  if (!(best < 0.95 * one_height)) return 0;
  int best_rows = 0;
  double best_gap = 1e30;
  for (int a = 1; a * 256 < M; a++) {
    if ((M - a * 256) % 192 != 0 || busiest(a) > 1.07 * best) continue;
    const double gap = std::abs((double)a * nn - 0.78 * (double)((M - a * 256) / 192) * nn);
    if (gap < best_gap) { best_gap = gap; best_rows = a * 256; }
  }
  return best_rows;
}

int elem_size(int dtype) {
  switch (dtype) {
    case MI355_F16: case MI355_BF16: return 2;
    case MI355_F8E4M3: case MI355_F8E5M2: return 1;
    case MI355_F32: return 4;
    default: return 0;
  }
}

// What the ring kernels (gemm_ring.h) would take for a product of `steps` 128-byte K steps, in us: a round of one tile per
// CU costs its prologue and epilogue plus its K steps; splits of K add the slices' way through memory and a second launch.
// Fitted to 60 shapes from 256 to 8192 (bf16, fp16, e4m3, both layouts of B): within 15 % except where the operands' pitch
// is not a multiple of 128 bytes (every line is then fetched in two pieces: up to 1.5 times as long, for every kernel alike).
// One row or column of tiles against a long weight is a stream from memory: a CU gets about 30 GB/s of lines that no other CU
// asks for (64 x 8192 x 8192 fp16, 128 tiles of 64x64: 48 us with rings of four and of eight stages alike, 35 us with two
// splits), so that there the splits also buy bandwidth.
struct RingPlan { int shape, splits; double us; };   // shape: 0 = tiles of 128x128, 1 = 128x64, 2 = 64x64, 3 = 64x32

// Ring tiles of 64x32, eight steps deep, for up to 64 rows next to a K-major weight: twice the workgroups of 64x64 tiles without a
// split and its second launch, one round of CUs.  Measured over 16 .. 64 rows, 1024 .. 16384 columns, K bytes of 2048 .. 16384, fp16 and
// e4m3, weights from memory, us, the best of the other rings, splits and the streaming kernel / these tiles: e4m3 33 x 8192 x 8192 18.2 /
// 13.7, 64 x 8192 x 8192 18.6 / 16.8, 48 x 4096 x 4096 8.3 / 6.9, 24 x 6016 x 5376 8.6 / 8.2; fp16 24 x 4096 x 4096 11.1 / 9.5, 33 x 6016 x 5376 22.0 /
// 15.5, 48 x 3000 x 2304 8.4 / 7.1; beyond one round behind (64 x 12288 x 4096 27 / 33).  A row-major weight's 64-byte pieces are no
// faster on them (fp16 64 x 8192 x 8192 34.5 / 45).
bool thin_ok(int M, int N, int64_t k_bytes, bool b_kmajor, int cus) { return b_kmajor && M <= 64 && (N + 31) / 32 <= cus && k_bytes > 2048; }

constexpr double kLaunchUs = 3.5;
RingPlan ring_plan(int M, int N, int steps, int cus, int splits_lo, int splits_hi, double step_share = 1.0, bool thin = false) {
  const double streamed = 128.0 * steps * std::max(M, N);   // bytes of the longer operand
  static const struct { int bm, bn; double round_us, step_us; } kShapes[3] = {{128, 128, 2.5, 0.42}, {128, 64, 1.5, 0.265}, {64, 64, 0.6, 0.165}};
  RingPlan best{0, 1, 1e30};
  for (int shape = 0; shape < 3; shape++) {
    const auto& t = kShapes[shape];
    const double step_us = (M <= t.bm || N <= t.bn) && streamed >= 64e6 ? std::max(t.step_us, (M <= t.bm ? t.bn : t.bm) * 128 / 30e3) : t.step_us * step_share;
    const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    for (int splits = splits_lo; splits <= splits_hi; splits++) {
      const int per = (steps + splits - 1) / splits;
      const long rounds = (tiles * splits + cus - 1) / cus;
      // (several rounds overlap a little at their ends, and keep the operands' lines moving for a sixth more per step)
      const double n = rounds > 1 ? 0.5 * ((double)rounds + (double)tiles * splits / cus) : 1.0;
      double us = kLaunchUs + n * (t.round_us + per * step_us * (rounds > 1 ? 1.18 : 1.0));
      if (splits > 1) us += 2.5 + (double)splits * M * N * 8.0 / 3e6;   // (written and read again at about 3 TB/s)
      if (us < best.us) best = {shape, splits, us};
      if (splits > 1 && rounds > 1) break;   // (more splits only add rounds)
    }
  }
  // 64x32 tiles (thin_ok): a step is latency, or the weight's way - from memory where it is larger than the last-level cache keeps next
  // to others (fp16, 24 rows, 128 tiles: 4096 x 4096, 33 MB, 9.4 us, 4096 x 8192, 67 MB, 20.0 - two splits of 64x64 tiles 16.2)
  const long tiles = (N + 31) / 32;
  const bool far = N * 128.0 * steps > 48e6;
  for (int splits = splits_lo; thin && splits <= splits_hi && tiles * splits <= cus; splits++) {
    const int per = (steps + splits - 1) / splits;
    const double rows = std::max(M - 16, 0);
    double us = 3.2 + per * std::max(far ? 0.15 + 1.4e-3 * std::max(M - 24, 0) : 0.095 + 4.5e-4 * rows, far ? 7.6e-4 * tiles * splits + 1.05e-3 * rows : 7.1e-4 * tiles * splits + 6e-4 * rows);
    if (splits > 1) us += 2.5 + (double)splits * M * N * 8.0 / 3e6;
    if (us < best.us) best = {3, splits, us};
  }
  return best;
}

// The same plan against kernels of other tiles: what one split's rounds take (195 products of up to 2800 tiles and 4 .. 64 steps: within 6 %
// rms).  The estimates above, up to a fifth longer for several rounds, are for the choice among the rings and splits that they were fitted to.
double ring_rounds_us(int M, int N, int steps, int cus, int shape) {
  static const struct { int bm, bn; double round_us, step_us, whole; } kShapes[3] = {{128, 128, 3.4, 0.365, 0.86}, {128, 64, 2.2, 0.25, 0.91}, {64, 64, 1.1, 0.158, 0.7}};
  const auto& t = kShapes[shape];
  const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn), rounds = (tiles + cus - 1) / cus;
  return 1.2 + (rounds > 1 ? t.whole * rounds + (1.0 - t.whole) * tiles / cus : 1.0) * (t.round_us + steps * t.step_us * (rounds > 1 ? 1.0 : 1.04));
}

// Ring tiles of 128x128 in two stages, two workgroups on a CU (more tiles than CUs only): while one waits for its first steps or stores, the other
// multiplies, which four stages with a CU to themselves pay for in every tile.  us, before / so: bf16 K-major 3200 x 3072 x 192 19.6 / 11.4, 3456 x 1664 x 256
// 11.1 / 8.2, row-major B 1408 x 6784 x 192 19.4 / 11.9, 3840 x 5376 x 448 37.7 / 27.0, 8064 x 2048 x 576 32.4 / 26.5; e4m3 1536 x 4224 x 640 13.0 / 10.8, 4352 x 5888
// x 384 28.5 / 25.0; MXFP4 6400 x 4224 x 768 34.3 / 24.2, 2432 x 4992 x 1280 22.4 / 16.9, MXFP8 4224 x 4992 x 384 30.1 / 18.6.  A long K hides the waits anyway, and
// two stages less of the latency: K-major 3712 x 4736 x 1920 63.7 / 77.4, e4m3 5376 x 2304 x 2048 26.0 / 33.6, MXFP8 3584 x 3968 x 4352 60.7 / 89.2, 3543 x 5760 x 4736 117 / 125 (block-scaled products of more than sixteen steps are left out); up to a round of tiles
// a workgroup is alone either way: 1024 x 3712 x 768 9.5 / 10.2.  (150 products of 200 .. 3000 tiles and 2 .. 40 steps: within 6 % rms, block-scaled 12.)
// `apart`: rows that do not begin on 128-byte lines (K-major bf16 2048 x 7808 x 984 37.8 / 44.0).  `epilogue`: us a round for what C takes beyond plain stores.
double pairs_us(int M, int N, int steps, int cus, bool mx, bool apart, double epilogue = 0.0) {
  const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128), rounds = (tiles + cus - 1) / cus;
  if (tiles <= cus || (mx && steps > 16)) return 1e30;
  const double k = (apart ? 1.5 : 1.0) * steps;
  return mx ? 1.2 + (double)rounds * (1.9 + 0.6 * k) : 1.2 + (0.8 * rounds + 0.2 * tiles / cus) * (2.0 + epilogue + 0.45 * k);
}

// A group on the ring kernels, its problems in `order`, the longest K first: which tiles (0 = 128x128, 2 = 64x64, 4 = 128x128 in two stages, 5 = each
// problem on 0 or 2 by its cost) and in which order.
// chunk: an eighth of the tiles for each XCD, one after the other (0), keeps the operands in its L2; but where the first eighth has the tiles of
// the longest K, one XCD works when the others are done: then runs of `chunk` tiles are dealt to the XCDs in turn.
// us, eighths | runs, of shapes 2 / 0 / 4 / 5: twelve problems of 80 .. 1904 rows and K of 88 .. 1832 27.5 / 31.5 / 25.7 / 31.6 | 14.3 / 18.8 / 24.0 / 19.0,
// seven of 192 .. 2048, K of 128 .. 2048 40.3 / 30.9 / 30.2 / 31.8 | 24.5 / 21.5 / 27.5 / 21.7; twelve of 64 .. 1792, K of 64 .. 768 11.1 / 10.9 / 12.8 / 9.0 |
// 10.8 / 11.2 / 13.0 / 9.3; seven 512 -> 4096 31.2 / 28.8 / 23.0 / 29.7 | 31.2 / 29.3 / 23.7 / 29.0; seven of 20 .. 1110 x 872 x 664 15.1 / 11.7 / 13.1 / 11.9 | 17.7 / 12.9
// / 14.4 / 13.0; nine of 21 .. 1686 x 448 x 1088 10.5 / 12.7 / 15.9 / 12.8 | 12.0 / 13.1 / 17.3 / 13.1.
// The estimate of each (1360 drawn groups of 2 .. 16 problems: within 9 to 12 % rms) is base + the largest of one tile of the longest K (`lone`) and, w : 1 - w, of what
// the CU with the most tiles of the first problems has (most, `slots` workgroups a CU) and all tiles' time spread over the CUs, or over those of the first XCD;
// `runs`: what their misses in the L2 cost.  Another form than the one of least cost, in eighths, has to be estimated 2 % shorter: of 1000 other drawn groups 17 are then
// more than 2 % slower than by cost alone, six more than 5 % and one more than 10, and in the geometric mean they are 1.184 times as fast (5 %: the same 17, 1.182, but 85
// for 70 groups more than 2 % behind a choice by a coarser estimate of three forms; no margin: 23, nine and one, 1.185); the best of the eight forms is 1 % ahead of the one taken.
struct GroupPlan { int shape, chunk; uint64_t small_tiles; };   // small_tiles: the problems on 64x64, a bit for each of `order`
GroupPlan group_plan(const int32_t* sizes, const int* order, int n, int cus, int forced) {
  struct Tile { double us, step_us; };
  static const struct { int shape, slots, chunk; double base; Tile large, small; double most, w, lone, lone_step, runs; } kForms[4] = {
      {2, 2, 16, 3.06, {0.0, 0.0}, {0.97, 0.258}, 0.72, 0.376, 0.64, 0.13, 1.11}, {0, 1, 8, 3.2, {3.92, 0.594}, {0.0, 0.0}, 0.68, 0.541, 2.02, 0.31, 1.09},
      {4, 2, 8, 2.36, {2.14, 0.634}, {0.0, 0.0}, 1.24, 0.559, 2.96, 0.2, 1.11}, {5, 1, 8, 3.52, {3.63, 0.565}, {1.2, 0.235}, 0.77, 0.55, 0.0, 0.15, 1.08}};
  // Which shape costs least: all tiles' time (at the rates of ring_plan with several rounds under way) over the CUs, one tile at least.
  double steps[GroupedTable::kMax], tiles64[GroupedTable::kMax], tiles128[GroupedTable::kMax];
  double all[3] = {0.0, 0.0, 0.0}, top[3] = {0.0, 0.0, 0.0};   // on 64x64, on 128x128, each on the better one
  uint64_t better64 = 0;
  for (int i = 0; i < n; i++) {
    const int32_t* s = sizes + 3 * order[i];
    steps[i] = (s[2] + 63) / 64;
    tiles64[i] = (double)((s[0] + 63) / 64) * ((s[1] + 63) / 64);
    tiles128[i] = (double)((s[0] + 127) / 128) * ((s[1] + 127) / 128);
    const double one64 = 0.6 + 0.195 * steps[i], one128 = 2.5 + 0.5 * steps[i], us64 = one64 * tiles64[i], us128 = one128 * tiles128[i];
    const bool small = us64 <= us128;
    if (small) better64 |= 1ull << i;
    all[0] += us64; all[1] += us128; all[2] += small ? us64 : us128;
    top[0] = std::max(top[0], one64); top[1] = std::max(top[1], one128); top[2] = std::max(top[2], small ? one64 : one128);
  }
  for (int e = 0; e < 3; e++) all[e] = std::max(all[e] / cus, top[e]);
  const int least = all[0] <= all[1] && all[0] <= all[2] ? 2 : all[1] <= all[2] ? 0 : 5;
  auto small_of = [&](int shape) { return shape == 2 ? ~0ull : shape == 5 ? better64 : 0ull; };

  GroupPlan best{least, 0, small_of(least)};
  double best_us = 1e30, least_us = 1e30;
  for (const auto& f : kForms) {
    if (forced >= 0 && f.shape != forced) continue;
    const uint64_t small = small_of(f.shape);
    const double slots = f.slots * cus;
    double eighth = 0.0, tiles = 0.0, sum = 0.0, most = 0.0, first = 0.0;
    for (int i = 0; i < n; i++) eighth += small >> i & 1 ? tiles64[i] : tiles128[i];
    eighth *= 0.125;
    for (int i = 0; i < n; i++) {
      const bool s = small >> i & 1;
      const double us = s ? f.small.us + f.small.step_us * steps[i] : f.large.us + f.large.step_us * steps[i], count = s ? tiles64[i] : tiles128[i];
      first += us * std::max(0.0, std::min(count, eighth - tiles));
      tiles += count;
      sum += count * us;
      most = std::max(most, f.most * us * (double)((int64_t)((tiles - 1.0) / slots) + 1));
    }
    const double lone = f.lone + f.lone_step * steps[0];
    auto blend = [&](double spread) { return std::max(lone, f.w * most + (1.0 - f.w) * spread / cus); };
    const double eighths = f.base + blend(std::max(sum, 8 * first)), runs = f.base + f.runs * blend(sum);
    if (f.shape == least) least_us = eighths;
    // (both tile sizes in eighths where one of them costs less: estimated shorter, but 17.2 -> 20.7 and 22.5 -> 26.3)
    if (eighths < best_us && (f.shape != 5 || least == 5 || forced >= 0)) { best = {f.shape, 0, small}; best_us = eighths; }
    if (runs < best_us) { best = {f.shape, f.chunk, small}; best_us = runs; }
  }
  return best_us < 0.98 * least_us ? best : GroupPlan{least, 0, small_of(least)};
}

// The same for the kernels of 256-column tiles with `rows` rows of C each (gemm_wave128.hip; edges: the eight-wave kernel, for
// what that one does not take).  A K step of a 256-row tile is bound by its 64 KiB of operands and by power: with idle CUs it is
// somewhat shorter, and several rounds are dealt evenly, so that an unfilled last round is spread over all of them.  180 products
// of 64 .. 768 tiles and 8 .. 128 steps, bf16 in both layouts and e4m3: within 3 % rms, 11 % at most.
double tiles256_us(long tiles, int rows, int steps, int cus, bool edges, bool fp8) {
  const long rounds = (tiles + cus - 1) / cus;
  const double fill = (double)tiles / (double)(rounds * cus), busy = rounds > 1 ? 0.48 + 0.52 * fill : 0.62 + 0.38 * fill;
  const double share = rows == 256 ? 1.0 : rows == 192 ? 0.78 : 0.64, step = (fp8 ? 1.28 : 1.34) * (edges ? fp8 ? 1.0 : 1.12 : 1.0);
  return 3.2 + (double)rounds * share * ((edges ? 10.0 : 8.0) + step * busy * steps);
}

// A product that needs part of one more round of tiles, in two calls: rows (or columns) for whole rounds of CUs - of 256 x 256 tiles,
// or of 128x128 ring tiles where those are what it runs on -, the rest on whatever is best for it; and up to 64 columns or rows beyond
// whole 256-column tiles likewise.  `tile` as in gemm_impl (1: ring kernels only, 6: four-wave kernels; else the eight-wave one),
// `ring` the ring shape that one call would take or -1.  us of a call, in one / in two parts: e4m3 6707 x 2944 x 3968 78 / 69, fp16 6016
// x 2880 x 7232 255 / 209, bf16 4100 x 4096 x 4096 135 / 99 (K-major B 129 / 93), 2050 x 8192 x 4096 136 / 101, 4096 x 4160 x 1024 50 / 38; on ring
// tiles bf16 5696 x 832 x 3456 48.1 / 41.8, fp16 2048 x 2560 x 2048 35.8 / 31.5.  No round saved, one part: 2048 x 2052 x 4096, 6150 x 6144 x 4096.
struct Cut { int m, n; double us; };   // sizes of the first part
Cut best_cut(int M, int N, int steps, int cus, int tile, int ring, bool is8) {
  const bool rounds = tile == 6 || tile == 1;
  auto best_us = [&](int m, int n) {
    const RingPlan plan = ring_plan(m, n, steps, cus, 1, 1);
    const double ring_us = rounds ? ring_rounds_us(m, n, steps, cus, plan.shape) : plan.us;
    if (tile == 1 || (tile == 6 && (m < 256 || n < 256))) return ring_us;
    return std::min(ring_us, tiles256_us((long)((m + 255) / 256) * ((n + 255) / 256), 256, steps, cus, tile != 6, is8));
  };
  Cut best{M, N, 1e30};
  auto cut = [&](int m, int n) {
    if (m <= 0 || n <= 0 || (m >= M && n >= N)) return;
    const double us = best_us(m, n) + (m < M ? best_us(M - m, N) : best_us(M, N - n));
    if (us < best.us) best = {m, n, us};
  };
  auto whole_rounds = [&](int edge) {
    const int nn = (N + edge - 1) / edge, mm = (M + edge - 1) / edge;
    const long tiles = (long)nn * mm;
    if (tiles <= cus) return;
    const int slots = (int)(tiles / cus) * cus;
    cut(std::min(M, slots / nn * edge), N);
    cut(M, std::min(N, slots / mm * edge));
  };
  const int rn = N % 256, rm = M % 256;
  if (tile != 1 && rn > 0 && rn <= 64 && N > 256) cut(M, N - rn);
  if (tile != 1 && rm > 0 && rm <= 64 && M > 256) cut(M - rm, N);
  if (tile == 6) whole_rounds(256);
  if (ring == 0 && rounds) whole_rounds(128);
  return best;
}

// Products of a short K whose 128x128 tiles are more than the CUs: the kernel of one barrier per 64-byte step on those tiles, two
// workgroups on a CU where a ring leaves room for one.  Measured over 16 .. 1280 tiles and K bytes of 16 .. 2048, this kernel / ring or
// 256x256 tiles, us: 2688 x 2688 x 64 fp16 8.2 / 11.5, x 192 11.5 / 13.2, x 256 12.4 / 13.0; e4m3 x 384 10.6 / 12.6, x 512 12.3 / 12.7; row-major B, x 256
// 12.0 / 13.6; edges cost it more (2659 x 2656 x 64 9.4 / 11.4, x 192 12.2 / 13.0).  Up to half as many tiles, whole ones only (1792 x 1920 x 64 6.0 / 7.1, 1763 x 1888
// 1.06).  Not where one round of 256x256 tiles fills the CUs (3840 x 4096 x 16 1.1).  With more tiles than CUs the rings of two stages take them, that kernel /
// ring: fp16 3840 x 1792 x 256 11.1 / 8.2, row-major B 1642 x 3586 x 128 14.8 / 10.2, but where one_barrier_ahead says otherwise.
bool short_k(int M, int N, int k_bytes, bool b_kmajor, int cus) {
  const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128), tiles256 = (long)((M + 255) / 256) * ((N + 255) / 256);
  if (tiles256 <= cus && tiles256 * 10 >= cus * 9) return false;
  if (tiles > cus) return k_bytes <= (!b_kmajor && tiles * 4 <= cus * 7 ? 512 : 384);
  return M % 128 == 0 && N % 128 == 0 && k_bytes <= 256 && tiles * 2 > cus;
}

// Which of those products of more tiles than CUs stay on that kernel: its steps are 64 bytes long, the rings' 128, so that where half of the last one would be empty, or
// there are few anyway, it is ahead - with whole columns of tiles, since edges there cost it more.  us, that kernel / rings of two stages, by K bytes: e4m3 5120 x 3712 x 64
// 13.1 / 16.8, 4096 x 2304 x 64 9.1 / 11.1, 2432 x 3456 x 192 9.9 / 11.2, 4096 x 1664 x 320 8.6 / 9.7, 2944 x 5888 x 128 15.0 / 16.0; fp16 768 x 6400 x 64 6.3 / 6.7; the
// time ratio, 100 products of each type, e4m3 64 0.84, 128 0.97, 192 0.92, 256 1.04, 320 0.91, 384 1.04; row-major B 64 0.90, 128 0.99, 192 0.93, 256 1.06, 320 0.98; K-major 64
// 0.90, 128 1.02, 144 1.03, 192 0.95, 256 1.09, 320 1.0.  Other N: e4m3 64 0.92 above two rounds, else 1.04 and more.
bool one_barrier_ahead(int M, int N, int k_bytes, bool is8, bool b_kmajor, int cus) {
  const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128);
  if (N % 128 != 0) return is8 && k_bytes <= 64 && tiles > 2 * cus;
  if (is8) return k_bytes <= 192 || (k_bytes > 256 && k_bytes <= 320);
  return b_kmajor ? k_bytes <= 64 || (k_bytes > 160 && k_bytes <= 192) : k_bytes <= 192;
}

// Operands as the ring kernels want them, on top of what every tile kernel asks (16-byte chunks, or dword_rows): 16-bit with either layout
// of B, fp8 with a K-major one.
bool ring_ok(int elem_bytes, bool b_kmajor) { return elem_bytes == 2 || (elem_bytes == 1 && b_kmajor); }

// Whether the streaming kernel (gemm_skinny.hip: a workgroup per 32 rows of the long operand, K split over its four waves)
// takes a product of at most 64 rows on a side ahead of the ring kernels (17 .. 64 rows of C next to a K-major weight are the 64x32 ring
// tiles', `thin`: the figures of 33 rows and more below hold for the columns of C, and for what those tiles are compared with).  Measured over rows 1 .. 64, long sides of 1024 ..
// 32768, K of 512 .. 16384, fp16 and e4m3, all layouts, weights from memory and from cache; ring / streaming, us:
//   * a K-contiguous long operand: as long as its workgroups are one round of CUs (16 x 8192 x 2048 fp16 12.0 / 10.0, 16 x
//     12288 x 2048 12 / 16.5), from 2048 bytes of K on (16 x 4096 x 512 fp16 4.6 / 4.6; below, the ring up to 15 % ahead) - for
//     the columns of C with any K (4096 x 16 x 512 e4m3 even, x 1024 1.07 times as long in the ring).  33 .. 40 rows: from 8192
//     bytes of K on (33 x 2048 x 8192 fp16 33.3 / 29.9, e4m3 18.9 / 17.6; x 4096 e4m3 even; 48 rows: ring 34.7 / 36.5); 49 .. 64
//     rows of 16 bits, whose own form moves whole lines: the same (64 x 2048 x 8192 37.0 / 30.6, 8192 x 64 x 8192 42.4 / 38.1, x 2048
//     even - with the weight in memory; from cache the ring is up to 30 % ahead there), fp8: ring (64 x 4096 x 8192 0.88)
//   * a row-major long operand: up to 32 rows, three quarters of a round (16 x 2048 x 2048 fp16 8.1 / 6.3 from cache, even from
//     memory; 16 x 8192 x 8192 39 / 43)
bool streams(int M, int N, int64_t k_bytes, int elem_bytes, bool b_kmajor, int cus, bool thin = true) {
  const bool cols = M > 64;
  // (64x32 ring tiles: above 16 rows, and below from 70 % of a round of CUs on - 16 x 8192 x 8192 fp16 33.6 / 29.0, e4m3 13.7 / 13.2; 16 x
  // 4096 x 8192 e4m3 8.8 / 9.3)
  // (but not next to a weight of 44 MB (fp8: 47) and more, which is memory's to bound: 1 x 6016 x 24832 fp16 33.1 / 28.1, 4 x 6144 x 10496 bf16 16.4 / 14.1, 8 x
  // 7008 x 4096 17.1 / 13.0, 12 x 7424 x 7168 e5m2 13.1 / 10.9; smaller ones 6.2 / 6.6; fp8 to 9000 bytes of K: 4 x 6912 x 11520 13.9 / 14.6.  More than eight (twelve) rows
  // only up to 64 MiB: 16 x 7680 x 4096 fp16 18.3 / 14.5, x 6272 e5m2 12.5 / 10.8.  Now and then behind: 8 x 6656 x 8192 bf16 25.1 / 27.7; from cache 3 %)
  const double weight = (double)N * k_bytes;
  const bool far = (elem_bytes == 2 ? weight >= 44e6 : weight >= 47e6 && k_bytes < 9000) && (M <= (elem_bytes == 2 ? 8 : 12) || weight < 64.0 * (1 << 20));
  if (!cols && thin && thin_ok(M, N, k_bytes, b_kmajor, cus) && (M > 16 || ((N + 31) / 32 * 10 > cus * 7 && !far))) return false;
  const int S = cols ? N : M, L = cols ? M : N;
  const bool y_kmajor = cols || b_kmajor;
  if (!gemm_skinny_sizes_ok(S, L, k_bytes, y_kmajor, cols ? b_kmajor : true, elem_bytes)) return false;
  if (!y_kmajor) return L <= 24 * cus;
  if (L > 32 * cus) return false;
  if (S <= 32) return cols || k_bytes >= 2048;
  return k_bytes >= 8192 && (S <= 40 || (elem_bytes == 2 && S > 48));
}

// fp8 and up to four rows against a long side that is not whole blocks of 32: the kernel that streams straight into registers
// (gemm8.hip; 1 x 2056 x 2048 5.4 / 5.0, 1 x 1000 x 4096 7.6 / 7.2, 8 x 2056 x 2048 even, 16 x 8200 x 2048 the ring 15 % ahead)
bool streams8(int M, int N, int64_t k_bytes, int elem_bytes, bool b_kmajor, int cus) {
  return elem_bytes == 1 && b_kmajor && M <= 4 && N % 32 != 0 && N <= 32 * cus && k_bytes % 256 == 0;
}

// us of a product that `streams` says yes to: within 15 % with K-contiguous operands, 30 % with a row-major long one (a weight
// from cache that much faster, from memory slower)
double stream_us(int M, int N, int64_t k_bytes, bool b_kmajor, int cus) {
  const double steps = (double)k_bytes / 128, fill = (double)std::max(M, N) / (32.0 * cus);
  if (M <= 64 && !b_kmajor) return 2.5 + steps * std::max(0.2, 0.33 * fill);
  const int rows = std::min(M, N);
  if (rows > 32) return 5.0 + steps * std::max(0.17, 0.24 * fill);
  return rows > 16 ? 3.9 + steps * std::max(0.152, 0.235 * fill) : 3.5 + steps * std::max(0.105, 0.18 * fill);
}

// Splits of K that `mi355_gemm_splitk` takes by itself (1 = the plain call).  thin_too = false: without the 64x32 ring tiles.
int auto_splits(int M, int N, int64_t k_bytes, int in_dtype, bool b_kmajor, bool ring, int cus, bool thin_too = true) {
  if (ring) {
    const int steps = (int)((k_bytes + 127) / 128);
    // (up to 64 rows or columns: nothing to gain from 32 K steps - 64 x 2048 x 2048 fp16 8.4 us, in the best splits 9.6, 1 x
    // 1000 x 4096 e4m3 7.6 / 10.2; 64 x 2048 x 4096 18.0 / 12.1 - or in slices of fewer than eight)
    const bool few = std::min(M, N) <= 64, stream = streams(M, N, k_bytes, elem_size(in_dtype), b_kmajor, cus, thin_too);
    const int most = (int)std::min<int64_t>(std::min<int64_t>(32, steps / (few ? 8 : 2)), (64ll << 20) / std::max<int64_t>(1, 4ll * M * N));   // 64 MiB of partial sums
    if (most < 2 || steps < (few ? 48 : 16)) return 1;   // (below that a second launch costs more than the K steps it would save)
    const bool thin = !stream && thin_too && thin_ok(M, N, k_bytes, b_kmajor, cus);
    const double plain = stream ? stream_us(M, N, k_bytes, b_kmajor, cus)
                                : std::min(ring_plan(M, N, steps, cus, 1, 1, 1.0, thin).us,
                                           tiles256_us((long)((M + 255) / 256) * ((N + 255) / 256), 256, steps, cus, false, elem_size(in_dtype) == 1));
    const RingPlan split = ring_plan(M, N, steps, cus, 2, most, 1.0, thin);
    // (columns that are not groups of four are added up one by one: 8192 x 33 x 8192 e4m3 19.0 us, in two slices 22.1;
    // and the few workgroups that add up many slices take 0.4 us for each: 16 x 320 x 4704 fp16 9.1 us, in nine slices 10.2)
    const double sums = few ? (N % 4 != 0 ? 1.5 : 0.0) + 0.4 * std::max(0, split.splits - 4) : 0.0;
    // (next to 64x32 tiles: a weight from memory at 5.8 TB/s at best - 16 x 8192 x 8192 fp16, two splits, 25 us by their steps, measured 32)
    const double least = thin && 128.0 * steps * N >= 64e6 ? kLaunchUs + 2.5 + 128.0 * steps * N / 5.8e6 + (double)split.splits * M * N * 8.0 / 3e6 : 0.0;
    return std::max(split.us, least) + sums < (stream ? 0.8 : 0.95) * plain ? split.splits : 1;
  }
  // the one-barrier-per-step kernel on 128x128 tiles, 64-byte K steps: a workgroup per CU, at least sixteen K steps each, at most
  // 32 slices; nothing to gain from half a round of tiles on or below 64 K steps
  const int small = std::min(M, N);
  if (small <= 32) return 1;
  const long tiles = (long)((M + 127) / 128) * ((N + 127) / 128);
  const int ksteps = (int)((k_bytes + 63) / 64);
  long splits = tiles * 2 > cus || ksteps < 64 ? 1 : std::min<long>(std::min<long>(cus / tiles, ksteps / 16), 32);
  if (in_dtype == MI355_F32) {
    // bound by the fp32 MFMA rate alone: a CU takes 1.05 us for a K step of every 128x128 tile that it has, so what counts is how
    // many that is on the fullest CU; the slices' way through memory and the second launch come on top.  (A workgroup or two for every
    // CU, whatever the remainder, was up to 1.6 times as long as the unsplit product: 2048 x 1920 x 256 40.7 us for 25.8; 1024 x 1408 x
    // 4096 in six slices 149, in five 121, unsplit 271)
    auto us = [&](long s) { return (double)((tiles * s + cus - 1) / cus) * ((ksteps + s - 1) / s) * 1.05 + (s > 1 ? 5.0 + (double)s * M * N * 8.0 / 6e6 : 0.0); };
    splits = 1;
    for (long s = 2; tiles < cus && s <= std::min<long>(32, ksteps / 8); s++)
      if (us(s) < us(splits)) splits = s;
  }
  splits = std::min<long>(splits, (64ll << 20) / std::max<int64_t>(1, 4ll * M * N));
  return splits >= 2 ? (int)splits : 1;
}

// Whether an addend's elements lie among C's (a call that adds in place).
bool addend_in_c(const GemmArgs& p) {
  if (!p.aux) return false;
  auto span = [&](const void* at, int64_t sm, int64_t sn, int dtype) {   // (strides of either sign)
    const int64_t m = (p.M - 1) * sm, n = (p.N - 1) * sn;
    const char* first = (const char*)at + (std::min<int64_t>(m, 0) + std::min<int64_t>(n, 0)) * elem_size(dtype);
    return std::pair<const char*, const char*>(first, (const char*)at + (std::max<int64_t>(m, 0) + std::max<int64_t>(n, 0) + 1) * elem_size(dtype));
  };
  const auto c = span(p.C, p.ldc, p.scn, p.out_dtype), d = span(p.aux, p.aux_sm, p.aux_sn, p.aux_dtype);
  return d.first < c.second && c.first < d.second;
}

// Which tile kernel a product runs on (not fp32's); `tile_arg` as in gemm_impl.
struct TileChoice { int tile = 1, tile_m = 0; bool w128_ok = false; };   // tile_m: 0, or 192 / 128 rows of a four-wave tile
TileChoice tile_choice(const GemmArgs& p, int in_dtype, bool b_kmajor, int tile_arg, int cus) {
  const int M = p.M, N = p.N;
  const bool is8 = elem_size(in_dtype) == 1;
  const long tiles256 = (long)((M + 255) / 256) * ((N + 255) / 256);
  TileChoice c;
  // large problems run the software-pipelined 8-wave kernel
  // (5 = the persistent form of the pipelined kernel; it falls back to 4 for edge tiles or a K tail)
  // persistent only when every program gets the same number of tiles: with a remainder the hardware's
  // dynamic dispatch of one workgroup per tile balances better (6144^3: 1011 vs 942 TFLOP/s)
  c.tile = (tiles256 * 2 >= cus) ? (tiles256 % cus == 0 ? 5 : 4) : 1;
  // 16-bit operands, from 256 rows and columns and at least half a round of tiles on: four waves of
  // 16x16x32 MFMAs (at 8192^3 bf16 +5 % over the persistent form with a row-major
  // B, +14 % with a K-major B; at 3072^3, 144 tiles, 790 vs 660 TFLOP/s for the 128x128 tiles)
  // (fp8, K-major B: 16x16x128 MFMAs, 8192^3 e4m3 2790-2810 vs 2570-2600 TFLOP/s)
  // (fp8 from three quarters of a round: at 144 tiles the eight-wave kernel is 4-7 % ahead - 3072^3 1520 vs
  // 1450, 3072x3072x8192 2040 vs 1890 TFLOP/s -, at 196 tiles the four-wave one by 2 %, at 225 by 13 %)
  // (partial tiles are whole ones moved back over their neighbours: an addend that is C itself must be read only once)
  const bool once = (M % 256 != 0 || N % 256 != 0) && addend_in_c(p);
  c.w128_ok = !once && (is8 ? gemm_wave128_f8_ok(p, b_kmajor) : gemm_wave128_ok(p, b_kmajor));
  if (tiles256 * (is8 ? 4 : 2) >= cus * (is8 ? 3 : 1) && c.w128_ok) c.tile = 6;
  c.tile = tile_arg >= 0 ? tile_arg : knob(knobs().tile, c.tile);
  // 16-bit products whose 256 x 256 tiles fill the last round of CUs badly (or whose M is a multiple of 192 only): the
  // same kernel on tiles of 192 x 256 where those use the CUs better (3072^3: 192 tiles instead of 144 for 256 CUs)
  if (!is8 && tile_arg < 0 && (knobs().tile == UNSET || knobs().tile_m == 192) && gemm_wave128_192_ok(p, b_kmajor, in_dtype)) {
    auto fill = [&](long t) { return t <= 0 ? 0.0 : (double)t / (double)(((t + cus - 1) / cus) * cus); };
    const long tiles192 = (long)((M + 191) / 192) * ((N + 255) / 256);
    const int want = knob(knobs().tile_m, 0);
    // (below half a round of 256-row tiles the 128-row tiles further down may fill better still: 3072 x 2048 x 4096 bf16,
    // 128 tiles of 192 rows 734 TFLOP/s, 192 tiles of 128 rows 815)
    const long tiles128 = (long)((M + 127) / 128) * ((N + 255) / 256);
    const bool rather128 = c.tile == 1 && tiles128 <= cus && fill(tiles128) > fill(tiles192) &&
                           gemm_wave128_192_ok(p, b_kmajor, in_dtype, 128);
    if (want == 192 || (want == 0 && !rather128 && tiles192 * 2 >= cus && (c.tile != 6 || fill(tiles192) > fill(tiles256) + 0.08))) {
      c.tile = 6;
      c.tile_m = 192;
    }
  }
  // fp8 likewise (K-major B, 16-bit C), from three quarters of a round of the 192-row tiles on.  Flushed do_bench, e4m3,
  // 256-row choice / 192-row tiles: 3072^3 (144 / 192 tiles) 1100 / 1565 TFLOP/s, 3072 x 3072 x 8192 1365 / 2145, 2304 x
  // 4096 x 4096 1220 / 1785, 4608 x 4096 x 4096 (288 / 384) 1600 / 2070, 6144^3 (576 / 768) 2510 / 2805, 1536 x 8192 x 8192
  // (192 / 256) 2100 / 2680; not taken where they fill worse: 3840 x 3840 x 4096 (225 / 300) 2270 / 1530, 5376 x 5120 x
  // 4096 (420 / 560) 2185 / 1995
  if (is8 && tile_arg < 0 && (knobs().tile == UNSET || knobs().tile_m == 192) && gemm_wave128_f8_192_ok(p, b_kmajor)) {
    auto fill = [&](long t) { return t <= 0 ? 0.0 : (double)t / (double)(((t + cus - 1) / cus) * cus); };
    const long tiles192 = (long)((M + 191) / 192) * ((N + 255) / 256);
    const int want = knob(knobs().tile_m, 0);
    if (want == 192 || (want == 0 && tiles192 * 4 >= cus * 3 && (c.tile != 6 || fill(tiles192) > fill(tiles256) + 0.08))) {
      c.tile = 6;
      c.tile_m = 192;
    }
  }
  // and on tiles of 128 x 256 where the 256 x 256 tiles are too few for their kernel (less than half a round) but these
  // fill more than half of one round (2560^3: 100 and 200 tiles; 716 -> 825 TFLOP/s against the 128 x 128 tiles; 2304 x
  // 2048 x 8192, 144 tiles: 650 -> 692; at half a round the 128 x 128 tiles stay ahead, 2048 x 2048 x 4096: 627 vs 569)
  if (!is8 && tile_arg < 0 && (knobs().tile == UNSET || knobs().tile_m == 128) && c.tile_m == 0 &&
      gemm_wave128_192_ok(p, b_kmajor, in_dtype, 128)) {
    const long tiles128 = (long)((M + 127) / 128) * ((N + 255) / 256);
    const int want = knob(knobs().tile_m, 0);
    if (want == 128 || (want == 0 && c.tile == 1 && tiles128 * 16 >= cus * 9 && tiles128 <= cus)) {
      c.tile = 6;
      c.tile_m = 128;
    }
  }
  // fp8 likewise, where the same part of a round is filled
  if (is8 && tile_arg < 0 && (knobs().tile == UNSET || knobs().tile_m == 128) && c.tile_m == 0 &&
      gemm_wave128_f8_192_ok(p, b_kmajor, 128)) {
    const long tiles128 = (long)((M + 127) / 128) * ((N + 255) / 256);
    const int want = knob(knobs().tile_m, 0);
    if (want == 128 || (want == 0 && c.tile == 1 && tiles128 * 16 >= cus * 9 && tiles128 <= cus)) {
      c.tile = 6;
      c.tile_m = 128;
    }
  }
  return c;
}

// 16-bit and fp8 products of more than one round of tiles whose last round is badly filled: the upper rows on 256-row
// tiles and the lower ones on 192-row tiles in ONE launch, split by mixed_split.  MI355_GEMM_MIXED_ROWS forces the rows
// of the 256-row part (0 = never).
int mixed_choice(const GemmArgs& p, const TileChoice& c, int in_dtype, bool b_kmajor, int cus) {
  const int M = p.M, N = p.N;
  const long tiles256 = (long)((M + 255) / 256) * ((N + 255) / 256);
  const bool is8 = elem_size(in_dtype) == 1;
  auto mixed_ok = [&](int rows256) {
    return is8 ? gemm_wave128_f8_mixed_ok(p, b_kmajor, rows256) : gemm_wave128_mixed_ok(p, b_kmajor, in_dtype, rows256);
  };
  if (knobs().tile == UNSET && knobs().tile_m == UNSET && N % 256 == 0) {
    const int want = knob(knobs().mixed_rows, -1);
    if (want > 0) {
      if (mixed_ok(want)) return want;
    } else if (want < 0 && c.tile == 6 && c.tile_m == 0 && tiles256 > cus && M % 256 == 0) {
      const int rows = mixed_split(M, N / 256, cus);
      if (rows > 0 && mixed_ok(rows)) return rows;
    }
  }
  return 0;
}

// Whether a product goes to a ring kernel (`ring`: its shape, else -1; in place of the other 128x128 kernel but for the short K
// of short_k) and whether it is worth two calls (`cut`, us 1e30: one).  The one place that decides: for the call, and for the room that
// the second part of a cut product is given (gemm_route).
struct PartChoice { int tile, ring; Cut cut; };
PartChoice part_choice(const GemmArgs& p, const TileChoice& c, int es, bool b_kmajor, bool by_knob, int mixed_rows, int cus) {
  const int M = p.M, N = p.N, steps = (p.k_bytes + 127) / 128, tile = c.tile;
  const bool is8 = es == 1;
  PartChoice r{tile, -1, {M, N, 1e30}};
  // (partial four-wave tiles pay for a prologue and edges over a short K: fp16 K-major 4224 x 1408 x 128 9.1 / 7.7 us, 6640 x 5448 x 144 40 / 37, e4m3 4240 x 4224 x
  // 152 25.8 / 22; row-major B 7256 x 4688 x 192 37 / 32; not where 256-row tiles fill more than half of their one round: fp16 1216 x 7488 x 128 11.4 / 12.6, K-major
  // 2464 x 5376 x 168 17.2 / 18.6, e4m3 4152 x 3212 x 320 15.6 / 18.7; nor with an activation: 3104 x 5456 x 152 23.2 / 28.8)
  const long tiles256 = (long)((M + 255) / 256) * ((N + 255) / 256);
  const bool partial = knobs().tile_m == UNSET && knobs().mixed_rows == UNSET && (M % (c.tile_m ? c.tile_m : 256) != 0 || N % 256 != 0) &&
                       p.activation == MI355_ACT_NONE && (tiles256 > cus || tiles256 * 2 <= cus) && p.k_bytes <= (tiles256 > cus || !b_kmajor ? 384 : 320);
  const bool pairs_ok = !by_knob && knobs().tile_m == UNSET && knobs().mixed_rows == UNSET && ring_ok(es, b_kmajor);
  if (!by_knob && (tile != 6 || partial) && !p.aux && p.c_vec_ok && short_k(M, N, p.k_bytes, b_kmajor, cus)) {   // (its addends and odd rows of C cost more)
    if (pairs_ok && (long)((M + 127) / 128) * ((N + 127) / 128) > cus && !one_barrier_ahead(M, N, p.k_bytes, is8, b_kmajor, cus)) r.ring = 4;
    else r.tile = 1;
  }
  else if (tile == 1 && by_knob) r.ring = 0;
  else if (tile >= 8 && tile <= 10) r.ring = tile - 8;
  else if (tile == 12 && b_kmajor) r.ring = 3;
  else if (tile == 13) r.ring = 4;
  else if (tile == 11) r.tile = 1;   // the one-barrier-per-step kernel on 128x128 tiles
  else if (tile == 1 || (!by_knob && knobs().tile_m == UNSET && knobs().mixed_rows == UNSET)) {
    const int rows = tile == 6 && c.tile_m ? c.tile_m : 256;
    const RingPlan plan = ring_plan(M, N, steps, cus, 1, 1, 1.0, thin_ok(M, N, p.k_bytes, b_kmajor, cus));
    const bool rounds = (tile == 6 || tile == 1) && plan.shape < 3;
    const double plan_us = rounds ? ring_rounds_us(M, N, steps, cus, plan.shape) : plan.us;
    double other = tile == 1 ? 1e30 : tiles256_us((long)((M + rows - 1) / rows) * ((N + 255) / 256), rows, steps, cus, tile != 6, is8);
    if (mixed_rows > 0) other *= 0.9;   // (two tile heights in one launch are chosen where they gain at least 5 %)
    if (plan_us < (tile == 6 ? 0.92 : 1.0) * other) r.ring = plan.shape;   // (pitches move the rings by up to 15 %: 1664 x 6912 x 2112 bf16, 702 tiles, 53 us for the estimate's 47)
    const Cut cut = best_cut(M, N, steps, cus, tile, r.ring, is8);
    if (cut.us < (tile == 1 ? 0.88 : 0.92) * std::min(plan_us, other)) r.cut = cut;
    // (an addend: fp16 3799 x 2304 x 512 23.2 / 23.7, row-major B 3840 x 6016 x 64, on the eight-wave kernel, 35.9 / 25.0; rows of C that are no whole groups of four:
    // K-major 1468 x 4405 x 128 13.2 / 10.7; both, 2176 x 4234 x 256 18.3 / 19.3; rows that do not begin on 16 bytes, K-major 3085 x 2804 x 704 21.5 / 23.8, 4204 x 2012 x 640 21.3 / 22.8)
    const double epilogue = (p.aux ? 2.2 : 0.0) + (p.c_vec_ok && p.ldc % 8 == 0 ? 0.0 : 2.0);
    const double added = p.aux && tile != 1 ? (tile == 6 ? 2.8 : 6.5) * (double)(((long)((M + rows - 1) / rows) * ((N + 255) / 256) + cus - 1) / cus) : 0.0;
    // What the two-stage rings are compared with is shorter than `other` says on 192 and 128 rows (0.91 .. 0.97 and 0.83 .. 0.95 of it, 60 products: K-major 2304 x 3648 x 384
    // 14.6 / 16.7), and for two steps on the eight-wave fp8 kernel with whole columns of tiles (1920 x 7680 x 64 10.5 / 12.9, 4608 x 3584 x 64 10.8 / 13.4); fp8 of more
    // than twenty steps is not worth the risk of either estimate (1344 x 6144 x 2944 33.8 / 39.7).  1472 drawn products that could run on either are 1.043 times as fast
    // as without these rings, seven of them more than 5 % slower and none 10 % (17 without these factors).
    const double shorter = tile == 6 ? (rows == 192 ? 0.95 : rows == 128 ? 0.9 : 1.0) : is8 && steps <= 2 && N % 256 == 0 ? 0.75 : 1.0;
    const double rings = plan_us + epilogue * (double)((M + 127) / 128) * ((N + 127) / 128) / cus;
    if (pairs_ok && !(is8 && steps > 20) && pairs_us(M, N, steps, cus, false, (p.lda | p.ldb) % 128 != 0, epilogue) < 0.97 * std::min({rings, shorter * other + added, r.cut.us})) {
      r.ring = 4;
      r.cut = {M, N, 1e30};
    }
  }
  return r;
}

bool aligned(const void* p, size_t a) { return ((uintptr_t)p % a) == 0; }

// 16-bit operands whose rows begin on dwords and are whole ones: what the ring and the four-wave kernels take where the rows are not whole
// 16-byte chunks.  (Eight elements at least: the chunk that a row ends inside is read as the row's last 16 bytes.  `behind`: where those reach
// in front of N columns of a row-major B there are others.)
struct DwordRows { bool a, bk, bn; };
DwordRows dword_rows(const void* A, const void* B, int M, int N, int K, int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int es, bool behind) {
  if (es != 2) return {false, false, false};
  const bool k = K % 2 == 0 && K >= 8;
  return {k && sak == 1 && sam % 2 == 0 && sam >= K && aligned(A, 4), k && sbk == 1 && sbn % 2 == 0 && sbn >= K && aligned(B, 4),
          sbn == 1 && ((sbk != 1 && sbk % 2 == 0 && N % 2 == 0 && (N >= 8 || behind) && sbk >= N && aligned(B, 4)) ||
                       (sbk % 8 == 0 && sbk >= (N + 7) / 8 * 8 && aligned(B, 16)))};
}

// us of the any-stride kernel: 64x64 tiles, about 1.3 us per 64 k (1024 x 1024 x 1000 bf16 23 us, x 4100 107; e4m3, row-major B 2.8: 3 x 1442 x 2161 98)
double any_stride_us(int M, int N, int K, int cus, double step64 = 1.3) {
  const long tiles = (long)((M + 63) / 64) * ((N + 63) / 64);
  return kLaunchUs + (double)((tiles + cus - 1) / cus) * (1.0 + step64 * ((K + 63) / 64));
}

// Whether a 16-bit product stays on that kernel whatever its operands' rows: K is a single step of it, and rows of C that are no whole groups
// of four or an addend make the tile kernels' epilogues slow (see gemm_route), or its rounds are shorter.
bool short_for_any_stride(int M, int N, int K, bool addend) { return K < 48 && (int64_t)M * N * K < 1 << 30 && (N % 4 != 0 || addend); }

bool any_stride_ahead(int M, int N, int K, bool addend, int cus) {
  if (short_for_any_stride(M, N, K, addend)) return true;
  const int steps = (K + 63) / 64;
  const double tiles = std::min(ring_plan(M, N, steps, cus, 1, 1).us, tiles256_us((long)((M + 255) / 256) * ((N + 255) / 256), 256, steps, cus, M < 256 || N < 256, false));
  return any_stride_us(M, N, K, cus) <= tiles;
}

bool copy_strides(const int64_t* src, int64_t* dst) {
  if (!src) return false;
  for (int i = 0; i < 4; i++) dst[i] = src[i];
  return true;
}

}  // namespace

extern "C" {

int mi355_query(int what) {
  if (what == MI355_Q_ABI_VERSION) return MI355_ABI_VERSION;   // (answered without touching the device)
  const DeviceInfo& d = device_info();
  switch (what) {
    case MI355_Q_ABI_VERSION: return MI355_ABI_VERSION;
    case MI355_Q_CU_COUNT: return d.cus;
    case MI355_Q_IS_GFX950: return d.gfx950;
    case MI355_Q_LDS_BYTES: return d.lds;
    case MI355_Q_CLOCK_KHZ: return d.clock_khz;
    case MI355_Q_WALL_CLOCK_KHZ: return d.wall_clock_khz;
    case MI355_Q_STREAMK_WORKSPACE_BYTES: return (d.cus > 0 ? d.cus : 256) * 2 * 256 * 256 * 4;
    default: return -1;
  }
}

void mi355_refresh_env(void) { load_knobs(); }

const char* mi355_strerror(int code) {
  switch (code) {
    case MI355_OK: return "ok";
    case MI355_EINVAL: return "invalid argument (null pointer, non-positive size or unknown enum)";
    case MI355_EDTYPE: return "unsupported dtype combination";
    case MI355_ESHAPE: return "shape not supported by this kernel family";
    case MI355_ESTRIDE: return "stride or alignment not supported by this kernel family";
    case MI355_EDEVICE: return "current device is not a gfx950 GPU";
    case MI355_ESCRATCH: return "the library's static scratch array is too small for this call (more than 256 programs)";
    default: break;
  }
  if (code > 0) return hipGetErrorString((hipError_t)code);
  return "unknown error";
}

static int splitk_impl(const void* A, const void* B, void* C, int M, int N, int K,
                       int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int64_t scm, int64_t scn,
                       int in_dtype, int out_dtype, const float* a_scale, const float* b_scale,
                       int activation, const void* aux, int64_t aux_sm, int64_t aux_sn, int aux_dtype,
                       int splits, void* workspace, size_t workspace_bytes, void* stream_, int k_rows, bool behind = false);

// `workspace`: stream-K's.  `spare`: room for the slices of a second part that is split along K (see best_cut), or none.  `behind`: eight columns of
// B at least lie in front of these (see dword_rows).
static int gemm_impl(const void* A, const void* B, void* C, int M, int N, int K,
                     int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int64_t scm, int64_t scn,
                     int in_dtype, int out_dtype, const float* a_scale, const float* b_scale,
                     int activation, const void* aux, int64_t aux_sm, int64_t aux_sn, int aux_dtype,
                     int tile_arg, int group_m_arg, void* stream_, float* workspace = nullptr, int k_rows = 0, void* spare = nullptr, size_t spare_bytes = 0, bool behind = false) {
  if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0) return MI355_EINVAL;
  if (aux && aux_dtype != MI355_F16 && aux_dtype != MI355_BF16 && aux_dtype != MI355_F32) return MI355_EDTYPE;
  if (activation != MI355_ACT_NONE && activation != MI355_ACT_LEAKY_RELU) return MI355_EINVAL;
  if (in_dtype < MI355_F16 || in_dtype > MI355_F32) return MI355_EDTYPE;
  if (out_dtype < MI355_F16 || out_dtype > MI355_F32) return MI355_EDTYPE;
  if (!device_info().gfx950) return MI355_EDEVICE;
  hipStream_t stream = (hipStream_t)stream_;
  const int es = elem_size(in_dtype);
  const bool is32 = in_dtype == MI355_F32;   // fp32 operands: fp32 MFMAs with a K-major B, the any-stride FMA kernel otherwise
  const bool is8 = es == 1;
  const int vec = 16 / es;  // elements per 16-byte chunk

  const bool out_ok = true;   // every output type of the ABI has a store in the MFMA epilogues (fp8: hardware conversion, saturating)
  const bool a_ok = sak == 1 && sam % vec == 0 && sam >= K && aligned(A, 16) && K % vec == 0;
  const bool b_kmajor16 = sbk == 1 && sbn % vec == 0 && sbn >= K && aligned(B, 16);
  // (a row-major B: rows of whole 16-byte chunks - N itself need not be one: the last chunk of a row then reaches into
  // the padding that the pitch provides, and the columns beyond N are never stored)
  const bool b_nmajor = !is32 && sbn == 1 && sbk % vec == 0 && sbk >= (N + vec - 1) / vec * vec && aligned(B, 16);
  // Rows of 16-bit elements that begin on dwords: the ring and the four-wave kernels' (`loose`), where no kernel of 16-byte chunks takes the operands
  const bool chunks = a_ok && (b_kmajor16 || b_nmajor);
  const DwordRows rows = dword_rows(A, B, M, N, K, sam, sak, sbk, sbn, es, behind);
  const bool loose = !chunks && rows.a && (rows.bk || rows.bn) && (k_rows > 0 || tile_arg >= 0 || knobs().tile != UNSET || !any_stride_ahead(M, N, K, aux != nullptr, device_info().cus > 0 ? device_info().cus : 256));
  const bool b_kmajor = loose ? rows.bk : b_kmajor16;
  // the tile copies address 256 rows of an operand with 32-bit byte offsets from a 64-bit tile base
  const bool pitch_ok = (int64_t)sam * es < (1 << 23) && (b_kmajor ? (int64_t)sbn * es < (1 << 23) : (int64_t)sbk * es < (1 << 26));
  const bool fast = pitch_ok && out_ok && (chunks || loose) && knob(knobs().force_strided, 0) == 0;

  if (!fast && k_rows > 0) K = k_rows;   // (the kernels of any stride have no use for A's padding, and B ends before it)
  if (!fast && is32) {
    GemmStridedArgs s{A, B, C, M, N, K, sam, sak, sbk, sbn, scm, scn, a_scale, b_scale, activation, in_dtype, out_dtype,
                      aux, aux_sm, aux_sn, aux_dtype};
    return gemm_strided_launch(s, stream);   // (the masked MFMA kernel converts to 16 bits on its way through LDS: not for fp32)
  }
  if (!fast) {
    GemmStridedArgs s{A, B, C, M, N, K, sam, sak, sbk, sbn, scm, scn, a_scale, b_scale, activation, in_dtype, out_dtype,
                      aux, aux_sm, aux_sn, aux_dtype};
    // (MI355_GEMM_FORCE_STRIDED=2: the fp32-FMA kernel, a second implementation kept for tests)
    return knob(knobs().force_strided, 0) == 2 ? gemm_strided_launch(s, stream) : gemm_masked_launch(s, stream);
  }

  GemmArgs p{};
  p.A = (const char*)A; p.B = (const char*)B; p.C = (char*)C;
  p.M = M; p.N = N; p.K = K; p.k_bytes = K * es;
  p.lda = sam * es;
  p.ldb = (b_kmajor ? sbn : sbk) * es;
  p.ldc = scm; p.scn = scn;
  p.a_scale = a_scale; p.b_scale = b_scale;
  p.activation = activation; p.out_dtype = out_dtype;
  p.group_m = group_m_arg > 0 ? group_m_arg : knob(knobs().group_m, 8);
  // four consecutive C elements as one store: rows of 16-bit / fp32 elements 16-byte aligned (for fp8 that
  // makes every group of four 4-byte aligned)
  p.c_vec_ok = scn == 1 && scm % 4 == 0 && aligned(C, 16);
  p.lean_ok = knob(knobs().lean_epilogue, 1);
  p.aux = aux; p.aux_sm = aux_sm; p.aux_sn = aux_sn; p.aux_dtype = aux_dtype;

  const int cus = device_info().cus > 0 ? device_info().cus : 256;
  // 256x256 tiles once they fill half of the CUs, 128x128 tiles (two workgroups per CU) below that
  // (bf16, 144 tiles: 912 vs 651 TFLOP/s; 100 tiles: 654 vs 715)
  const long tiles256 = (long)((M + 255) / 256) * ((N + 255) / 256);
  if (is32) {
    p.num_programs = std::min(knob(knobs().programs, cus), cus);
    // fp32 products are bound by the fp32 MFMA rate alone (1/16 of the bf16 rate on the same bytes), so what counts is
    // how evenly the tiles fill the CUs: 256x256 tiles (pipelined kernel: 8192^3 152 TFLOP/s, 4096^3 149; one barrier per
    // step 141 / 139) against 128x128 tiles, two workgroups per CU, at about 0.9 of that rate (137 / 135; 2048^3: 102
    // against 36 for its 64 large tiles)
    auto fill = [&](long t, long slots) { return (double)t / (double)(((t + slots - 1) / slots) * slots); };
    const long tiles128 = (long)((M + 127) / 128) * ((N + 127) / 128);
    const bool large = fill(tiles256, cus) >= 0.9 * fill(tiles128, 2 * cus);
    const int t32 = tile_arg >= 0 ? tile_arg : knob(knobs().tile, large ? (tiles256 % cus == 0 ? 5 : 4) : 1);
    return gemm32_launch(p, t32 == 6 || t32 == 7 ? 4 : t32, stream);   // (the four-wave 16x16 kernels and stream-K have no fp32 form)
  }
  const TileChoice choice = tile_choice(p, in_dtype, b_kmajor, tile_arg, cus);
  int tile = choice.tile;
  p.tile_m = choice.tile_m;
  const int mixed_rows = tile_arg < 0 ? mixed_choice(p, choice, in_dtype, b_kmajor, cus) : 0;
  p.num_programs = knob(knobs().programs, cus);  // persistent and stream-K forms (tile 5 / 7): one workgroup per CU
  if (p.num_programs > cus) p.num_programs = cus;       // (the stream-K workspace is sized for one program per CU)
  p.workspace = workspace;
  const bool skinny_allowed = tile_arg < 0 && knob(knobs().skinny, 1);  // an explicit tile means a tile kernel
  const bool can_ring = ring_ok(es, b_kmajor);
  const int ksteps128 = (p.k_bytes + 127) / 128;
  // at most 64 rows on one side: stream the other operand once (X = small side, Y = streamed side) where that is the faster
  // way, or where MI355_GEMM_SKINNY asks for it
  if (skinny_allowed && k_rows == 0 && !loose &&
      (knobs().skinny != UNSET || streams(M, N, p.k_bytes, es, b_kmajor, cus) || streams8(M, N, p.k_bytes, es, b_kmajor, cus))) {
    SkinnyArgs sk{};
    sk.K = K; sk.C = (char*)C; sk.a_scale = a_scale; sk.b_scale = b_scale;
    sk.activation = activation; sk.out_dtype = out_dtype;
    bool y_kmajor = true, x_kmajor = true;
    if (M <= 64) {
      sk.X = (const char*)A; sk.Y = (const char*)B; sk.S = M; sk.L = N;
      sk.x_pitch = p.lda; sk.y_pitch = p.ldb; sk.cs = scm; sk.cl = scn;
      sk.aux = aux; sk.aux_ss = aux_sm; sk.aux_sl = aux_sn; sk.aux_dtype = aux_dtype;
      y_kmajor = b_kmajor;
    } else {
      sk.X = (const char*)B; sk.Y = (const char*)A; sk.S = N; sk.L = M;
      sk.x_pitch = p.ldb; sk.y_pitch = p.lda; sk.cs = scn; sk.cl = scm;
      sk.aux = aux; sk.aux_ss = aux_sn; sk.aux_sl = aux_sm; sk.aux_dtype = aux_dtype;
      x_kmajor = b_kmajor;
    }
    if (gemm_skinny_ok(sk, y_kmajor, x_kmajor, es)) return gemm_skinny_launch(sk, in_dtype, y_kmajor, x_kmajor, stream);
    if (is8 && b_kmajor && !aux && gemm8_skinny_ok(p)) return gemm8_skinny_launch(p, in_dtype == MI355_F8E5M2, stream);
  }
  // the ring kernels of 64 .. 128-row tiles, and products in two calls
  int ring = -1;
  if (can_ring) {
    if (k_rows > 0) {   // a row-major B that ends before A's padding does: the ring kernels know
      ring = ring_plan(M, N, ksteps128, cus, 1, 1).shape;
      p.K = k_rows;
    } else {
      const PartChoice parts = part_choice(p, choice, es, b_kmajor, tile_arg >= 0 || knobs().tile != UNSET, mixed_rows, cus);
      tile = parts.tile;
      ring = parts.ring;
      if (!workspace && parts.cut.us < 1e30) {
        const int m = parts.cut.m, n = parts.cut.n;
        const int64_t dm = m < M ? m : 0, dn = m < M ? 0 : n;
        const int rc = gemm_impl(A, B, C, m, n, K, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale, activation,
                                 aux, aux_sm, aux_sn, aux_dtype, -1, group_m_arg, stream_);
        if (rc) return rc;
        const int m2 = M - (int)dm, n2 = N - (int)dn;
        A = (const char*)A + dm * sam * es; B = (const char*)B + dn * sbn * es; C = (char*)C + (dm * scm + dn * scn) * elem_size(out_dtype);
        if (aux) aux = (const char*)aux + (dm * aux_sm + dn * aux_sn) * elem_size(aux_dtype);
        const int splits = spare_bytes > 0 ? auto_splits(m2, n2, p.k_bytes, in_dtype, b_kmajor, true, cus) : 1;
        if (splits > 1 && (size_t)splits * m2 * n2 * 4 <= spare_bytes)
          return splitk_impl(A, B, C, m2, n2, K, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale, activation,
                             aux, aux_sm, aux_sn, aux_dtype, splits, spare, spare_bytes, stream_, 0, dn >= 8);
        return gemm_impl(A, B, C, m2, n2, K, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale, activation,
                         aux, aux_sm, aux_sn, aux_dtype, -1, group_m_arg, stream_, nullptr, 0, nullptr, 0, dn >= 8);
      }
    }
    if (loose && ring < 0 && mixed_rows == 0 && !(tile == 6 && (p.tile_m != 0 || choice.w128_ok))) ring = ring_plan(M, N, ksteps128, cus, 1, 1).shape;
  }
  if (ring >= 0)
    return is8 ? gemm_ring8_launch(p, in_dtype == MI355_F8E5M2, ring, 1, 0, stream)
               : gemm_ring16_launch(p, in_dtype == MI355_BF16, b_kmajor, ring, 1, 0, stream);
  if (is8 && mixed_rows > 0) return gemm_wave128_f8_mixed_launch(p, mixed_rows, in_dtype == MI355_F8E5M2, stream);
  if (is8 && tile == 6 && (p.tile_m == 192 || p.tile_m == 128 || choice.w128_ok)) return gemm_wave128_f8_launch(p, in_dtype == MI355_F8E5M2, b_kmajor, stream);
  if (is8) return gemm8_launch(p, in_dtype == MI355_F8E5M2, b_kmajor, tile, stream);
  // 6: four waves, 128x128 of C per wave from 16x16x32 MFMAs
  // (a tile height of 192 / 128 rows was set above only after gemm_wave128_192_ok had accepted the shape for it)
  if (mixed_rows > 0 && !is8) return gemm_wave128_mixed_launch(p, mixed_rows, in_dtype == MI355_BF16, b_kmajor, stream);
  if (tile == 6 && (p.tile_m == 192 || p.tile_m == 128 || choice.w128_ok)) return gemm_wave128_launch(p, in_dtype == MI355_BF16, b_kmajor, stream);
  return gemm16_launch(p, in_dtype == MI355_BF16, b_kmajor, tile, stream);
}

int mi355_gemm(const void* A, const void* B, void* C, int M, int N, int K,
               int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int64_t scm, int64_t scn,
               int in_dtype, int out_dtype, const float* a_scale, const float* b_scale,
               int activation, void* stream_) {
  return gemm_impl(A, B, C, M, N, K, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale,
                   activation, nullptr, 0, 0, 0, -1, 0, stream_);
}

int mi355_gemm_tuned(const void* A, const void* B, void* C, int M, int N, int K,
                     int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int64_t scm, int64_t scn,
                     int in_dtype, int out_dtype, const float* a_scale, const float* b_scale,
                     int activation, int tile, int group_m, void* stream_) {
  if (tile < -1 || tile > 6 || group_m < 0) return MI355_EINVAL;
  return gemm_impl(A, B, C, M, N, K, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale,
                   activation, nullptr, 0, 0, 0, tile, group_m, stream_);
}

static int splitk_impl(const void* A, const void* B, void* C, int M, int N, int K,
                       int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int64_t scm, int64_t scn,
                       int in_dtype, int out_dtype, const float* a_scale, const float* b_scale,
                       int activation, const void* aux, int64_t aux_sm, int64_t aux_sn, int aux_dtype,
                       int splits, void* workspace, size_t workspace_bytes, void* stream_, int k_rows, bool behind) {
  if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0 || splits < 0) return MI355_EINVAL;
  if (activation != MI355_ACT_NONE && activation != MI355_ACT_LEAKY_RELU) return MI355_EINVAL;
  if (in_dtype < MI355_F16 || in_dtype > MI355_F32) return MI355_EDTYPE;
  if (out_dtype < MI355_F16 || out_dtype > MI355_F32) return MI355_EDTYPE;
  if (!device_info().gfx950) return MI355_EDEVICE;
  const int es = elem_size(in_dtype), vec = 16 / es;
  // what the tile kernels ask of the operands (as in mi355_gemm); anything else, or nothing to split: the plain call
  const bool a_ok = sak == 1 && sam % vec == 0 && sam >= K && aligned(A, 16) && K % vec == 0;
  const bool b_kmajor16 = sbk == 1 && sbn % vec == 0 && sbn >= K && aligned(B, 16);
  const bool is32 = in_dtype == MI355_F32;   // (fp32 operands: the fp32 MFMAs, K-major B only)
  const bool b_nmajor = !is32 && sbn == 1 && sbk % vec == 0 && sbk >= (N + vec - 1) / vec * vec && aligned(B, 16);
  const bool chunks = a_ok && (b_kmajor16 || b_nmajor);
  const DwordRows rows = dword_rows(A, B, M, N, K, sam, sak, sbk, sbn, es, behind);
  const bool loose = !chunks && rows.a && (rows.bk || rows.bn);
  const bool b_kmajor = loose ? rows.bk : b_kmajor16;
  const bool pitch_ok = (int64_t)sam * es < (1 << 23) && (b_kmajor ? (int64_t)sbn * es < (1 << 23) : (int64_t)sbk * es < (1 << 26));
  const int64_t k_bytes = (int64_t)K * es;
  const bool ring = ring_ok(es, b_kmajor);
  const int step_bytes = ring ? 128 : 64, ksteps = (int)((k_bytes + step_bytes - 1) / step_bytes);
  const int cus = device_info().cus > 0 ? device_info().cus : 256;
  if (splits == 0) splits = auto_splits(M, N, k_bytes, in_dtype, b_kmajor, ring, cus);
  const int per = splits >= 2 ? (ksteps + splits - 1) / splits : ksteps;
  const int used = (ksteps + per - 1) / per;   // (no split is left empty)
  // (dword rows need no room for slices to be taken: a call without it is the plain one)
  const bool room = workspace && aligned(workspace, 16) && used >= 2 && workspace_bytes >= (size_t)used * M * N * sizeof(float);
  if (!(pitch_ok && (chunks || (loose && room))) || used < 2 || knob(knobs().force_strided, 0) != 0)
    return gemm_impl(A, B, C, M, N, K, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale, activation,
                     aux, aux_sm, aux_sn, aux_dtype, -1, 0, stream_, nullptr, k_rows, nullptr, 0, behind);
  if (!room) return MI355_EINVAL;
  hipStream_t stream = (hipStream_t)stream_;
  GemmArgs p{};
  p.A = (const char*)A; p.B = (const char*)B; p.C = (char*)C;
  p.M = M; p.N = N; p.K = k_rows > 0 ? k_rows : K; p.k_bytes = (int)k_bytes;
  p.lda = sam * es;
  p.ldb = (b_kmajor ? sbn : sbk) * es;
  p.group_m = knob(knobs().group_m, 8);
  p.workspace = (float*)workspace;
  const int shape = ring ? ring_plan(M, N, ksteps, cus, used, used, 1.0, thin_ok(M, N, k_bytes, b_kmajor, cus)).shape : 0;
  const int rc = is32    ? gemm32_splitk_launch(p, used, per * 64, stream)
                 : ring && es == 1 ? gemm_ring8_launch(p, in_dtype == MI355_F8E5M2, shape, used, per * 128, stream)
                 : ring    ? gemm_ring16_launch(p, in_dtype == MI355_BF16, b_kmajor, shape, used, per * 128, stream)
                           : gemm8_splitk_launch(p, in_dtype == MI355_F8E5M2, used, per * 64, stream);
  if (rc != 0) return rc;
  GemmStridedArgs out{};
  out.C = C; out.M = M; out.N = N; out.scm = scm; out.scn = scn;
  out.a_scale = a_scale; out.b_scale = b_scale; out.activation = activation; out.out_dtype = out_dtype;
  out.aux = aux; out.aux_sm = aux_sm; out.aux_sn = aux_sn; out.aux_dtype = aux_dtype;
  return splitk_reduce_launch(out, (const float*)workspace, used, stream);
}

int mi355_gemm_splitk(const void* A, const void* B, void* C, int M, int N, int K,
                      int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int64_t scm, int64_t scn,
                      int in_dtype, int out_dtype, const float* a_scale, const float* b_scale,
                      int activation, int splits, void* workspace, size_t workspace_bytes, void* stream_) {
  return splitk_impl(A, B, C, M, N, K, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale, activation,
                     nullptr, 0, 0, 0, splits, workspace, workspace_bytes, stream_, 0);
}

// a row that fits one tile: product, addend, activation and softmax in ONE launch, on the fp32 accumulator,
// one rounding at the store - what the reference's single tile does
// (that kernel is one workgroup per 128 rows with operands of any strides, built for the small products of the
// reference's test, where the single rounding is the point: on time the tiled GEMM plus a softmax launch wins at every
// size - flushed caches, bf16: 32^3 10.8 against 9.3 us, 128 x 256 x 128 50 / 13, 1024 x 256 x 256 59 / 14, 8192 x 256 x 256
// 59 / 19, 256 x 256 x 2048 237 / 33 - and takes over beyond 2^18 elements of A by default, MI355_ROWFUSED_MAX_MK)
static bool rowfused(int M, int N, int K, int in_dtype) {
  return N <= 256 && (in_dtype == MI355_F16 || in_dtype == MI355_BF16) && (int64_t)M * K <= (int64_t)knob(knobs().rowfused_max_mk, 1 << 18);
}

// ---- mi355_gemm_ws: how a product with a workspace runs.  Operands whose rows the MFMA kernels cannot load (rows that are not
// whole 16-byte chunks nor, in 16 bits, whole dwords) or only at more than the copies' cost are first copied into rows of a padded pitch, both in one launch, zeros behind K; few tiles with a
// long K are split.  The any-stride kernel stays where the copies would cost more than they gain.
namespace {

struct GemmRoute {
  bool pack_a = false, pack_b = false;
  bool kmajor = false;
  int k = 0;                     // K as the kernels see it
  int k_rows = 0;                // > 0: rows of a row-major B that is not copied while A's K was padded beyond them
  int b_rows = 0;                // rows of the copy of B
  int64_t a_pitch = 0, b_pitch = 0;   // bytes
  int splits = 1;
  size_t a_bytes = 0, b_bytes = 0, slice_bytes = 0;   // (slices of the whole product, or of a second part of it)
};

size_t up(size_t v, size_t to) { return (v + to - 1) / to * to; }

GemmRoute gemm_route(const void* A, const void* B, int M, int N, int K, int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int in_dtype, bool addend) {
  GemmRoute r;
  r.k = K;
  const int es = elem_size(in_dtype), vec = 16 / es, cus = device_info().cus > 0 ? device_info().cus : 256;
  if (knob(knobs().force_strided, 0) != 0) return r;
  auto split = [&](bool kmajor) {
    if (knob(knobs().splitk, 1) == 0) return;
    const int64_t k_bytes = (int64_t)r.k * es;
    r.splits = auto_splits(M, N, k_bytes, in_dtype, kmajor, ring_ok(es, kmajor), cus);
    r.slice_bytes = r.splits > 1 ? (size_t)r.splits * M * N * 4 : 0;
    if (ring_ok(es, kmajor) && thin_ok(M, N, k_bytes, kmajor, cus)) {   // (the bytes stay at least those of a split on other tiles)
      const int others = auto_splits(M, N, k_bytes, in_dtype, kmajor, true, cus, false);
      if (others > 1) r.slice_bytes = std::max(r.slice_bytes, (size_t)others * M * N * 4);
    }
    if (r.splits > 1 || r.k_rows > 0 || !ring_ok(es, kmajor) || k_bytes < 2048 || (long)((M + 127) / 128) * ((N + 127) / 128) <= cus) return;
    // Room for the slices of what a cut leaves to a second call, by gemm_impl's own rule for a dense C of a 16-bit type without an addend
    // (what this function is told).  For another C the rule may differ: then the room is not used, or that part is not split.
    GemmArgs p{};
    p.A = (const char*)A; p.B = (const char*)B;
    p.M = M; p.N = N; p.K = r.k; p.k_bytes = (int)k_bytes;
    p.lda = r.pack_a ? r.a_pitch : sam * es;
    p.ldb = r.pack_b ? r.b_pitch : (kmajor ? sbn : sbk) * es;
    p.ldc = N; p.scn = 1; p.out_dtype = in_dtype == MI355_BF16 ? MI355_BF16 : MI355_F16;
    p.c_vec_ok = N % 4 == 0; p.lean_ok = knob(knobs().lean_epilogue, 1);
    const TileChoice c = tile_choice(p, in_dtype, kmajor, -1, cus);
    PartChoice parts = part_choice(p, c, es, kmajor, knobs().tile != UNSET, 0, cus);
    if (parts.cut.us < 1e30)   // (two tile heights only make one call shorter: looked at where a cut is left without them)
      if (const int rows = mixed_choice(p, c, in_dtype, kmajor, cus)) parts = part_choice(p, c, es, kmajor, knobs().tile != UNSET, rows, cus);
    const Cut cut = parts.cut;
    if (cut.us >= 1e30) return;
    const int m2 = cut.m < M ? M - cut.m : M, n2 = cut.m < M ? N : N - cut.n, splits = auto_splits(m2, n2, k_bytes, in_dtype, kmajor, true, cus);
    const size_t bytes = splits > 1 ? (size_t)splits * m2 * n2 * 4 : 0;
    if (bytes <= (16u << 20)) r.slice_bytes = bytes;
  };
  // (as in gemm_impl)
  const bool a_ok = sak == 1 && sam % vec == 0 && sam >= K && aligned(A, 16) && K % vec == 0;
  const bool bk_ok = sbk == 1 && sbn % vec == 0 && sbn >= K && aligned(B, 16) && K % vec == 0;
  const bool bn_ok = es != 4 && sbn == 1 && sbk % vec == 0 && sbk >= (N + vec - 1) / vec * vec && aligned(B, 16);
  if (a_ok && (bk_ok || bn_ok)) {
    split(bk_ok);
    return r;
  }
  if (es == 4 || sak != 1 || sam < K || (sbk == 1) == (sbn == 1)) return r;
  r.kmajor = sbk == 1;
  if (r.kmajor ? sbn < K : sbk < N) return r;
  // K is a single step of the any-stride kernel, and rows of C that are no whole groups of four or an addend make the tile kernels'
  // epilogues slow: the copies do not pay (us, that kernel / padded copies: 4024 x 5214 x 16 e4m3 49 / 78, 5246 x 2775 x 30 fp16 31 / 53, 520 x
  // 3873 x 32 8.7 / 11.6, 5164 x 2532 x 24 26 / 22 but 35 / 45 with an addend; whole groups of four: 5248 x 1792 x 28 e4m3 27 / 15)
  if (short_for_any_stride(M, N, K, addend)) return r;
  // (what stays in place has rows within the kernels' lane offsets, as in gemm_impl: only their kernels know k_rows)
  const int64_t a_most = 1 << 23, b_most = r.kmajor ? 1 << 23 : 1 << 26;
  // (16-bit rows of whole dwords stay too, `loose`, but for what the rows between 128-byte lines cost the kernels where that is more than the copies do)
  const DwordRows rows = dword_rows(A, B, M, N, K, sam, sak, sbk, sbn, es, false);
  // (next to a row-major B of whole chunks A alone is copied, with K rounded up, which B's rows need not be)
  const bool round_a = !r.kmajor && bn_ok && K % vec != 0;
  const bool a_line = (a_ok || (rows.a && !round_a)) && sam * es < a_most, b_line = r.kmajor ? (bk_ok || rows.bk) && sbn * es < b_most : (bn_ok || rows.bn) && sbk * es < b_most;
  // us: the copies at about 4.5 TB/s of reads and writes, then the best kernel
  auto copy_us = [&](bool a, bool b) { return 2.0 + 2.0 * es * ((a ? (double)M * K : 0.0) + (b ? (double)N * K : 0.0)) / 4.5e6; };
  const int steps = (int)(((int64_t)K * es + 127) / 128);
  const double ring = ring_ok(es, r.kmajor) ? ring_plan(M, N, steps, cus, 1, 1).us : 1e30;
  const long tiles256 = (long)((M + 255) / 256) * ((N + 255) / 256);
  // (fp8 next to a row-major B, which no ring kernel takes: the 128x128 kernel of one barrier per 64-byte step, and what its copies take
  // beyond the 2 us below.  104 x 2496 x 776 e4m3 any-stride kernel / copies 39 / 14 us, 240 x 100 x 648 e5m2 18.5 / 13, 272 x 550 x 226 11.3 / 11;
  // with less K the any-stride kernel stays: e5m2 198 x 707 x 154 9.1 / 11.4, 732 x 3038 x 54 9.3 / 14.5, e4m3 2303 x 674 x 49 10.2 / 13.2)
  const long rounds128 = ((long)((M + 127) / 128) * ((N + 127) / 128) + cus - 1) / cus;
  const bool one_barrier = !ring_ok(es, r.kmajor) && K >= (in_dtype == MI355_F8E4M3 ? 65 : 256);
  const double other = one_barrier ? 5.3 + 0.34 * (double)rounds128 * ((K + 63) / 64) : ring;
  const double any = std::min(other, tiles256_us(tiles256, 256, steps, cus, M < 256 || N < 256, es == 1));
  // What rows that do not begin on 128-byte lines add to a kernel's time, a line being fetched in two pieces, against the copies.  In the probe of both, bf16, us, pitch
  // a multiple of 128 bytes / 4 bytes more: 256x256 tiles, row-major B 4096^3 103 / 109, 8192^3 747 / 790, K-major 101 / 112, 721 / 830; ring tiles 1024^3 8.1 / 8.3, 2048^3
  // 18.6 / 24.4, 1024 x 4096 x 4096 32 / 39.  Ring tiles: 0.4 of a step for each operand, below 24 steps 0.24 (copied / in place: 684 x 1113 x 1554 15.4 / 8.3, 2732 x 426 x 972
  // 15.3 / 9.7, 771 x 2608 x 1460 21 / 13.8, 1349 x 5067 x 276 26 / 21; a long K is copied, 1282 x 604 x 6798 31.2 / 34.3).  256-row tiles: 0.08 of their time, K-major
  // 0.11 (5506 x 7021 x 2926 219 / 242, 2472 x 4042 x 1030 40.1 / 36.3); a K that is not whole pairs of steps runs on no others (1581 x 7168 x 5428 146 / 169), nor as one stream
  // over several rounds, and with 24 steps and more and both operands so a round that they leave unfilled costs up to half of that again (2154 x 5428 x 6548, 198
  // tiles, 175 / 215, 7454 x 2496 x 4234, 300, 199 / 240; row-major B 4390 x 1838 x 1838, 144, 59 / 73).  2387 drawn products of such rows are 1.30 times as fast as all
  // copied, eight of them more than 5 % slower and none 10 % (without that term 18, ten of them by up to 23 %).
  const bool loose_a = a_line && !a_ok, loose_b = b_line && !(r.kmajor ? bk_ok : bn_ok);
  bool loose = false;
  if (loose_a || loose_b) {
    const bool launch = !a_line || !b_line;   // (a copy is needed in any case)
    const double copies = (launch ? 0.0 : 5.0) + 2.0 * es * ((loose_a ? (double)M * K : 0.0) + (loose_b ? (double)N * K : 0.0)) / 6.2e6;
    double lines;
    if (any == ring) {
      const int s = auto_splits(M, N, (int64_t)K * es, in_dtype, r.kmajor, true, cus), shape = ring_plan(M, N, steps, cus, s, s).shape;
      const int bm = shape == 2 ? 64 : 128, bn = shape == 0 ? 128 : 64;
      const double rounds = std::max(1.0, (double)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * s / cus);
      lines = (loose_a + loose_b) * (steps < 24 && !launch ? 0.24 : 0.4) * (shape == 0 ? 0.42 : shape == 1 ? 0.265 : 0.165) * ((steps + s - 1) / s) * rounds;
    } else {
      const double here = M >= 256 && N >= 256 ? std::min(any, best_cut(M, N, steps, cus, 6, -1, false).us) : any;
      double other_rows = here;
      if (K * es % 256 != 0)
        for (int h : {192, 128}) other_rows = std::min(other_rows, tiles256_us((long)((M + h - 1) / h) * ((N + 255) / 256), h, steps, cus, false, false));
      auto blocks = [](int n) { return n > 256 && n % 256 <= 64 ? n / 256 : (n + 255) / 256; };   // (up to 64 rows or columns more are a call of their own: best_cut)
      const long tiles = (long)blocks(M) * blocks(N);
      const double filled = (double)tiles / (double)((tiles + cus - 1) / cus * cus);
      const double idle = steps >= 24 && K * es % 256 != 0 && loose_a && loose_b ? (r.kmajor ? 0.5 : 0.3) * std::max(0.0, 0.9 - filled) * any : 0.0;
      lines = (loose_a + loose_b) * ((r.kmajor ? 0.11 : 0.08) * here + idle) + here - other_rows;
    }
    loose = lines <= copies;
  }
  const bool a_stays = a_line && (loose || !loose_a), b_stays = b_line && (loose || !loose_b);
  r.pack_a = !a_stays;
  // a row-major B with good rows only lacks the zero rows beyond K, which the ring kernels do not read
  const bool even = es == 2 && K % 2 == 0 && K >= 8 && !round_a;   // (K as it is will do for dword rows, next to copies too)
  const bool short_b = !r.kmajor && K % vec != 0 && !even;
  r.pack_b = !b_stays || (short_b && ring + copy_us(!a_stays, false) > any + copy_us(!a_stays, true));
  const double packed = (r.pack_a || r.pack_b ? copy_us(r.pack_a, r.pack_b) : 0.0) + (r.pack_b || !short_b ? any : ring);
  const double masked = any_stride_us(M, N, K, cus, in_dtype == MI355_F8E4M3 && !r.kmajor && K > 64 ? 2.8 : 1.3);
  if (masked <= packed) {
    r.pack_a = r.pack_b = false;
    return r;
  }
  if (K % vec != 0 && !(even && !(r.pack_a && r.pack_b))) {
    // (whole pairs of 128-byte K steps where there are several rounds of 256 x 256 tiles, whose kernel then walks them as one stream)
    const int to = tiles256 > cus && (int64_t)K * es >= 1024 ? 256 : 128;
    r.k = (int)up(K, r.pack_b || r.kmajor ? to / es : vec);
    if (!r.kmajor && !r.pack_b) r.k_rows = K;
  }
  if (r.pack_a) {
    r.a_pitch = (int64_t)up((size_t)r.k * es, 128);
    r.a_bytes = up((size_t)r.a_pitch * M, 256);
  }
  if (r.pack_b) {
    r.b_rows = r.kmajor ? N : r.k;
    r.b_pitch = (int64_t)(r.kmajor ? up((size_t)r.k * es, 128) : up((size_t)N * es, 512));
    r.b_bytes = up((size_t)r.b_pitch * r.b_rows, 256);
  }
  if (r.a_pitch >= a_most || r.b_pitch >= b_most) {   // (beyond the kernels' lane offsets)
    GemmRoute plain;
    plain.k = K;
    return plain;
  }
  split(r.kmajor);
  return r;
}

}  // namespace

int64_t mi355_gemm_workspace(const void* A, const void* B, int M, int N, int K,
                             int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int in_dtype) {
  if (M <= 0 || N <= 0 || K <= 0 || in_dtype < MI355_F16 || in_dtype > MI355_F32) return 0;
  const GemmRoute r = gemm_route(A, B, M, N, K, sam, sak, sbk, sbn, in_dtype, false);
  return (int64_t)(r.a_bytes + r.b_bytes + r.slice_bytes);
}

int mi355_gemm_ws(const void* A, const void* B, void* C, int M, int N, int K,
                  int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int64_t scm, int64_t scn,
                  int in_dtype, int out_dtype, const float* a_scale, const float* b_scale,
                  const void* addend, int64_t sdm, int64_t sdn, int addend_dtype,
                  int activation, int softmax, void* workspace, size_t workspace_bytes, void* stream_) {
  if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0) return MI355_EINVAL;
  if (in_dtype < MI355_F16 || in_dtype > MI355_F32) return MI355_EDTYPE;
  if (!device_info().gfx950) return MI355_EDEVICE;
  if (softmax != 0 && softmax != 1) return MI355_EINVAL;
  if (softmax && out_dtype != MI355_F16 && out_dtype != MI355_BF16 && out_dtype != MI355_F32) return MI355_EDTYPE;
  if (workspace_bytes == 0 || (softmax && rowfused(M, N, K, in_dtype)))
    return mi355_gemm_epilogue(A, B, C, M, N, K, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale,
                               addend, sdm, sdn, addend_dtype, activation, softmax, stream_);
  if (addend && addend_dtype != MI355_F16 && addend_dtype != MI355_BF16 && addend_dtype != MI355_F32) return MI355_EDTYPE;
  const GemmRoute r = gemm_route(A, B, M, N, K, sam, sak, sbk, sbn, in_dtype, addend != nullptr);   // (with an addend no more than without)
  if (!workspace || !aligned(workspace, 256) || workspace_bytes < r.a_bytes + r.b_bytes + r.slice_bytes) return MI355_EINVAL;
  const int es = elem_size(in_dtype);
  char* ws = (char*)workspace;
  RepackRows op[2];
  int ops = 0;
  if (r.pack_a) {
    op[ops++] = {(const char*)A, ws, M, M, K * es, (int)up((size_t)r.k * es, 16), sam * es, r.a_pitch};
    A = ws; sam = r.a_pitch / es;
  }
  if (r.pack_b) {
    char* to = ws + r.a_bytes;
    if (r.kmajor) op[ops++] = {(const char*)B, to, N, N, K * es, (int)up((size_t)r.k * es, 16), sbn * es, r.b_pitch};
    else op[ops++] = {(const char*)B, to, K, r.b_rows, N * es, (int)up((size_t)N * es, 16), sbk * es, r.b_pitch};
    B = to; (r.kmajor ? sbn : sbk) = r.b_pitch / es;
  }
  if (ops > 0) {
    const int rc = repack_launch(op, ops, (hipStream_t)stream_);
    if (rc) return rc;
  }
  int rc;
  if (r.splits > 1)
    rc = splitk_impl(A, B, C, M, N, r.k, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale, activation,
                       addend, sdm, sdn, addend_dtype, r.splits, ws + r.a_bytes + r.b_bytes, r.slice_bytes, stream_, r.k_rows);
  else
    rc = gemm_impl(A, B, C, M, N, r.k, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale, activation,
                   addend, sdm, sdn, addend_dtype, -1, 0, stream_, nullptr, r.k_rows, ws + r.a_bytes + r.b_bytes, r.slice_bytes);
  if (rc || !softmax) return rc;
  return softmax_rows_launch(C, M, N, scm, scn, out_dtype, (hipStream_t)stream_);
}

int mi355_gemm_streamk(const void* A, const void* B, void* C, int M, int N, int K,
                       int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int64_t scm, int64_t scn,
                       int in_dtype, int out_dtype, const float* a_scale, const float* b_scale,
                       int activation, void* workspace, size_t workspace_bytes, void* stream_) {
  if (!workspace || !aligned(workspace, 16)) return MI355_EINVAL;
  if (workspace_bytes < (size_t)mi355_query(MI355_Q_STREAMK_WORKSPACE_BYTES)) return MI355_EINVAL;
  // partial 256x256 tiles, or fewer than 64 rows on a side (the streaming kernels): the plain call
  const bool whole_tiles = M > 0 && N > 0 && M % 256 == 0 && N % 256 == 0;
  return gemm_impl(A, B, C, M, N, K, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale,
                   activation, nullptr, 0, 0, 0, whole_tiles ? 7 : -1, 0, stream_, (float*)workspace);
}

// ---- stream-K without an allocation anywhere: the partial-tile workspace is a static device array.
// Host code must never use the array's NAME as an address (there it is a host-side stand-in; a kernel
// handed it would fault): the address on each device comes from hipGetSymbolAddress, once per device,
// and only that pointer is passed on.
constexpr int kStaticStreamKPrograms = 256;                                   // one program per CU of an MI355X
constexpr size_t kStaticStreamKBytes = (size_t)kStaticStreamKPrograms * 2 * 256 * 256 * 4;   // 128 MiB
static __device__ __align__(256) unsigned char scratch[kStaticStreamKBytes];

namespace {
constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices];          // per device: each GPU holds its own copy of the array
std::mutex g_scratch_mutex;

int static_scratch(void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return MI355_EDEVICE;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));   // with device `dev` current: that device's copy
    if (e != hipSuccess) return (int)e;
    if (!ptr) return MI355_EDEVICE;
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return MI355_OK;
}
}  // namespace

int mi355_gemm_streamk_static(const void* A, const void* B, void* C, int M, int N, int K,
                              int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int64_t scm, int64_t scn,
                              int in_dtype, int out_dtype, const float* a_scale, const float* b_scale,
                              int activation, void* stream_) {
  if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0) return MI355_EINVAL;
  // the static array holds two partial tiles for each of at most 256 programs (one per CU)
  const int cus = device_info().cus > 0 ? device_info().cus : 256;
  const int programs = knob(knobs().programs, cus) < cus ? knob(knobs().programs, cus) : cus;
  if (programs > kStaticStreamKPrograms) return MI355_ESCRATCH;
  void* ws = nullptr;
  const int rc = static_scratch(&ws);
  if (rc) return rc;
  const bool whole_tiles = M > 0 && N > 0 && M % 256 == 0 && N % 256 == 0;
  return gemm_impl(A, B, C, M, N, K, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale,
                   activation, nullptr, 0, 0, 0, whole_tiles ? 7 : -1, 0, stream_, (float*)ws);
}

int mi355_gemm_epilogue(const void* A, const void* B, void* C, int M, int N, int K,
                        int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int64_t scm, int64_t scn,
                        int in_dtype, int out_dtype, const float* a_scale, const float* b_scale,
                        const void* addend, int64_t stride_dm, int64_t stride_dn, int addend_dtype,
                        int activation, int softmax, void* stream_) {
  if (softmax != 0 && softmax != 1) return MI355_EINVAL;
  if (softmax && out_dtype != MI355_F16 && out_dtype != MI355_BF16 && out_dtype != MI355_F32) return MI355_EDTYPE;
  if (softmax && rowfused(M, N, K, in_dtype)) {
    if (!A || !B || !C || M <= 0 || N <= 0 || K <= 0) return MI355_EINVAL;
    if (addend && addend_dtype != MI355_F16 && addend_dtype != MI355_BF16 && addend_dtype != MI355_F32) return MI355_EDTYPE;
    if (activation != MI355_ACT_NONE && activation != MI355_ACT_LEAKY_RELU) return MI355_EINVAL;
    if (!device_info().gfx950) return MI355_EDEVICE;
    RowFusedArgs r{A, B, C, nullptr, M, N, K, 0, sam, sak, sbk, sbn, 0, 0, scm, scn, a_scale, b_scale,
                   activation, 1, out_dtype, addend, stride_dm, stride_dn, addend_dtype};
    return gemm_rowfused_launch(r, in_dtype == MI355_BF16, (hipStream_t)stream_);
  }
  int rc = gemm_impl(A, B, C, M, N, K, sam, sak, sbk, sbn, scm, scn, in_dtype, out_dtype, a_scale, b_scale,
                     activation, addend, stride_dm, stride_dn, addend_dtype, -1, 0, stream_);
  if (rc || !softmax) return rc;
  return softmax_rows_launch(C, M, N, scm, scn, out_dtype, (hipStream_t)stream_);
}

int mi355_gemm_chain(const void* A, const void* B, const void* W, void* C, int M, int N, int K, int N2,
                     int64_t sam, int64_t sak, int64_t sbk, int64_t sbn, int64_t swn, int64_t swn2, int64_t scm, int64_t scn,
                     int in_dtype, int out_dtype, const float* a_scale, const float* b_scale,
                     const void* addend, int64_t stride_dm, int64_t stride_dn, int addend_dtype,
                     int activation, int softmax, void* stream_) {
  if (!A || !B || !W || !C || M <= 0 || N <= 0 || K <= 0 || N2 <= 0) return MI355_EINVAL;
  if (softmax != 0 && softmax != 1) return MI355_EINVAL;
  if (activation != MI355_ACT_NONE && activation != MI355_ACT_LEAKY_RELU) return MI355_EINVAL;
  if (in_dtype != MI355_F16 && in_dtype != MI355_BF16) return MI355_EDTYPE;
  if (out_dtype != MI355_F16 && out_dtype != MI355_BF16 && out_dtype != MI355_F32) return MI355_EDTYPE;
  if (addend && addend_dtype != MI355_F16 && addend_dtype != MI355_BF16 && addend_dtype != MI355_F32) return MI355_EDTYPE;
  if (N > 256 || N2 > 256) return MI355_ESHAPE;   // the intermediate row must fit one tile (callers chain two products otherwise)
  if (!device_info().gfx950) return MI355_EDEVICE;
  RowFusedArgs r{A, B, C, W, M, N, K, N2, sam, sak, sbk, sbn, swn, swn2, scm, scn, a_scale, b_scale,
                 activation, softmax, out_dtype, addend, stride_dm, stride_dn, addend_dtype};
  return gemm_rowfused_launch(r, in_dtype == MI355_BF16, (hipStream_t)stream_);
}

int mi355_grouped_gemm(const void* d_a_ptrs, const void* d_b_ptrs, const void* d_c_ptrs,
                       const int32_t* d_sizes, const int32_t* d_lds, int group_size,
                       int dtype, int num_programs, void* stream_) {
  if (!d_a_ptrs || !d_b_ptrs || !d_c_ptrs || !d_sizes || !d_lds || group_size < 0 || num_programs < 0) return MI355_EINVAL;
  if (dtype != MI355_F16 && dtype != MI355_BF16) return MI355_EDTYPE;
  if (!device_info().gfx950) return MI355_EDEVICE;
  if (group_size == 0) return MI355_OK;
  GroupedArgs ga{};
  ga.a_ptrs = (const uint64_t*)d_a_ptrs; ga.b_ptrs = (const uint64_t*)d_b_ptrs; ga.c_ptrs = (const uint64_t*)d_c_ptrs;
  ga.sizes = d_sizes; ga.lds = d_lds; ga.group_size = group_size; ga.out_dtype = dtype;
  const int cus = device_info().cus > 0 ? device_info().cus : 256;
  const int nprog = num_programs > 0 ? num_programs : 2 * cus;
  // groups with at least one 256x256 tile per CU run 256x256 tiles, one program per CU (never more
  // programs than the caller asked for); MI355_GROUPED_BIG_MIN moves the threshold (a huge value = never)
  const int nprog_big = nprog < cus ? nprog : cus;
  ga.big_tiles_min = knob(knobs().grouped_big_min, cus);
  // smallest K of a group of whole 256x256 tiles that the four-wave 16x16-MFMA kernel takes (0 = never)
  ga.wave128_min_k = knob(knobs().grouped_wave128_min_k, 512);
  ga.chunk = knob(knobs().grouped_chunk, 4);
  if (ga.chunk < 1) ga.chunk = 1;
  return gemm16_grouped_launch(ga, dtype == MI355_BF16, nprog, nprog_big, (hipStream_t)stream_);
}

int mi355_grouped_gemm_host(const void* const* a, const void* const* b, void* const* c,
                            const int32_t* sizes, const int32_t* lds, int group_size,
                            int dtype, int num_programs, void* stream_) {
  if (!a || !b || !c || !sizes || !lds || group_size < 0 || num_programs < 0) return MI355_EINVAL;
  if (dtype != MI355_F16 && dtype != MI355_BF16) return MI355_EDTYPE;
  for (int i = 0; i < group_size; i++) {
    const int32_t *s = sizes + 3 * i, *l = lds + 3 * i;
    if (!a[i] || !b[i] || !c[i] || s[0] <= 0 || s[1] <= 0 || s[2] <= 0) return MI355_EINVAL;
    if (l[2] < s[1]) return MI355_ESTRIDE;   // (rows of C must not overlap; those of A and B may)
  }
  if (!device_info().gfx950) return MI355_EDEVICE;
  hipStream_t stream = (hipStream_t)stream_;
  const int cus = device_info().cus > 0 ? device_info().cus : 256;
  const bool bf16 = dtype == MI355_BF16;
  constexpr int G = GroupedTable::kMax;
  for (int g0 = 0; g0 < group_size; g0 += G) {
    const int count = std::min(G, group_size - g0);
    int order[G], n = 0, odd[G], nodd = 0;
    bool whole = true;
    long tiles256 = 0;
    for (int i = 0; i < count; i++) {
      const int32_t *s = sizes + 3 * (g0 + i), *l = lds + 3 * (g0 + i);
      // rows of 16-byte chunks that do not overlap, pitches within the kernels' lane offsets: else the kernel of any strides
      if (s[2] % 8 || l[0] % 8 || l[0] < s[2] || l[1] % 8 || l[1] < (s[1] + 7) / 8 * 8 || !aligned(a[g0 + i], 16) || !aligned(b[g0 + i], 16) || l[0] >= (1 << 22) || l[1] >= (1 << 25)) {
        odd[nodd++] = i;
        continue;
      }
      tiles256 += (long)((s[0] + 255) / 256) * ((s[1] + 255) / 256);
      whole = whole && s[0] % 256 == 0 && s[1] % 256 == 0 && s[2] % 128 == 0 && s[2] >= knob(knobs().grouped_wave128_min_k, 512) && l[1] % 256 == 0 &&
              (int64_t)l[0] * 16 + s[2] * 2 < (1ll << 31) && (int64_t)s[2] * l[1] * 2 + 512 < (1ll << 31);
      order[n++] = i;
    }
    auto put = [&](GroupedTable& ga, int at, int i) {
      ga.a_ptrs[at] = (uint64_t)a[g0 + i]; ga.b_ptrs[at] = (uint64_t)b[g0 + i]; ga.c_ptrs[at] = (uint64_t)c[g0 + i];
      for (int e = 0; e < 3; e++) { ga.sizes[3 * at + e] = sizes[3 * (g0 + i) + e]; ga.lds[3 * at + e] = lds[3 * (g0 + i) + e]; }
    };
    int rc;
    if (nodd > 0) {
      GroupedTable ga{};
      int64_t tiles = 0;
      for (int at = 0; at < nodd; at++) {
        put(ga, at, odd[at]);
        ga.first_tile[at] = (int)std::min<int64_t>(tiles, INT_MAX);
        tiles += (int64_t)((ga.sizes[3 * at] + 63) / 64) * ((ga.sizes[3 * at + 1] + 63) / 64);
      }
      for (int at = nodd; at < G; at++) ga.first_tile[at] = INT_MAX;
      if (nodd > 1 && tiles <= INT_MAX / 2) {
        ga.group_size = nodd; ga.out_dtype = dtype; ga.total_tiles = (int)tiles;
        rc = gemm_masked_grouped_launch(ga, bf16, stream);
        if (rc) return rc;
      } else {
        for (int at = 0; at < nodd; at++) {
          const int32_t *s = sizes + 3 * (g0 + odd[at]), *l = lds + 3 * (g0 + odd[at]);
          rc = mi355_gemm(a[g0 + odd[at]], b[g0 + odd[at]], c[g0 + odd[at]], s[0], s[1], s[2], l[0], 1, l[1], 1, l[2], 1, dtype, dtype, nullptr, nullptr, MI355_ACT_NONE, stream_);
          if (rc) return rc;
        }
      }
    }
    if (n == 0) continue;
    GroupedTable ga{};
    ga.group_size = n; ga.out_dtype = dtype;
    ga.chunk = std::max(1, knob(knobs().grouped_chunk, 4));
    if (whole && knobs().grouped_wave128_min_k != 0 && tiles256 >= knob(knobs().grouped_big_min, cus)) {
      // whole 256x256 tiles, at least one per CU: runs of them as one stream of K steps
      for (int at = 0; at < n; at++) put(ga, at, order[at]);
      ga.total_tiles = (int)tiles256;
      rc = gemm_wave128_grouped_table_launch(ga, bf16, num_programs > 0 ? std::min(num_programs, cus) : cus, stream);
    } else {
      // the longest tiles first, so that the last ones to be started are short
      std::stable_sort(order, order + n, [&](int x, int y) { return sizes[3 * (g0 + x) + 2] > sizes[3 * (g0 + y) + 2]; });
      const int forced = knobs().grouped_shape;
      GroupPlan plan = group_plan(sizes + 3 * g0, order, n, cus, forced == 0 || forced == 2 || forced == 4 || forced == 5 ? forced : -1);
      plan.chunk = std::min(knob(knobs().grouped_run, plan.chunk), 1024);
      int64_t tiles = 0;
      for (int at = 0; at < n; at++) {
        put(ga, at, order[at]);
        ga.first_tile[at] = (int)tiles;
        const int edge = plan.small_tiles >> at & 1 ? 64 : 128;
        tiles += (int64_t)((ga.sizes[3 * at] + edge - 1) / edge) * ((ga.sizes[3 * at + 1] + edge - 1) / edge);
        if (tiles > INT_MAX / 2) return MI355_ESHAPE;
      }
      for (int at = n; at < G; at++) ga.first_tile[at] = INT_MAX;
      ga.total_tiles = (int)tiles;
      ga.small_tiles = plan.small_tiles;
      ga.chunk = plan.chunk;
      ga.padded_tiles = plan.chunk > 0 ? (ga.total_tiles + 8 * plan.chunk - 1) / (8 * plan.chunk) * (8 * plan.chunk) : ga.total_tiles;
      rc = gemm_ring_grouped_launch(ga, bf16, plan.shape, num_programs > 0 ? std::min(num_programs, ga.total_tiles) : ga.padded_tiles, stream);
    }
    if (rc) return rc;
  }
  return MI355_OK;
}

// A K step of the block-scaled ring kernels takes 1.3 times the others' (1024 x 4096 x 4096, 128x128 tiles: e4m3 18.3 us, MXFP8
// 23.7; 4096^3 MXFP8 90, MXFP4 59, half as many steps).
constexpr double kMxStep = 1.3;

// Splits of K of a block-scaled product that has a workspace (1 = none), as auto_splits for the other ring kernels.
static int mx_splits(int M, int N, int64_t k_bytes, int cus) {
  const int steps = (int)((k_bytes + 127) / 128);
  const int most = (int)std::min<int64_t>(std::min<int64_t>(32, steps / 2), (64ll << 20) / std::max<int64_t>(1, 4ll * M * N));
  if (knob(knobs().splitk, 1) == 0 || most < 2 || steps < 16) return 1;
  const RingPlan split = ring_plan(M, N, steps, cus, 2, most, kMxStep);
  return split.us < 0.95 * ring_plan(M, N, steps, cus, 1, 1, kMxStep).us ? split.splits : 1;
}

int64_t mi355_mx_gemm_workspace(int M, int N, int K, int fmt) {
  if (M <= 0 || N <= 0 || K <= 0 || K % 128 != 0 || (fmt != MI355_MXFP4 && fmt != MI355_MXFP8)) return 0;
  const int splits = mx_splits(M, N, fmt == MI355_MXFP4 ? K / 2 : K, device_info().cus > 0 ? device_info().cus : 256);
  return splits > 1 ? (int64_t)splits * M * N * 4 : 0;
}

static int mx_impl(const uint8_t* A, const uint8_t* sA, const uint8_t* B, const uint8_t* sB, void* C,
                   int M, int N, int K, int fmt, int out_dtype,
                   int64_t lda, int64_t ldb, int64_t lds_a, int64_t lds_b, int64_t ldc, void* workspace, size_t workspace_bytes, void* stream_) {
  if (!A || !sA || !B || !sB || !C || M <= 0 || N <= 0 || K <= 0) return MI355_EINVAL;
  if (fmt != MI355_MXFP4 && fmt != MI355_MXFP8) return MI355_EINVAL;
  if (out_dtype != MI355_F16 && out_dtype != MI355_BF16 && out_dtype != MI355_F32) return MI355_EDTYPE;
  if (!device_info().gfx950) return MI355_EDEVICE;
  if (K % 32 != 0) return MI355_ESHAPE;  // whole scale blocks only
  const int64_t row_bytes = fmt == MI355_MXFP4 ? K / 2 : K;
  if (lda < row_bytes || ldb < row_bytes || lds_a < K / 32 || lds_b < K / 32 || ldc < N) return MI355_ESTRIDE;
  if (lda % 16 || ldb % 16 || !aligned(A, 16) || !aligned(B, 16)) return MI355_ESTRIDE;
  if (lda >= (1 << 23) || ldb >= (1 << 23)) return MI355_ESTRIDE;  // 32-bit offsets inside a 256-row tile
  GemmArgs p{};
  p.A = (const char*)A; p.B = (const char*)B; p.C = (char*)C;
  p.M = M; p.N = N; p.K = K; p.k_bytes = (int)row_bytes;
  p.lda = lda; p.ldb = ldb; p.ldc = ldc; p.scn = 1;
  p.out_dtype = out_dtype;
  p.group_m = knob(knobs().group_m, 8);
  p.c_vec_ok = ldc % 4 == 0 && aligned(C, 16);
  p.lean_ok = knob(knobs().lean_epilogue, 1);
  p.sA = sA; p.sB = sB; p.lds_a = lds_a; p.lds_b = lds_b;
  const int cus = device_info().cus > 0 ? device_info().cus : 256;
  const long tiles256 = (long)((M + 255) / 256) * ((N + 255) / 256);
  int tile = (tiles256 * 2 >= cus) ? (tiles256 % cus == 0 ? 5 : 4) : 1;
  // MXFP4 from 256 rows and columns, 256 bytes of K and half a round of tiles on: four waves of
  // scaled 16x16x128 MFMAs (8192^3: 4000-4050 vs 3340-3640 TFLOP/s for the persistent eight-wave kernel)
  const int group = fmt == MI355_MXFP4 ? 512 : 1024;   // bytes of a row in a group of K steps of their streaming forms
  // (below half a round of tiles too where K is long, next to the ring kernels below)
  const bool enough = tiles256 * 2 >= cus || (tiles256 >= 16 && p.k_bytes >= 1024);
  if (fmt == MI355_MXFP4 && enough && gemm_wave128_mxfp4_ok(p)) tile = 6;
  // (MXFP8 likewise: 2530-2570 vs 2110-2240)
  if (fmt == MI355_MXFP8 && enough && gemm_wave128_mxfp8_ok(p)) tile = 6;
  // the same kernels on tiles of 128 x 256 wherever those fit one round of CUs (from 16 on): flushed do_bench, best of
  // the other forms / 128-row tiles, MXFP4: 1024^3 141 / 162 TFLOP/s, 2048 x 2048 x 1024 503 / 600, 2048 x 2048 x 4096 1012 /
  // 1309, 1536 x 2048 x 8192 1071 / 1216, 3072 x 2048 x 4096 1661 / 1854, 2304 x 2048 x 8192 1606 / 1795; MXFP8: 92 / 127,
  // 360 / 491, 644 / 856, 627 / 754, 1072 / 1244, 947 / 1120; beyond one round they lose (3072^3, 288 tiles: MXFP4 2084 for
  // the 192-row tiles / 1555, 4096^3 3209 / 2834)
  if ((knobs().tile == UNSET || knobs().tile_m == 128) && gemm_wave128_mx_192_ok(p, group, 128)) {
    const long tiles128 = (long)((M + 127) / 128) * ((N + 255) / 256);
    const int want = knob(knobs().tile_m, 0);
    if (want == 128 || (want == 0 && tiles128 >= 16 && tiles128 <= cus)) {
      tile = 6;
      p.tile_m = 128;
    }
  }
  // and on tiles of 192 x 256 where those fill the CUs better (as for the 16-bit and fp8 products).  Flushed
  // do_bench, 256-row choice / 192-row tiles, MXFP4: 3072^3 1750 / 2100 TFLOP/s, 4608 x 4096 x 4096 2475 / 2885, 6144^3
  // 3725 / 3970, 1536 x 8192 x 8192 3205 / 3780, 1536 x 2048 x 8192 880 / 1080; MXFP8: 1255 / 1420, 1480 / 1830, 2275 / 2520,
  // 1945 / 2345, 519 / 630; not taken where they fill worse (3840 x 3840 x 4096: 3080 / 2230)
  if ((knobs().tile == UNSET || knobs().tile_m == 192) && p.tile_m == 0 && gemm_wave128_mx_192_ok(p, group)) {
    auto fill = [&](long t) { return t <= 0 ? 0.0 : (double)t / (double)(((t + cus - 1) / cus) * cus); };
    const long tiles192 = (long)((M + 191) / 192) * ((N + 255) / 256);
    const int want = knob(knobs().tile_m, 0);
    const bool enough192 = tiles192 * 2 >= cus || (tiles192 >= 16 && p.k_bytes >= 1024);
    if (want == 192 || (want == 0 && enough192 && (tile != 6 || fill(tiles192) > fill(tiles256) * 1.1))) {
      tile = 6;
      p.tile_m = 192;
    }
  }
  // Few K steps and more than a round of tiles: the kernels without a ring's prologue, 128x128 tiles of one barrier per step below half a round of
  // 256x256 tiles and the eight-wave kernel from there on where its columns are whole.  us, ring / these, MXFP4: 1024 x 5888 x 128 10.5 / 8.1, 4352 x 1600 x 256
  // 11.4 / 9.2, 4608 x 3328 x 128 17.9 / 10.6, 4800 x 7168 x 128 36.4 / 23.2, 7680 x 7936 x 384 69 / 44; MXFP8 3608 x 1720 x 128 10.3 / 8.7, 2368 x 5376 x 128 17.3 / 11.8; partial
  // columns: MXFP4 4608 x 3264 x 256 17.8 / 21.5, MXFP8 2240 x 4160 x 128 13.2 / 15.4; odd rows of C 5924 x 2670 x 128 21 / 67.  MXFP8 of several rounds ahead of the four-wave
  // kernel too: 6144 x 6656 x 512 48.6 / 40.7, 5632 x 4608 x 256 28.4 / 24.7, not of one and a bit: 4608 x 4096 x 256 22 / 24.
  bool few_steps = false;
  if (knobs().tile == UNSET && knobs().tile_m == UNSET && knobs().mixed_rows == UNSET && K % 128 == 0 && p.c_vec_ok) {
    if (tile == 1) few_steps = p.k_bytes <= 256 && (long)((M + 127) / 128) * ((N + 127) / 128) > cus;
    else if (tile != 6) few_steps = p.k_bytes <= 192 && N % 256 == 0;
    else if (fmt == MI355_MXFP8 && p.tile_m == 0 && p.k_bytes <= 512 && N % 256 == 0 && tiles256 * 5 > 7 * cus) {
      few_steps = true;
      tile = tiles256 % cus == 0 ? 5 : 4;
    }
  }
  p.num_programs = knob(knobs().programs, cus);
  // the ring kernels of 64 .. 128-row tiles, split along K where there is a workspace, where they are the faster ones by the
  // estimates of the other products (MXFP4 steps hold twice the elements in the same bytes, which are what bounds both).  us, the
  // 128x128 kernel of one barrier per step / ring: MXFP8 567 x 1280 x 5888 73 / 18, 2304 x 1536 x 4480 64 / 26, 256 x 3968 x 3840 42 /
  // 9, MXFP4 192 x 1152 x 5120 38 / 7, 1024 x 1920 x 5632 39 / 14; the four-wave kernels on few tiles / ring: MXFP4 1024 x 4096 x 4096
  // 18.6 / 15.1, MXFP8 31.5 / 23.7, 512 x 8192 x 8192 56 / 41; these stay ahead from about a round of their tiles on (2048 x 4096 x 4096
  // MXFP4 23.6 / 29.8, MXFP8 34 / 45)
  const bool ring_takes = K % 128 == 0 && lds_a % 4 == 0 && lds_b % 4 == 0 && aligned(sA, 4) && aligned(sB, 4) && lds_a < (1 << 24) && lds_b < (1 << 24);
  if (ring_takes && !few_steps && knobs().tile_m == UNSET && knobs().mixed_rows == UNSET) {
    const int steps = (p.k_bytes + 127) / 128;
    int shape = -1, splits = 1;
    if (knobs().tile != UNSET) {
      if ((knobs().tile >= 8 && knobs().tile <= 10) || knobs().tile == 13) shape = knobs().tile == 13 ? 4 : knobs().tile - 8;
    } else {
      // (less room than mi355_mx_gemm_workspace asks for: the plain call)
      if (workspace) splits = mx_splits(M, N, p.k_bytes, cus);
      if (splits > 1 && workspace_bytes < (size_t)splits * M * N * sizeof(float)) splits = 1;
      const RingPlan plan = ring_plan(M, N, steps, cus, splits, splits, kMxStep);
      double other = 1e30;
      if (tile == 6) {
        // (within 15 % of: 4096 x 4096 x 1024 .. 4224 MXFP8 23 .. 58 us, MXFP4 18 .. 45; unlike the 16-bit kernels hardly shorter where
        // they leave CUs idle: 4096 x 1664 x 1408 MXFP8, 112 tiles, 24.7 us - ring 16.5 -, 3072 x 3072 x 3200, 144 tiles, 42 - ring 51)
        const int rows = p.tile_m ? p.tile_m : 256;
        const long tiles = (long)((M + rows - 1) / rows) * ((N + 255) / 256), rounds = (tiles + cus - 1) / cus;
        const double fill = rounds > 1 ? 1.0 : (double)tiles / cus, share = rows == 256 ? 1.0 : rows == 192 ? 0.78 : 0.64;
        other = kLaunchUs + (double)rounds * share * (8.0 + 1.5 * steps * (0.7 + 0.3 * fill));
      }
      if (splits <= 1 && pairs_us(M, N, steps, cus, true, (p.lda | p.ldb) % 128 != 0) < 0.97 * std::min(plan.us, other)) shape = 4;
      else if (plan.us < other) shape = plan.shape;
      else splits = 1;
    }
    if (shape >= 0) {
      const int per = (steps + splits - 1) / splits, used = (steps + per - 1) / per;
      if (used < 2) return gemm_ring_mx_launch(p, fmt == MI355_MXFP4, shape, 1, 0, (hipStream_t)stream_);
      if (!aligned(workspace, 16)) return MI355_EINVAL;
      p.workspace = (float*)workspace;
      const int rc = gemm_ring_mx_launch(p, fmt == MI355_MXFP4, shape, used, per * 128, (hipStream_t)stream_);
      if (rc) return rc;
      GemmStridedArgs out{};
      out.C = C; out.M = M; out.N = N; out.scm = ldc; out.scn = 1; out.out_dtype = out_dtype;
      return splitk_reduce_launch(out, (const float*)workspace, used, (hipStream_t)stream_);
    }
  }
  // and on both tile heights in one launch, as for the 16-bit and fp8 products
  if (knobs().tile == UNSET && knobs().tile_m == UNSET && N % 256 == 0) {
    const int want = knob(knobs().mixed_rows, -1);
    int rows = 0;
    if (want > 0) rows = want;
    else if (want < 0 && tile == 6 && p.tile_m == 0 && tiles256 > cus) rows = mixed_split(M, N / 256, cus);
    if (rows > 0 && gemm_wave128_mx_mixed_ok(p, group, rows)) return gemm_wave128_mx_mixed_launch(p, fmt == MI355_MXFP4 ? 0 : 1, rows, (hipStream_t)stream_);
  }
  tile = knob(knobs().tile, tile);
  return mx_gemm_launch(p, fmt, tile, (hipStream_t)stream_);
}

int mi355_mx_gemm(const uint8_t* A, const uint8_t* sA, const uint8_t* B, const uint8_t* sB, void* C,
                  int M, int N, int K, int fmt, int out_dtype,
                  int64_t lda, int64_t ldb, int64_t lds_a, int64_t lds_b, int64_t ldc, void* stream_) {
  return mx_impl(A, sA, B, sB, C, M, N, K, fmt, out_dtype, lda, ldb, lds_a, lds_b, ldc, nullptr, 0, stream_);
}

int mi355_mx_gemm_ws(const uint8_t* A, const uint8_t* sA, const uint8_t* B, const uint8_t* sB, void* C,
                     int M, int N, int K, int fmt, int out_dtype,
                     int64_t lda, int64_t ldb, int64_t lds_a, int64_t lds_b, int64_t ldc, void* workspace, size_t workspace_bytes, void* stream_) {
  return mx_impl(A, sA, B, sB, C, M, N, K, fmt, out_dtype, lda, ldb, lds_a, lds_b, ldc, workspace_bytes ? workspace : nullptr, workspace_bytes, stream_);
}

int mi355_clock_probe(uint64_t* ticks, int duration_us, void* stream_) {
  if (!ticks || !aligned(ticks, 8) || duration_us <= 0 || duration_us > 2000000) return MI355_EINVAL;
  if (!device_info().gfx950 || device_info().wall_clock_khz <= 0) return MI355_EDEVICE;
  const unsigned long long real_ticks = (unsigned long long)duration_us * (unsigned long long)device_info().wall_clock_khz / 1000ull;
  return clock_probe_launch((unsigned long long*)ticks, real_ticks, (hipStream_t)stream_);
}

int mi355_mfma_burn(float* sink, int shape, int random_operands, int iters, int waves_per_simd, void* stream_) {
  if (!sink || !aligned(sink, 4) || shape < MI355_BURN_BF16_32X32X16 || shape > MI355_BURN_MXFP4_16X16X128) return MI355_EINVAL;
  if (iters <= 0 || iters > (1 << 24) || waves_per_simd < 1 || waves_per_simd > 2) return MI355_EINVAL;
  if (!device_info().gfx950) return MI355_EDEVICE;
  return mfma_burn_launch(sink, shape, random_operands != 0, iters, waves_per_simd, device_info().cus > 0 ? device_info().cus : 256,
                          (hipStream_t)stream_);
}

int mi355_dequant(const uint8_t* codes, float* out, int64_t n, int fmt, void* stream_) {
  if (!codes || !out || n < 0) return MI355_EINVAL;
  if (fmt < MI355_DEQ_E4M3 || fmt > MI355_DEQ_E8M0) return MI355_EINVAL;
  if (n == 0) return MI355_OK;
  if (n > (int64_t)0x7FFFFFFF * 256) return MI355_ESHAPE;
  return dequant_launch(codes, out, n, fmt, (hipStream_t)stream_);
}

static int attn_common(AttnArgs& p, int Z, int H, int N_CTX, int D, int dtype) {
  if (Z <= 0 || H <= 0 || N_CTX <= 0) return MI355_EINVAL;
  if (dtype != MI355_F16 && dtype != MI355_BF16) return MI355_EDTYPE;
  // head_dim 256 and the padded forms of head dims 16 / 32: the forward kernels of every type and the backward
  const bool small = D == 16 || D == 32;
  if (D != 64 && D != 128 && D != 256 && !small) return MI355_ESHAPE;
  if (N_CTX % 128 != 0) return MI355_ESHAPE;
  if (!device_info().gfx950) return MI355_EDEVICE;
  // 16 / 32: the 64-column kernels, which pad with zeros on the fly (loads, LDS tiles and stores know d_real)
  p.Z = Z; p.H = H; p.N = N_CTX; p.D = small ? 64 : D; p.d_real = D;
  p.cus = std::min(device_info().cus > 0 ? device_info().cus : 256, 32767);
  return MI355_OK;
}

static bool attn_stride_ok(const int64_t* s, const void* ptr, int D) {
  // rows at most 2^24 elements apart: the kernels address 64 rows of a tile with 32-bit byte offsets
  return s[3] == 1 && s[2] >= D && s[2] < (1 << 24) && s[0] % 8 == 0 && s[1] % 8 == 0 && s[2] % 8 == 0 && aligned(ptr, 16);
}

// Steps of 64 keys that the busiest program of the causal persistent form walks: blocks of 256 rows dealt one after the other to
// `programs`, whole rounds of heads long-to-short and short-to-long in turn (attn_fwd_stream_kernel).
// A round of heads is at most one block a program, so it is added as one run (512 heads x 2048: 1.2 us of host time, block by block 15).
static int64_t stream_busiest(int64_t heads, int N, int programs) {
  constexpr int kMost = 1024;
  const int nb = (N + 255) / 256, G = (int)std::min<int64_t>(std::min(programs, kMost), heads * nb), per_round = std::max(1, G / nb);
  int steps[kMost], run[2][kMost];
  std::fill(steps, steps + G, 0);
  auto block = [&](int b) { return (std::min(N, (b + 1) * 256) + 63) / 64; };
  int at = 0;
  if (nb > G) {   // (a head is more than a block a program)
    for (int64_t h = 0; h < heads; h++)
      for (int j = 0; j < nb; j++) {
        steps[at] += block(h & 1 ? j : nb - 1 - j);
        if (++at == G) at = 0;
      }
    return *std::max_element(steps, steps + G);
  }
  for (int j = 0; j < nb; j++) run[0][nb - 1 - j] = run[1][j] = block(j);
  const int round = (int)std::min<int64_t>(heads, per_round) * nb;
  for (auto& r : run)
    for (int n = nb; n < round; n *= 2) std::copy_n(r, std::min(n, round - n), r + n);
  bool up = false;
  for (int64_t left = heads; left > 0; left -= per_round, up = !up) {
    const int len = (int)std::min<int64_t>(left, per_round) * nb, first = std::min(len, G - at);
    for (int i = 0; i < first; i++) steps[at + i] += run[up][i];
    for (int i = first; i < len; i++) steps[i - first] += run[up][i];
    at += len;
    if (at >= G) at -= G;
  }
  return *std::max_element(steps, steps + G);
}

// Which form of the forward: the fewer query rows there are for the CUs, the smaller a workgroup's block of rows and the more
// of its waves go along the keys instead (us, fp16, causal / not, by form: 2 = 256 rows, 4 = its persistent form, 1 = 128
// rows, 8 = 128 rows x 2 groups, 6 = 64 x 2, 7 = 32 x 4).
static int attn_fwd_variant(const AttnArgs& p, int cus) {
  const int dflt = p.causal ? 4 : 2;
  if (p.D == 256 || p.d_real < p.D) return dflt;
  const int64_t rows = (int64_t)p.Z * p.H * p.N;
  // head_dim 64, 8 heads x 1024: 7 8.3 / 8.2, 6 10.3 / 10.2, 8 12.7 / 12.6, 1 15.0 / 14.6
  if (p.D == 64 && p.N % 256 == 0 && rows <= 32ll * cus) return 7;
  // 16 x 1024: 6 10.4 / 10.5, 7 12.1 / 15.0, 8 12.9 / 12.8; head_dim 128: 6 15.7 / 16.3, 8 18.7 / 18.5, 1 20.9 / 20.6
  if (rows <= 64ll * cus) return 6;
  // 16 x 2048: 8 22.4 / 24.9, 6 24.0 / 27.0, 1 26.7 / 27.5; head_dim 128: 8 32.6 / 40.1, 6 32.2 / 50.6, 1 36.9 / 41.5
  // (two blocks of keys are not worth the groups' meeting: 256 x 128, no mask, head_dim 128: 8 10.2, 2 8.8; causal 8 ahead)
  if (!p.causal) return rows <= 128ll * cus && p.N > 128 ? 8 : dflt;
  // Under the mask, with the blocks dealt by length (deal_blocks).  us, 6 / 8 / 1 / 2 / 4:
  if (p.D == 64) {
    // (one round of blocks of 256 rows, 104 x 384 9.2 / 8.9 on 1 / 2; 86 x 512 10.7 / 12.4)
    if (p.N > 256 && p.N <= 384 && rows > 128ll * cus && (int64_t)p.Z * p.H * 2 <= cus) return 2;
    // short rows: 48 x 640 9.4 / 10.3 / 11.1 / 12.6 / 14.6, 77 x 512 14.3 / 11.0 / 10.9 / 13.1 / 14.8, 256 x 512 26.6 / 21.9 / 18.9 / 19.1 / 22.7
    if (p.N < 1024) return rows <= 128ll * cus ? 6 : 1;
    // 14 x 2688 26.1 / 29.8 / 34.2 / 44.6 / 48.0, 24 x 2048 25.7 / 25.8 / 28.8 / 37.3 / 39.8, 25 x 2304 35.2 / 32.3 / 34.2 / 41.3 / 44.3
    // 16 x 3200 35.4 / 37.0 / 40.9 / 53.3 / 57.0
    if (rows <= (p.N >= 2560 ? 200ll : 192ll) * cus) return 6;
    // 24 x 5632 145 / 127 / 136 / 148 / 239, 64 x 2048 57.1 / 48.0 / 49.4 / 52.8 / 51.8; 66 x 1024 24.0 / 21.6 / 21.4 / 23.1 / 30.0, 128 x 1024
    // 37.2 / 29.3 / 28.4 / 29.8 / 32.1; 64 x 4096 199 / 170 / 177 / 161 / 180, 174 x 1152 66.1 / 52.5 / 48.6 / 51.0 / 66.6
    if (p.N < 1536) return 1;
    return rows <= 640ll * cus ? 8 : 2;
  }
  // 24 x 896 15.4 / 17.1 / 18.8 / 21.6 / 24.8, 16 x 1536 20.7 / 24.4 / 28.4 / 36.8 / 40.8; 30 x 768 16.5 / 15.7 / 17.0 / 21.7 / 25.0
  if (rows <= 96ll * cus && p.N >= 896) return 6;
  // 76 x 384 15.0 / 11.6 / 11.3 / 11.5 / 14.4, 52 x 512 16.5 / 12.9 / 13.0 / 16.6 / 19.7, 51 x 640 23.2 / 15.6 / 16.8 / 17.1 / 20.2; 88 x 640 31.4 /
  // 23.7 / 20.8 / 23.5 / 33.1, 256 x 256 29.2 / 20.6 / 14.8 / 15.7 / 17.5; one round of blocks of 256 rows, 105 x 384 24.7 / 19.4 / 15.0 / 13.1 / 15.3,
  // 125 x 512 39.3 / 26.1 / 21.4 / 20.7 / 22.0
  const int64_t heads = (int64_t)p.Z * p.H, nb = (p.N + 255) / 256, blocks = heads * nb, blocks128 = heads * ((p.N + 127) / 128);
  if (p.N <= 640) return blocks128 <= cus ? (p.N >= 512 ? 8 : 1) : p.N > 256 && blocks <= cus ? 2 : 1;
  // More than a round of blocks of 128 rows in short heads, where what two rounds by length even out (deal_blocks) is most of a head: 1 / 2 / 4 / 8: 54 x 768 20.0 / 22.5 / 25.9 / 21.5, 60 x 1024
  // 27.6 / 29.7 / 33.2 / 29.4, 54 x 1152 30.2 / 30.8 / 52.6 / 31.8, 128 x 896 39.2 / 40.7 / 46.9 / 52.8, 216 x 896 60.7 / 77.8 / 87.7 / 82.9, 154 x 1280 79 / 83 / 106 / 99
  // (few rounds of longer ones stay: 40 x 1024 23.7 on 1, 21.6 on 8, 35 x 1280 28.9 / 25.7)
  if (p.N <= 1280 && blocks128 * 10 > cus * (p.N < 1024 ? 12ll : 16ll)) return 1;
  // 32 x 2048 60.8 / 44.4 / 47.9 / 52.4 / 56.4, 10 x 4736 92.8 / 74.2 / 88.3 / 98.7 / 106
  if (rows <= 256ll * cus) return 8;
  // 16 x 5248 168 / 139 / 135 / 143 / 175, 30 x 2944 116 / 88.7 / 78.5 / 80.1 / 110; 20 x 5632 237 / 178 / 181 / 166 / 236, 39 x 2560 161 / 92 / 84 / 75 / 112
  if (rows <= 360ll * cus) return 1;
  // The persistent form where its programs get the same work (`dealt`: the busiest program's share against an even one) over
  // many rounds: 256 x 1024 161 / 118 / 98.0 / 99.9 / 96.1, 128 x 4096 879 / 658 / 584 / 579 / 567; 64 x 4096 411 / 307 / 286 / 272 / 277
  if (blocks >= 4ll * cus) {
    const double work = 0.5 * (double)heads * p.N * (p.N + 256.0);
    const double dealt = (double)stream_busiest(heads, p.N, cus) * 64 * 256 * cus / work;
    if (dealt < 1.02) return 4;
  }
  return 2;
}

// The same for fp8: 1 = 128 rows a workgroup (eight waves along 256 rows are 6 to 12 % slower), and as above 8, 6 and 7 = groups along the keys.
// us, e5m2, 1 / 6 / 8 / 7; rows per CU in brackets.  The groups' sums differ from the one's as their running maxima do (P has two bits of fraction): with
// unit scores by up to 2.2 % of the result without a mask at 4096 keys, with it 1 % at 6144 and 1.3 % at 24576, with scores three times as wide 4 to 6 %.  They are as close to
// 64 bits as the one's or closer, with the mask 0.998 .. 1.0003 of its error at 1024 .. 32768 keys with unit scores and 0.93 .. 0.98 with the wide ones, whose maxima rise less
// often within a group.  So the mask has no limit of length; longer rows without one stay on one group, which was not measured against 64 bits there.
static int attn_fwd8_variant(const AttnArgs& p, int cus) {
  if (p.D == 256 || p.d_real < p.D || p.N < 256 || (!p.causal && p.N > 4096)) return 1;
  const int64_t rows = (int64_t)p.Z * p.H * p.N;
  if (p.D == 64) {
    // mask: 2 x 3840 [30] 37.6 / 22.0 / 31.8 / 15.1, 4 x 6144 [96] 59.6 / 34.7 / 49.1 / 29.2, 8 x 3328 [104] 34.3 / 21.2 / 28.6 / 20.8, 37 x 256 [37] 6.3 / 5.4 /
    // 6.3 / 5.8; none: 4 x 4096 [64] 41.7 / 24.8 / 34.4 / 22.9, 27 x 1536 [162] 25.9 / 21.1 / 25.1 / 28.1; short rows, mask: 40 x 512 [80] 7.6 / 5.7 / 7.2 / 8.5, 24 x 768
    // [72] 9.8 / 6.9 / 8.9 / 8.3, 16 x 1536 [96] 16.7 / 10.6 / 14.6 / 12.0, 16 x 1024 [64] 12.0 / 8.0 / 10.7 / 6.6; none: 24 x 512 [48] 7.2 / 5.5 / 7.0 / 6.1, 16 x 768 [48] 9.5 / 6.7 / 8.8 / 7.1
    if (p.N % 256 == 0 && p.N >= 512 && rows <= (p.N < 2048 ? p.causal ? 64ll : 32ll : p.causal ? 96ll : 64ll) * cus) return 7;
    // mask: 17 x 2432 [162] 27.7 / 19.9 / 23.9, 83 x 512 [166] 9.3 / 8.5 / 9.3, 71 x 1024 [284] 16.3 / 15.8 / 16.2, 143 x 640 [358] 13.7 / 14.3 / 14.7, 61 x
    // 2048 [488] 38.3 / 37.2 / 35.5; none: 39 x 1152 [176] 20.8 / 17.3 / 19.9, 78 x 256 [78] 6.2 / 6.4 / 6.4, 211 x 384 [316] 13.0 / 13.4 / 14.5
    if (rows <= 64ll * cus || (rows <= (p.causal ? 200ll : 180ll) * cus && p.N >= (p.causal ? 256 : 640)) || (p.causal && rows <= 300ll * cus && p.N >= 1024)) return 6;
    return p.causal && rows <= 560ll * cus && p.N >= 1536 ? 8 : 1;
  }
  // mask: 2 x 2560 [20] 32.7 / 21.4 / 27.3, 63 x 384 [94] 9.5 / 8.5 / 9.6, 6 x 4992 [117] 59.9 / 40.7 / 48.2, 61 x 640 [152] 13.5 / 14.6 / 14.0, 35 x 2048
  // [280] 33.4 / 35.8 / 39.8; none: 5 x 2944 [58] 38.1 / 25.3 / 31.5, 31 x 640 [78] 11.9 / 12.2 / 11.6, 6 x 3968 [93] 51.2 / 44.3 / 41.4, 18 x 1664 [117]
  // 24.3 / 22.8 / 21.6, 17 x 2944 [196] 58.9 / 67.7 / 64.7
  if (rows <= 64ll * cus || (p.causal && rows <= 128ll * cus && p.N >= 384)) return 6;
  return !p.causal && rows <= 128ll * cus && p.N >= 1024 ? 8 : 1;
}

int mi355_attn_fwd(const void* q, const void* k, const void* v, void* o, float* Mlse,
                   int Z, int H, int N_CTX, int D,
                   const int64_t* sq, const int64_t* sk, const int64_t* sv, const int64_t* so,
                   float sm_scale, int causal, int dtype, void* stream_) {
  if (!q || !k || !v || !o || !Mlse) return MI355_EINVAL;
  AttnArgs p{};
  if (dtype == MI355_F8E5M2 || dtype == MI355_F8E4M3) {
    // fp8 forward: q, k, o with D contiguous, v with N_CTX contiguous (transposed in memory)
    int rc8 = attn_common(p, Z, H, N_CTX, D, MI355_F16);
    if (rc8) return rc8;
    if (!copy_strides(sq, p.sq) || !copy_strides(sk, p.sk) || !copy_strides(sv, p.sv) || !copy_strides(so, p.so))
      return MI355_EINVAL;
    auto rows16 = [&](const int64_t* s, const void* ptr) {
      return s[3] == 1 && s[2] >= D && s[2] < (1 << 24) && s[0] % 16 == 0 && s[1] % 16 == 0 && s[2] % 16 == 0 && aligned(ptr, 16);
    };
    if (!rows16(p.sq, q) || !rows16(p.sk, k) || !rows16(p.so, o)) return MI355_ESTRIDE;
    if (!(p.sv[2] == 1 && p.sv[3] >= N_CTX && p.sv[3] < (1 << 24) && p.sv[0] % 16 == 0 && p.sv[1] % 16 == 0 && p.sv[3] % 16 == 0 && aligned(v, 16)))
      return MI355_ESTRIDE;
    p.q = (const char*)q; p.k = (const char*)k; p.v = (const char*)v; p.o = (char*)o; p.lse = Mlse;
    p.sm_scale = sm_scale; p.causal = causal != 0;
    p.variant = knob(knobs().attn_fwd_variant, attn_fwd8_variant(p, p.cus));
    return attn_fwd8_launch(p, dtype == MI355_F8E5M2, (hipStream_t)stream_);
  }
  int rc = attn_common(p, Z, H, N_CTX, D, dtype);
  if (rc) return rc;
  if (!copy_strides(sq, p.sq) || !copy_strides(sk, p.sk) || !copy_strides(sv, p.sv) || !copy_strides(so, p.so))
    return MI355_EINVAL;
  if (!attn_stride_ok(p.sq, q, D) || !attn_stride_ok(p.sk, k, D) || !attn_stride_ok(p.sv, v, D) ||
      !attn_stride_ok(p.so, o, D))
    return MI355_ESTRIDE;
  p.q = (const char*)q; p.k = (const char*)k; p.v = (const char*)v; p.o = (char*)o; p.lse = Mlse;
  p.sm_scale = sm_scale; p.causal = causal != 0;
  // eight waves (256 query rows) per K/V stream halve the L2 -> LDS traffic.  Under the causal mask
  // their row ranges are uneven, which the persistent form (4) evens out by pairing long and short
  // query blocks per program; without a mask the one-item-per-workgroup form (2) is the faster one.
  p.variant = knob(knobs().attn_fwd_variant, attn_fwd_variant(p, p.cus));
  p.num_programs = std::min(knob(knobs().attn_programs, p.cus), 32767);
  // 5: four waves of 64 query rows, 16x16x32 MFMAs, software pipelined inside the wave (head_dim 128)
  if (p.variant == 5 && attn_fwd_pipe_ok(p)) return attn_fwd_pipe_launch(p, dtype == MI355_BF16, (hipStream_t)stream_);
  return attn_fwd_launch(p, dtype == MI355_BF16, (hipStream_t)stream_);
}

int mi355_attn_bwd_preprocess(const void* o, const void* d_o, float* delta,
                              int Z, int H, int N_CTX, int D, const int64_t* stride, int dtype, void* stream_) {
  if (!o || !d_o || !delta) return MI355_EINVAL;
  AttnArgs p{};
  int rc = attn_common(p, Z, H, N_CTX, D, dtype);
  if (rc) return rc;
  if (!copy_strides(stride, p.so)) return MI355_EINVAL;
  if (!attn_stride_ok(p.so, o, D) || !aligned(d_o, 16)) return MI355_ESTRIDE;
  p.o = (char*)o; p.d_o = (const char*)d_o; p.delta = delta;
  // delta is written through the non-const alias below
  p.lse = delta;
  return attn_bwd_pre_launch(p, dtype == MI355_BF16, (hipStream_t)stream_);
}

// Groups of waves of the backward kernels, dQ + 16 * dK/dV: more than one where the blocks of 128 rows leave CUs without
// work, or under the mask where a few long walks end the launch.  In comments: the backward's us with one group each, and
// what two (four) groups in dQ / in dK/dV change; fp16, causal.
static int attn_bwd_variant(const AttnArgs& p, int cus) {
  if (p.D == 256 || p.d_real < p.D) return 1 + 16;
  const int64_t blocks = (int64_t)p.Z * p.H * p.N / 128;
  // head_dim 64, 8 heads x 1024: 34.4, two -5.4 / -5.8, four -6.6 / -7.5; 16 x 1024: 35.2, four -2.3 / -2.2
  // (6 x 1536: two 29.7, four 25.6; 10 x 1536: 30.5, 35.1)
  if (p.D == 64 && p.N % 256 == 0 && blocks <= (p.causal && p.N >= 1280 ? cus * 5 / 16 : cus / 4)) return 4 + 64;
  // 16 x 1024: two -5.7 / -5.8; head_dim 128: 51.7, -6.9 / -8.2; 24 x 1024: 52.2, +1.1 / +0.3 (full 57.1, +8.1 / +7.6)
  if (blocks <= cus / 2) return 2 + 32;
  // Under the mask (blocks dealt by length, deal_blocks) also where one round of CUs is nearly full, since half as many rows a
  // block even out better: one / two groups in both, 24 x 768 29.4 / 22.3, 28 x 1024 36.2 / 33.8, 8 x 3968 108 / 80.2, 12 x 3328
  // 96.4 / 85.3, 58 x 512 23.5 / 26.1, 19 x 2432 77.9 / 82.6; head_dim 128: 12 x 1664 73.8 / 53.9, 4 x 6528 248 / 175, 24 x 1152 58.4 /
  // 55.6, 48 x 384 29.0 / 33.1, 12 x 3712 169 / 176
  if (!p.causal) return 1 + 16;
  if (p.N >= (p.D == 64 ? 768 : 1024) && blocks <= cus) return 2 + 32;
  // Beyond that round one group each / two in dQ / two in both, the longer the rows the further; head_dim 128: 6 x 5504 219 / 203 / 181, 9 x 4096 174 / 170 / 164,
  // 13 x 2560 112 / 111 / 107, 14 x 2560 114 / 115 / 114, 12 x 3328 148 / 155 / 156, 18 x 2048 95 / 99 / 101
  if (p.D == 128) return p.N >= 2560 && blocks * 8 <= cus * 9ll ? 2 + 32 : 1 + 16;
  // head_dim 64: 14 x 2560 77 / 68 / 65, 16 x 2560 79 / 70 / 70, 14 x 3072 93 / 85 / 85, 8 x 5248 147 / 131 / 125, 7 x 6528 189 / 171 / 168, 9 x 5248 154 / 141 / 142
  if (p.N >= 2560 && blocks * 20 <= cus * (p.N >= 5120 ? 28ll : 25ll)) return 2 + 32;
  // 36 x 1024 39.3 / 38.3, 40 x 1024 39.9 / 40.5, 29 x 1280 45.2 / 42.0, 36 x 1280 48.3 / 48.2, 24 x 1536 51.8 / 46.7, 32 x 1536 55.8 / 54.2, 43 x 1536 72.6 / 73.0, 20 x
  // 2048 65 / 60, 32 x 2048 80.6 / 80.1, 38 x 2048 99 / 100, 16 x 4096 143 / 138, 12 x 6528 264 / 256, 24 x 4096 206 / 208
  const int64_t tenths = p.N >= 4096 ? 24 : p.N >= 2048 ? 20 : p.N >= 1536 ? 15 : p.N >= 1024 ? 12 : 0;
  return blocks * 10 <= cus * tenths ? 2 + 16 : 1 + 16;
}

static int attn_bwd(const void* q, const void* k, const void* v, const void* o, const void* d_o,
                    const float* Mlse, const float* delta, void* dq, void* dk, void* dv,
                    int Z, int H, int N_CTX, int D, const int64_t* stride,
                    float sm_scale, int causal, int dtype, void* stream_) {
  if (!q || !k || !v || !d_o || !Mlse || !delta || !dq || !dk || !dv) return MI355_EINVAL;
  AttnArgs p{};
  int rc = attn_common(p, Z, H, N_CTX, D, dtype);
  if (rc) return rc;
  if (!copy_strides(stride, p.sq)) return MI355_EINVAL;
  if (!attn_stride_ok(p.sq, q, D) || !aligned(k, 16) || !aligned(v, 16) || !aligned(d_o, 16) ||
      !aligned(dq, 16) || !aligned(dk, 16) || !aligned(dv, 16) || !aligned(Mlse, 16) || !aligned(delta, 16))
    return MI355_ESTRIDE;
  p.q = (const char*)q; p.k = (const char*)k; p.v = (const char*)v; p.d_o = (const char*)d_o;
  if (o && !aligned(o, 16)) return MI355_ESTRIDE;
  p.o = (char*)const_cast<void*>(o); p.lse = const_cast<float*>(Mlse); p.delta = delta;
  p.dq = (char*)dq; p.dk = (char*)dk; p.dv = (char*)dv;
  p.sm_scale = sm_scale; p.causal = causal != 0;
  p.variant = knob(knobs().attn_bwd_groups, attn_bwd_variant(p, p.cus));
  return attn_bwd_launch(p, dtype == MI355_BF16, (hipStream_t)stream_);
}

int mi355_attn_bwd(const void* q, const void* k, const void* v, const void* d_o,
                   const float* Mlse, const float* delta, void* dq, void* dk, void* dv,
                   int Z, int H, int N_CTX, int D, const int64_t* stride,
                   float sm_scale, int causal, int dtype, void* stream) {
  return attn_bwd(q, k, v, nullptr, d_o, Mlse, delta, dq, dk, dv, Z, H, N_CTX, D, stride, sm_scale, causal, dtype, stream);
}

int mi355_attn_bwd_o(const void* q, const void* k, const void* v, const void* o, const void* d_o,
                     const float* Mlse, float* delta, void* dq, void* dk, void* dv,
                     int Z, int H, int N_CTX, int D, const int64_t* stride,
                     float sm_scale, int causal, int dtype, void* stream) {
  if (!o) return MI355_EINVAL;
  return attn_bwd(q, k, v, o, d_o, Mlse, delta, dq, dk, dv, Z, H, N_CTX, D, stride, sm_scale, causal, dtype, stream);
}

}  // extern "C"
