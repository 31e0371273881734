// Host-side launch of the contraction kernels; one translation unit per element type.
#pragma once

#include <atomic>

#include "../../include/rzlinear.h"
#include "rz_common.h"

namespace rz {

// Every planning function takes the caller's tuning overrides (all zero = automatic); nothing
// here reads the environment or keeps state, so a workspace query and the launch that follows
// it decide alike.
static inline rz_tuning tuning_or_default(const rz_tuning* t) {
  rz_tuning d = {};
  return t != nullptr ? *t : d;
}
static inline bool tuning_valid(const rz_tuning& t) {
  return (t.tile == 0 || t.tile == 32 || t.tile == 64 || t.tile == 128 || t.tile == 256) && (t.stages == 0 || t.stages == 1) &&
         (t.lds_image == 0 || t.lds_image == -1) && (t.window >= -1 && t.window <= 1) &&
         (t.split >= -1 && t.split <= 16) && (t.clamp == 0 || t.clamp == -1) &&
         (t.fold >= -1 && t.fold <= 2) && (t.fold_tiles == 0 || t.fold_tiles == -1) && (t.finish == 0 || t.finish == -1) && t.poll_limit >= 0;
}

// Kernels that use more than the default 64 KB of LDS need their limit raised once per kernel
// and device; `done` is that kernel's bit set of devices already served.
static inline hipError_t raise_lds_limit(const void* kernel, std::atomic<uint64_t>& done) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = 1ull << (dev & 63);
  if (done.load(std::memory_order_acquire) & bit) return hipSuccess;
  e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  if (e == hipSuccess) done.fetch_or(bit, std::memory_order_release);
  return e;
}

static constexpr int kComputeUnits = 256;
// Number of workgroups of the small tile that fills the compute units a few times over.
static constexpr int kTargetWorkgroups = 1024;

// Contracted elements per kernel step that every slice of a cut contraction must be a multiple
// of: 128 bytes, and 256 for the 16-bit 64 tile, whose sixteen wavefronts take 256-byte steps (a slice that began
// in the middle of such a step would start between two hashed tiles), and for the 16-bit 128 tile, whose plans the 32 x 128
// tile with its 256-byte steps may carry out.
static inline int slice_unit(int tile, int elem_bytes, bool weight_grad = false) {
  if (elem_bytes == 4 && tile <= 64 && !weight_grad) return 64;   // (fp32 forward / input-grad, 64 and 32 x 64 tiles: 256-byte steps as well)
  return ((tile <= 128 && elem_bytes == 2) ? 256 : 128) / elem_bytes;
}

// Tile codes: 64, 128, 256 are square C tiles; 32 stands for the 32 x 64 tile of the fp32 forward /
// input-grad kernels, for batches whose rows would leave the last 64-row tile at most half full
// (M = 32, 96, 160: that half would be padding).
static inline int tile_cols(int t) { return t == 32 ? 64 : t; }
static inline long long tile_count(int I, int J, int t) {
  return (long long)((I + t - 1) / t) * ((J + tile_cols(t) - 1) / tile_cols(t));
}

// Rate of `wgs` equal workgroups on the chip relative to a full one, when a compute unit runs at
// `lo` with one workgroup resident and at `hi` with `slots` (linear in between).  The hardware
// deals workgroups out evenly, so the busiest compute unit holds c = ceil(wgs / CUs) of them; up to
// `slots` they run side by side and finish together after c * w / e(c), while the chip's work is
// wgs * w: the rate is (wgs / CUs) * e(c) / c.  (320 workgroups on 256 compute units leave 64 of
// them with two: the launch takes as long as 512 would.)  Beyond `slots` per compute unit the
// workgroups go in rounds of CUs * slots and a last, partly filled round costs a full one.
static inline double occupancy_rate(double wgs, int slots, double lo, double hi, int knee = 0) {
  const double per_cu = wgs / kComputeUnits;
  if (per_cu <= 1.0) return lo * per_cu;
  // (`knee`: the number of resident workgroups from which the compute unit runs at `hi`, if fewer than `slots`)
  const double full = knee > 1 ? knee : slots;
  auto e = [&](double c) { return full > 1 ? lo + (hi - lo) * (c < full ? (c - 1.0) / (full - 1.0) : 1.0) : hi; };
  if (per_cu <= slots) {
    const double c = (double)((long long)(per_cu + 0.999999));
    return per_cu * e(c) / c;
  }
  const double cap = (double)kComputeUnits * slots;
  const double rounds = (double)((long long)((wgs + cap - 1) / cap));
  return hi * wgs / (rounds * cap);
}

// Relative throughput of a tile shape at a given number of workgroups, from measurements on
// MI355X (256 tile at one workgroup per compute unit = 1).  16-bit types: the 128 tile reaches
// 0.51 with one workgroup per compute unit and 0.75 with two or more, the 64 tile 0.16 and 0.33
// (four or more).  fp32 is bound by the slower fp32 MFMA rate, so the small tiles lose far less:
// 0.86 / 0.90 and 0.45 / 0.80.  How the number of workgroups enters: occupancy_rate above.
static inline double tile_score_full(int I, int J, int t, int elem_bytes) {
  const double wgs = (double)tile_count(I, J, t);
  const bool f32 = elem_bytes == 4;
  const int slots = (t == 256) ? 1 : (t == 128 ? 2 : 4);          // resident workgroups per CU
  const double lo = (t == 256) ? 1.0 : (t == 128 ? (f32 ? 0.86 : 0.51) : (f32 ? 0.45 : 0.16));  // one workgroup per CU
  const double hi = (t == 256) ? 1.0 : (t == 128 ? (f32 ? 0.90 : 0.75) : (f32 ? 0.80 : 0.33));  // `slots` per CU
  return occupancy_rate(wgs, slots, lo, hi);
}
// ... times the share of a tile grid's MFMA work that is not padding
static inline double tile_score(int I, int J, int t, int elem_bytes) {
  const double wgs = (double)tile_count(I, J, t);
  return tile_score_full(I, J, t, elem_bytes) * ((double)I * (double)J) / (wgs * t * t);
}

// Relative throughput of `wgs` workgroups of tile t (see tile_score_full, which this restates for
// a workgroup count that includes the slices of a cut contraction).
// (store_op: the figures of forward / input-grad as they are now — fp32 staged directly, 16-bit fitted
//  again with them; weight-grad keeps its own)
static inline double tile_rate(double wgs, int t, int elem_bytes, double lo64_f32 = 0.60, bool store_op = false) {
  const bool f32 = elem_bytes == 4;
  if (f32 && store_op) {
    // fp32 forward / input-grad, staged directly: every tile runs the MFMA pipe at the 256 tile's rate
    // once its loop is under way, at one workgroup per compute unit already (eight wavefronts); what a
    // smaller tile costs is the longer fill and drain per workgroup, which plan_split prices per slice.
    // (the 32 x 64 tile, four wavefronts, needs a second workgroup on the compute unit for that: 0.7 alone —
    //  M = 8, K = N = 8192: 256 workgroups 51 us, 512 45 us; M = 16, K = 4096, N = 11008: 172 workgroups 46 us,
    //  688 34 us)
    if (t == 32) return occupancy_rate(wgs, 4, 0.7, 1.0, 2);
    // (the 64 tile alone on a compute unit: 0.85 — M = 96, K = N = 4096 in two slices, 256 workgroups: 48 us)
    return occupancy_rate(wgs, t == 256 ? 1 : 2, t == 64 ? 0.85 : 1.0, 1.0);
  }
  // (32 x 64, four wavefronts: half a 64 workgroup's work in about its time, up to eight resident)
  if (t == 32) return occupancy_rate(wgs, 8, 0.40, 0.80);
  // (the 16-bit 128 tile in its eight-wavefront form — up to one and a half workgroups per compute unit, see
  //  kernel_form — has a compute unit to itself and runs at 0.80 there; beyond one per compute unit that
  //  means a second round: K = N = 10240, M = 128: 80 tiles whole 92 us, in two slices 55, three 43, four 62)
  if (!f32 && store_op && t == 128 && wgs <= kComputeUnits * 3 / 2) return occupancy_rate(wgs, 1, 0.80, 0.80);
  const int slots = (t == 256) ? 1 : (t == 128 ? 2 : 4);
  // (the 16-bit 64 tile: 0.29 with one workgroup per compute unit, 0.40 from two on — K = N = 10240, M = 128:
  //  320 workgroups 93 us, 640 68 us; M = 512, K = 4096, N = 1024 in four slices 16 us)
  const double lo = (t == 256) ? 1.0 : (t == 128 ? (f32 ? 0.86 : 0.51) : (f32 ? lo64_f32 : (store_op ? 0.29 : 0.24)));
  const double hi = (t == 256) ? 1.0 : (t == 128 ? (f32 ? 0.90 : 0.75) : (f32 ? 0.80 : (store_op ? 0.40 : 0.33)));
  return occupancy_rate(wgs, slots, lo, hi, (t == 64 && !f32) ? 2 : 0);
}

// C-tile edge for a contraction with an I x J result: the best-scoring of 256, 128, 64.
static inline int pick_tile(int I, int J, int elem_bytes, const rz_tuning& tuning) {
  if (tuning.tile) return (tuning.tile == 32 && elem_bytes != 4) ? 64 : tuning.tile;
  int best = 256;
  double best_score = tile_score(I, J, 256, elem_bytes);
  const int others[2] = {128, 64};
  for (int t : others) {
    const double sc = tile_score(I, J, t, elem_bytes);
    if (sc > best_score * 1.02) {   // prefer the larger tile on a near tie
      best = t;
      best_score = sc;
    }
  }
  return best;
}

// Weight-grad without any scatter in the contraction kernel: X^T.dY is stored tile by tile and a
// second kernel, whose workgroups own windows of hashed_weight, folds the tiles into dHW.
// (the fold kernel reads a kilobyte per wavefront from any 4-byte boundary: up to 1032 bytes before and after the tiles)
static constexpr size_t kFoldMarginBytes = 2048;

struct FoldPlan {
  int use;
  int small;             // few tiles: the kernel whose workgroups each look at every tile (no windows in LDS, no shares)
  int window, windows;   // floats per window (a multiple of 1024, at most 32768) and their number
  int shares;            // workgroups per window, each with an equal part of the window's tiles and an image of its own
  int tile_bytes;        // bytes of a stored element of X^T.dY: 4, or 2 (the layer's 16-bit dtype, see fold_tile_bytes)
  size_t tiles_bytes;    // the tile-by-tile X^T.dY: slices * tiles * BK*BN elements, with a margin before and after
  size_t partial_bytes;  // shares images of dHW (none with a single share: the fold kernel writes dHW)
  size_t offsets_bytes;  // where every tile starts in hashed_weight, one int32 per tile
};

// What the contraction kernel stores the tiles of X^T.dY as for the fold: floats — or, when the layer
// and its dHW are both 16-bit, the layer's dtype: the sum over M is complete (fp32) by then and the
// fold adds the stored values up in fp32 again, so this costs one more rounding per stored value (the
// reference rounds the running sum at every atomic add, RzLinearBackward.py:364-371) and halves the
// bytes written and read back, which is what the fold costs.
static inline int fold_tile_bytes(int elem_bytes, bool dhw_f32, const rz_tuning& t) {
  return (elem_bytes == 2 && !dhw_f32 && t.fold_tiles != -1) ? 2 : 4;
}

// The windows of hashed_weight that the fold kernel's workgroups own (a function of H alone: a layer
// plan lists every window's tiles).
static inline void fold_geometry(int H, int* window, int* windows) {
  const int kWindowMax = 32768, kThreads = 1024;
  int n = (int)(((long long)H + kWindowMax - 1) / kWindowMax);
  // from half a window per compute unit on, the windows are cut so that whole rounds of workgroups
  // come out, and every workgroup writes its window of dHW itself (no shares, no images)
  if (n * 2 >= kComputeUnits) n = (n + kComputeUnits - 1) / kComputeUnits * kComputeUnits;
  *window = (int)(((((long long)H + n - 1) / n) + kThreads - 1) / kThreads * kThreads);
  *windows = (int)(((long long)H + *window - 1) / *window);
}

static inline FoldPlan plan_fold(int K, int N, int H, int BK, int BN, int slices, bool windowed = false, int tile_bytes = 4) {
  FoldPlan f = {};
  f.tile_bytes = tile_bytes;
  const long long E = (long long)BK * BN;
  const long long tiles = (long long)((K + BK - 1) / BK) * ((N + BN - 1) / BN);
  // (element indices of the buffer are 32-bit in the kernels; the fold lists slices entries per tile)
  if (E > 16384 || slices > 64 || (long long)slices * tiles * E >= (1LL << 31)) return f;
  // (few tiles over a hashed_weight of up to 2^18 elements: measured 5 to 8 us; with a larger one every
  //  workgroup would still look at every tile for the handful that reach it, and the windowed kernel or
  //  the window kernel do better — K = 2048, N = 4096, H = 2^20: 20 us against the window kernel's 25 in all)
  if (tiles <= 4096 && H <= (1 << 18) && !windowed) {
    // every workgroup of 256 threads owns 256 elements of dHW
    f.small = 1;
    f.window = 256;
    f.windows = (H + f.window - 1) / f.window;
    f.shares = 1;
    f.tiles_bytes = (((size_t)slices * tiles * E * (size_t)tile_bytes + 255) & ~(size_t)255) + 2 * kFoldMarginBytes;
    f.partial_bytes = 0;
    f.offsets_bytes = ((size_t)tiles * sizeof(int32_t) + 255) & ~(size_t)255;
    f.use = 1;
    return f;
  }
  fold_geometry(H, &f.window, &f.windows);
  // (a workgroup fills a compute unit: no more workgroups than compute units, or two would wait for a second round)
  long long shares = f.windows * 2 >= kComputeUnits ? 1 : kComputeUnits / f.windows;
  if (shares > slices * tiles / 8) shares = slices * tiles / 8;   // a share is worth a workgroup from some tiles on
  if (shares < 1) shares = 1;
  f.shares = (int)shares;
  f.tiles_bytes = (((size_t)slices * tiles * E * (size_t)tile_bytes + 255) & ~(size_t)255) + 2 * kFoldMarginBytes;
  const size_t pitch = (size_t)((H + 3) & ~3);
  f.partial_bytes = f.shares > 1 ? ((size_t)f.shares * pitch * sizeof(float) + 255) & ~(size_t)255 : 0;
  f.offsets_bytes = ((size_t)tiles * sizeof(int32_t) + 255) & ~(size_t)255;
  f.use = 1;
  return f;
}

// How the weight-grad contraction C[K,N] = X^T.dY over M is cut into workgroups, and how the
// finished tiles reach dHW.
struct WeightGradPlan {
  int tile;          // C tile edge (128 or 256)
  int splits;        // slices of the reduction over M (blockIdx.y)
  int r_chunk;       // rows of M per slice, a multiple of the R step
  long long workgroups;
  int image_pitch;   // > 0: every workgroup first sums its tiles into an fp32 image of dHW held
                     // in LDS and stores it as one partial image; a second kernel adds the
                     // partial images up.  0: tiles go to dHW by global atomics.
  FoldPlan fold;        // fold.use: no scatter in the contraction kernel at all (tile-by-tile output)
  double fold_us;       // ... and roughly how long the whole weight-grad then takes, in microseconds
  size_t workspace_bytes;   // partial images, or the fp32 image for the atomics (16-bit dHW)
  // bias gradient computed in the same pass: partial column sums of dY, one row per
  // (slice, tile row), stored behind the first `workspace_bytes` of the workspace
  int colsum_rows, colsum_pitch;
  size_t colsum_bytes;
  bool lds_image() const { return image_pitch > 0; }
};

// LDS bytes of a compute unit that an fp32 image of dHW may take (the rest holds the small
// offset table of the scatter); the image reuses the operand stages, which are dead by then.
static constexpr size_t kMaxImageBytes = 147456;

static inline long long tile_cover(int K, int N, int t) {
  return (long long)((K + t - 1) / t) * ((N + t - 1) / t) * t * t;
}

// Slices of M for the 128 and 256 tiles with LDS images: as many as fill the compute units once.  A
// few workgroups beyond one per compute unit would make a second round that costs as much as the
// first (300 workgroups take as long as 512), so the count stays at or below the compute units
// (K = N = 2560, M = 2048 bf16: 3 slices x 100 tiles 57.9 us, 2 slices 46.8 us).
static inline long long image_slices(long long tiles, long long r_steps) {
  long long want = (kComputeUnits + tiles - 1) / tiles;
  if (want > 1 && tiles * want > kComputeUnits) want--;
  if (want > r_steps) want = r_steps;
  return want < 1 ? 1 : want;
}

// How well C tiles fill their rounds of workgroups, relative to an ideal distribution.  256 tiles
// go one to a compute unit in rounds of that many.  128 tiles go two to a compute unit; the
// busiest compute unit gets c = ceil(tiles / CUs) of them and works through them in pairs, a
// last odd one alone in about half the time of a pair.
static inline double filled_256(long long tiles) {
  return (double)tiles / (double)((tiles + kComputeUnits - 1) / kComputeUnits * kComputeUnits);
}
static inline double filled_128(long long tiles) {
  const long long c = (tiles + kComputeUnits - 1) / kComputeUnits;
  return ((double)tiles / (2.0 * kComputeUnits)) / ((double)(c / 2) + (c % 2 ? 0.52 : 0.0));
}
// fp32: the 128 tile in pairs runs at this fraction of the 256 tile's rate (weight-grad, measured:
// 4096^2 1067 against 1012 us in one round each; K = N = 5120, M = 4096: 1831 against 2000 us,
// 1600 tiles in seven half-rounds against 400 in two rounds)
static constexpr double kPairRate128F32 = 0.955;

// 16-bit forward / input-grad of more than 64 rows: roughly how long the contraction kernel takes, in microseconds, with C tiles
// of rows x cols over `slices` slices of `steps` steps of 64.  A round of workgroups takes its steps and a fixed part (fill,
// store of C); the 256-row tiles' steps take longer the fuller the chip is, because the board lowers its clock.  Fitted to
// 2790 measurements (forward and input-grad of 84 shapes of 40 to 16384 rows and 256 to 12000 columns, aligned and odd, every
// tile and one to eight slices): on those the plan taken with it was 1.5 % from the best form on average, that of the
// rate model before it, which knew neither the 256 x 128 tile nor the present 256 tile, 6.9 %; small calls: see plan_split.
static inline double store16_us(int rows, int cols, int I, int J, int slices, double steps) {
  const double wgs = (double)(((I + rows - 1) / rows) * (long long)((J + cols - 1) / cols)) * slices;
  auto rounds_of = [&](double per) { return (double)((long long)((wgs + per - 1) / per)); };
  const double rounds = rounds_of(kComputeUnits), fill = wgs / (rounds * kComputeUnits);
  const double launch = 2.8;
  if (rows == 256 && cols == 256) return launch + rounds * (steps * 0.973 * (1.0 + 0.394 * fill) + 11.4);
  if (rows == 256) return launch + rounds * (steps * 0.55 * (1.0 + 0.41 * fill) + 6.5);
  if (rows == 128) {
    const double one = steps * 0.474 + 4.5, two = steps * 1.079 + 3.8;   // a compute unit's one workgroup of eight wavefronts; two of four
    if (wgs <= kComputeUnits * 3 / 2) return launch + rounds * one;
    const double full = (double)((long long)(wgs / (2 * kComputeUnits))), rest = wgs - full * 2 * kComputeUnits;
    return launch + full * two + (rest <= 0.0 ? 0.0 : rest > kComputeUnits ? two : one * 1.217);
  }
  return launch + (wgs <= kComputeUnits ? steps * 0.214 + 2.3 : rounds_of(2 * kComputeUnits) * (steps * 0.441 + 2.3));
}

// The contraction kernel of a 16-bit weight-grad, in microseconds.  The 128 tile's loop loads both operands across the rows
// of its tile: 1.15 times its forward's with one workgroup on a compute unit, 0.88 with two and whole 16-byte pieces.
static inline double weight_grad16_us(int tile, int M, int K, int N, int slices) {
  const double steps = (double)((M + 63) / 64 + slices - 1) / slices;
  if (tile != 128) return store16_us(tile, tile, K, N, slices, steps);
  const bool one = tile_count(K, N, 128) * slices <= kComputeUnits * 3 / 2, whole = K % 8 == 0 && N % 8 == 0;
  return store16_us(128, 128, K, N, slices, steps * (one ? 1.15 : whole ? 0.88 : 1.0));
}

// ... and what its tiles cost beyond it, stored for the fold kernel and read back.
static inline double stored_tiles_us(int tile, int M, int K, int N, int slices, int tile_bytes) {
  return weight_grad16_us(tile, M, K, N, slices) + (double)slices * K * N * tile_bytes * (1.0 / 4.7e6 + 0.3 / 5.0e6);
}

// A 16-bit weight-grad through LDS images, in microseconds, its reduction included: `wgs` workgroups of `steps` steps of 64.  A round
// takes its steps (odd rows longer) and a fixed part of fill, image rounds (by hashed tiles of the C tile) and store; every workgroup
// writes an image that is read once.  Two workgroups of the 128 tile share a compute unit where two images fit its LDS.  Fitted to
// 752 shapes with either tile (M of 64 to 20000, K, N of 200 to 9000, H of 4200 to 36000, aligned and odd): 6 % rms.
static inline double image16_us(int tile, long long wgs, long long steps, int pitch, int K, int N, int BK, int BN) {
  const double bytes = (double)pitch * 4.0, hashed = (double)((tile + BK - 1) / BK) * ((tile + BN - 1) / BN);
  const double rounds = (double)((wgs + kComputeUnits - 1) / kComputeUnits);
  const bool odd = K % 8 != 0 || N % 8 != 0;
  const double both = 8.58 + 0.78 * (double)wgs * bytes * 2.0 / 5e6;
  if (tile == 256) {
    const double fill = (double)wgs / (rounds * kComputeUnits);
    return both + rounds * ((double)steps * 0.764 * (1.0 + 0.824 * fill) * (odd ? 1.036 : 1.0) + 7.17 + 0.236 * hashed);
  }
  const double n = (double)steps * (odd ? 1.197 : 1.0);
  const double one = n * 0.461 + 2.77 + 0.252 * hashed, two = n * 0.896 + 3.17 + 0.087 * hashed;
  if (wgs <= kComputeUnits * 3 / 2) return both + rounds * one;
  if (bytes > 78 * 1024) return both + rounds * (n * 0.627 + 2.77 + 0.132 * hashed);
  const long long full = wgs / (2 * kComputeUnits), rest = wgs - full * 2 * kComputeUnits;
  return both + (double)full * two + (rest == 0 ? 0.0 : rest > kComputeUnits ? two : one * 1.08);
}

// A plan for the fold that was chosen as a whole (see plan_weight_grad).
struct FoldChoice {
  int tile, slices, tile_bytes;
};

static inline WeightGradPlan plan_weight_grad_by_rate(int M, int K, int N, int H, int BK, int BN, int elem_bytes,
                                                      const rz_tuning& t, int tile_bytes, size_t limit, const FoldChoice* chosen = nullptr) {
  WeightGradPlan pl;
  const int pitch = (H + 3) & ~3;
  const bool image = t.lds_image != -1 && (size_t)pitch * sizeof(float) <= kMaxImageBytes;
  // The tile that the comparison with the window kernel prices, where it is not the one that runs: the window kernel adds in
  // fp32, so tiles that are stored in 16 bits are not to take a call from it because they have become cheaper.
  int priced_tile = 0;
  if (chosen != nullptr) {
    pl.tile = chosen->tile;
    tile_bytes = chosen->tile_bytes;
  } else if (t.tile) {
    pl.tile = t.tile == 32 ? 64 : t.tile;   // (the 32 x 64 tile serves forward / input-grad only)
  } else if (image) {
    // with the LDS image the M loop can be cut freely (a slice costs one partial image), so
    // the pipelined 256 tile is used unless it would mostly compute padding
    pl.tile = 64;
    if (tile_cover(K, N, 128) * 10 <= tile_cover(K, N, 64) * 13) pl.tile = 128;
    if (tile_cover(K, N, 256) * 10 <= tile_cover(K, N, pl.tile) * 13) pl.tile = 256;
    // a short M cut over many slices leaves a 256 workgroup a few steps between its prologue
    // and its scatter: the 128 tile then has less to set up and to scatter per workgroup
    // (fp32, M = 2048, K = N = 1024: 53.0 -> 47.5 us; M = 512, K = N = 2048: 51.8 -> 48.4 us; 2048^3 and
    //  M = 16384, K = 512, N = 1024 stay with the 256 tile: 135.8 against 138.8 us, 137 either way)
    const long long tiles256 = tile_count(K, N, 256);
    const int step256 = slice_unit(256, elem_bytes, true);
    const bool cover128 = tile_cover(K, N, 128) * 10 <= tile_cover(K, N, 256) * 13;
    if (pl.tile == 256 && elem_bytes == 4 && tiles256 < kComputeUnits &&
        (long long)((M + step256 - 1) / step256) * tiles256 < 16LL * kComputeUnits && cover128)
      pl.tile = 128;
    // (two 128 workgroups fit a compute unit only while two images fit its LDS: K = N = 10240, M = 2048,
    //  H = 36000: 3849 us against 3583 us with the 256 tile)
    if (pl.tile == 256 && elem_bytes == 4 && cover128 && tiles256 >= kComputeUnits && (size_t)pitch * sizeof(float) <= 78 * 1024) {
      // fp32, at least as many 256 tiles as compute units: the two tiles by how they fill their
      // rounds (K = N = 10240 is six rounds and a quarter of the one, twelve and a half pairs of
      // the other: M = 2048 3520 -> 3317 us, M = 4096 6972 -> 6486 us; K = N = 6000, M = 1024:
      // 848 -> 698 us); the image stores of paired workgroups are half hidden behind each other
      const long long tiles128 = tile_count(K, N, 128);
      const double work_us = 2.0 * (double)M * K * N / 137e6, image_us = (double)pitch * 8.0 / 5e6;
      const double t256 = work_us / filled_256(tiles256) + (double)tiles256 * image_us;
      const double t128 = work_us / (kPairRate128F32 * filled_128(tiles128)) + 0.5 * (double)tiles128 * image_us;
      if (t128 < t256 * 0.99) pl.tile = 128;
    }
    if (pl.tile == 256 && elem_bytes == 2 && cover128) {
      // 16-bit: the two tiles by estimated time.  Fitted on MI355X (weight-grad, 256 workgroups):
      // a 256 workgroup pays about 5.5 steps of 64 rows for its fill, its image rounds and the
      // store of its image, whatever the length of its loop; the 128 tile in its eight-wavefront
      // form (up to 384 workgroups) runs at 0.82 of the 256 tile's rate and pays about 4 times 128
      // rows.  Both write one image per workgroup.  These are the rates of earlier loops of both tiles: the rule
      // decides where the fitted times below see no clear difference.  (2048^3: 32.4 -> 30.5 us;
      // M = 8192, K = N = 2048 stays with the 256 tile: 72.8 against 82.1 us.)
      const long long tiles128 = tile_count(K, N, 128);
      const long long s256 = image_slices(tiles256, (M + 63) / 64), s128 = image_slices(tiles128, (M + 127) / 128);
      const long long w256 = tiles256 * s256, w128 = tiles128 * s128;
      if (w128 <= kComputeUnits * 3 / 2) {
        auto filled = [](long long w, long long cap) { return (double)w / (double)((w + cap - 1) / cap * cap); };
        const double st256 = (double)(((M + 63) / 64 + s256 - 1) / s256), st128 = (double)(((M + 127) / 128 + s128 - 1) / s128);
        const double work_us = 2.0 * (double)M * K * N / 1200e6;
        const double image_us = (double)pitch * 8.0 / 5e6;   // written once, read once
        const double t256 = work_us * (st256 + 5.5) / st256 / filled(w256, kComputeUnits) + (double)w256 * image_us;
        const double t128 = work_us * (st128 + 4.0) / st128 / (0.82 * filled(w128, kComputeUnits)) + (double)w128 * image_us;
        if (t128 < t256 * 0.97) pl.tile = 128;
      }
      // ... and the other one where the fitted times, which know two 128 workgroups on a compute unit and what a hashed tile costs in the
      // image rounds, promise more than the fit's usual error.  (bf16: M = 3200, K = 1536, N = 1152 35.4 -> 24.8 us with the 128
      // tile, 96 x 9344 x 3712 77.6 -> 52.0)  They were fitted from 64 rows on: with fewer a call is little but its images, and
      // what those of the 128 tile have more costs 0.22 us a MB from 8 MB on (M = 36, K = 1863, N = 1524, H = 33541: 24 MB of images
      // instead of 6 25.5 against 24.2 us).  Of 4000 drawn shapes of 4 to 32768 rows with a tile of either size 666 change theirs, 1.29 times as
      // fast in the mean; six are more than 2 % slower, the least 0.89 (M = 21162, K = 1152, N = 448).
      const double us256 = image16_us(256, w256, ((M + 63) / 64 + s256 - 1) / s256, pitch, K, N, BK, BN);
      double us128 = image16_us(128, w128, 2 * (((M + 127) / 128 + s128 - 1) / s128), pitch, K, N, BK, BN);
      const double more_mb = (double)(w128 - w256) * pitch * sizeof(float) * 1e-6;
      if (M <= 64 && w128 <= 2 * kComputeUnits && more_mb > 8.0) us128 += 0.22 * (more_mb - 8.0);
      const int by_rate = pl.tile, other = 384 - by_rate;
      const size_t other_bytes = (size_t)(other == 128 ? w128 : w256) * pitch * sizeof(float);
      if ((other == 128 ? us128 : us256) < 0.92 * (other == 128 ? us256 : us128) && other_bytes <= limit) pl.tile = other;
    }
  } else {
    pl.tile = pick_tile(K, N, elem_bytes, t);
    // 16-bit with a short M: a workgroup of the 256 tile is then mostly fill and store, which two workgroups of the 128 tile
    // on a compute unit hide behind each other — from two rounds of 256 tiles on (M = 64: K = N = 6000 78 -> 73 us, K = 12000,
    // N = 9000 140 -> 135; K = 8192, N = 4096, two rounds exactly, 65 either way; M = 512: 104 / 100 and 205 / 214 us)
    if (pl.tile == 256 && elem_bytes == 2 && t.fold != -1 && M <= 256 && tile_count(K, N, 256) > 2 * kComputeUnits) {
      const FoldPlan f = plan_fold(K, N, H, BK, BN, 1);
      if (f.use && !f.small) {
        pl.tile = 128;
        if (tile_bytes == 2) priced_tile = 256;
      }
    }
    // fp32 with the tiles stored for the fold kernel: by how the two tiles fill their rounds when
    // there are at least as many 256 tiles as compute units (K = N = 10240: M = 128 455 -> 401 us,
    // M = 1024 1938 -> 1797 us, M = 4096 7002 -> 6449 us; K = N = 4096, one round exactly, stays
    // with the 256 tile: 1043 against 1085 us); with fewer, a short M takes the 128 tile, whose
    // paired workgroups hide each other's stores
    if (pl.tile == 256 && elem_bytes == 4 && t.fold != -1 && plan_fold(K, N, H, BK, BN, 1).use) {
      const long long t256 = tile_count(K, N, 256), t128 = tile_count(K, N, 128);
      if (t256 >= kComputeUnits ? kPairRate128F32 * filled_128(t128) > filled_256(t256) * 1.01 : M <= 2048) pl.tile = 128;
    }
  }
  const long long tiles = (long long)((K + pl.tile - 1) / pl.tile) * ((N + pl.tile - 1) / pl.tile);
  const int TR = slice_unit(pl.tile, elem_bytes, true);
  const int r_steps = (M + TR - 1) / TR;
  // split the reduction over M when there are too few W tiles to fill the chip
  // (one workgroup per compute unit for the 128 tile too: a second one per compute unit would come
  //  with twice the partial images to write and to add up — 1024^3: bf16 22.3 -> 20.4 us, fp32 37.0 -> 33.9 us)
  const long long target = (pl.tile >= 128) ? kComputeUnits : kTargetWorkgroups;
  long long want = (target + tiles - 1) / tiles;
  if (want > r_steps) want = r_steps;
  if (want < 1) want = 1;
  if (image && pl.tile >= 128) want = image_slices(tiles, r_steps);
  if (chosen != nullptr) {
    want = chosen->slices;
  } else if (!image) {
    // every slice repeats the K*N adds of the scatter (global atomics, about 5.4 ps each, some 70 %
    // of which the contraction does not hide): the number of slices with the least estimated time
    if (want > 8) want = 8;
    const double peak = elem_bytes == 4 ? 137e6 : 1150e6;   // flop per microsecond of the 256 tile on a full chip
    double best_us = 0.0;
    long long best = 1;
    for (long long w = 1; w <= want; w++) {
      const long long per = (r_steps + w - 1) / w;
      if ((r_steps + per - 1) / per != w) continue;
      const double steps = (double)per * (TR * elem_bytes / 128);
      const double us = 2.0 * (double)M * K * N / (peak * tile_rate((double)tiles * w, pl.tile, elem_bytes) * steps / (steps + 2.0)) +
                        (double)w * K * N * 3.8e-6;
      if (best_us == 0.0 || us < best_us * 0.97) {
        best_us = us;
        best = w;
      }
    }
    want = best;
  }
  const int steps_per = (int)((r_steps + want - 1) / want);
  pl.splits = (r_steps + steps_per - 1) / steps_per;
  pl.r_chunk = steps_per * TR;
  pl.workgroups = tiles * pl.splits;
  pl.image_pitch = image ? pitch : 0;
  pl.fold = FoldPlan{};
  pl.fold_us = 0.0;
  if (!image && t.fold != -1) {
    const FoldPlan f = plan_fold(K, N, H, BK, BN, pl.splits, t.fold == 2, tile_bytes);
    if (f.use) {
      // what the two ways cost beyond the contraction itself, in microseconds: the part of the
      // K*N global atomics per slice that the contraction does not hide (2.8 to 5.2 ps each,
      // measured), against reading the tiles back (their stores overlap the contraction, unless
      // it is shorter than they are), writing and reading the images, and two more launches
      const double elems = (double)pl.splits * (double)K * (double)N;
      // (fp32, K = N = 10240: the contraction takes 427 us at M = 256, 805 us at M = 512)
      const double product_us = 2.0 * (double)M * K * N / (elem_bytes == 4 ? 145e6 : 900e6);
      const double store_us = elems * tile_bytes / 4.0e6;
      // (K*N atomics take about 5.2 ps each; a long contraction hides up to 2.4 ps of that — K = 2048,
      //  N = 8192, bf16: M = 128 87 us in all against 57 us folded, M = 1024 108 against 79 us)
      const double hidden = 0.45 * product_us < elems * 2.4e-6 ? 0.45 * product_us : elems * 2.4e-6;
      const double atomics_us = elems * 5.2e-6 - hidden;
      // (a workgroup of the fold kernel reads some 20 GB/s: few workgroups cannot use the memory system; all of
      //  them together 6 TB/s of fp32 tiles — K = N = 10240: 85 us — and 4.7 TB/s of 16-bit ones — 58 us —
      //  where the instructions per load set the pace)
      const double read_bytes = elems * tile_bytes * (1.0 + (double)BK * BN / f.window);
      const double all_us = (read_bytes + 2.0 * (double)f.partial_bytes) / (tile_bytes == 4 ? 6.0e6 : 4.7e6);
      const double one_us = read_bytes / ((double)f.windows * f.shares) / (tile_bytes == 4 ? 24e3 : 19e3);
      // (few tiles: every element is read once, by a kernel of a few microseconds; it is taken even where
      //  the atomics would be a little faster — K = N = 1024: 5 us against 3 us on top of the contraction —
      //  because it adds in a fixed order: the same bits on every call)
      const double fold_us = f.small ? (store_us > product_us ? store_us - product_us : 0.0) + elems * tile_bytes / 4.5e6 + 5.0
                                     : (store_us > product_us ? store_us - product_us : 0.0) + (all_us > one_us ? all_us : one_us) + 10.0;
      if (t.fold >= 1 || f.small || fold_us < atomics_us) {
        pl.fold = f;
        // (for the comparison with the window kernel: every round of workgroups of the contraction
        //  kernel also pays its fill, drain and store — about 5 us for a round of 256 tiles, 10 us
        //  in fp32, in proportion to the tile's area — which matters when M is small)
        const int priced = priced_tile ? priced_tile : pl.tile;
        const long long priced_wgs = priced_tile ? tile_count(K, N, priced_tile) * pl.splits : pl.workgroups;
        const double round_us = (elem_bytes == 4 ? 10.0 : 5.0) * (double)priced * priced / 65536.0;
        // (a contraction shorter than the stores of its tiles takes the time of the stores — fp32, K = N = 10240,
        //  H = 2^20, M = 32: 220 us in all)
        const double contraction_us = product_us + round_us * (double)((priced_wgs + kComputeUnits - 1) / kComputeUnits);
        pl.fold_us = (contraction_us > store_us ? contraction_us : store_us) + fold_us - (store_us > product_us ? store_us - product_us : 0.0);
      }
    }
  }
  size_t ws = 0;
  if (pl.fold.use) ws = pl.fold.tiles_bytes + pl.fold.partial_bytes + pl.fold.offsets_bytes;
  else if (pl.image_pitch > 0) ws = (size_t)pl.workgroups * pl.image_pitch * sizeof(float);
  else if (elem_bytes == 2) ws = (size_t)H * sizeof(float);   // fp32 image for the atomics
  pl.workspace_bytes = (ws + 255) & ~(size_t)255;
  pl.colsum_rows = pl.splits * ((K + pl.tile - 1) / pl.tile);
  pl.colsum_pitch = ((N + pl.tile - 1) / pl.tile) * pl.tile;
  pl.colsum_bytes = (size_t)pl.colsum_rows * pl.colsum_pitch * sizeof(float);
  return pl;
}

// 16-bit with the tiles stored for the fold kernel: tile and slices together, by the fitted times (the rates above cut M no
// further than the atomics' K*N adds per slice allow, and know neither what a workgroup's fill and store cost nor the present
// tiles).  A slice's stored tiles are partial sums: where there are more of them than in the plan by rate they are stored in
// fp32, whatever the layer's dtype, and so are they where that plan adds into an fp32 image.  (bf16, the module's
// call: M = 20442, K = 6647, N = 591 477 -> 221 us; 14592, 8448, 448 232 -> 128; from the atomics 11552, 5632, 768 195 -> 121;
// 368 drawn shapes whose plan changed 1.23 times as fast in the mean, the least 0.985.)
// limit: bytes of scratch memory that images or the fold may take.
static inline WeightGradPlan plan_weight_grad(int M, int K, int N, int H, int BK, int BN, int elem_bytes,
                                              const rz_tuning& t, int tile_bytes = 4, size_t limit = (size_t)-1) {
  const WeightGradPlan by_rate = plan_weight_grad_by_rate(M, K, N, H, BK, BN, elem_bytes, t, tile_bytes, limit);
  if (elem_bytes != 2 || by_rate.image_pitch > 0 || t.tile != 0 || t.fold == -1) return by_rate;
  FoldChoice best = {0, 0, 0};
  // (the plan by rate is left only for one that is faster by more than the fit's error; the 64 tile's times are not fitted for
  //  this; the atomics: the part of K*N per slice that the contraction does not hide)
  // (in place of atomics the fold is a kernel more, 12 us of launch and of looking for tiles that the fitted times leave out, as
  //  they are the same for every fold; with them both prices are within a few per cent of what is measured.  Of 438 drawn
  //  calls of 4 to 32768 rows whose plan by rate adds by atomics 289 leave it, 1.20 times as fast in the mean, the least 0.96; without
  //  the 12 us 343 left it, 40 of them slower, down to 0.88 — M = 1085, K = 4416, N = 1024, H = 282624 46 -> 50 us)
  const double by_rate_us = by_rate.fold.use ? stored_tiles_us(by_rate.tile, M, K, N, by_rate.splits, tile_bytes)
                                             : weight_grad16_us(by_rate.tile, M, K, N, by_rate.splits) + (double)by_rate.splits * K * N * 2.8e-6;
  double best_us = 0.90 * by_rate_us - 1.0;
  if (!by_rate.fold.use && by_rate_us - 12.0 < best_us) best_us = by_rate_us - 12.0;
  const int tiles_of[2] = {256, 128};
  for (int tile : tiles_of) {
    const int unit = slice_unit(tile, elem_bytes, true), steps = (M + unit - 1) / unit;
    for (int w = 1; w <= 8 && w <= steps; w++) {
      const int per = (steps + w - 1) / w;
      const int bytes = by_rate.fold.use && w <= by_rate.splits ? tile_bytes : 4;
      const FoldPlan f = plan_fold(K, N, H, BK, BN, w, t.fold == 2, bytes);
      if ((steps + per - 1) / per != w || !f.use || f.tiles_bytes + f.partial_bytes + f.offsets_bytes > limit) continue;
      const double us = stored_tiles_us(tile, M, K, N, w, bytes);
      if (us < best_us * (best.tile == 0 ? 1.0 : 0.97)) {
        best_us = us;
        best = {tile, w, bytes};
      }
    }
  }
  if (best.tile == 0 || (best.tile == by_rate.tile && best.slices == by_rate.splits)) return by_rate;
  WeightGradPlan pl = plan_weight_grad_by_rate(M, K, N, H, BK, BN, elem_bytes, t, tile_bytes, limit, &best);
  if (!pl.fold.use) return by_rate;
  // (the window kernel adds in fp32: 16-bit tiles take no call from it that the plan by rate leaves to it)
  if (by_rate.fold.use && best.tile_bytes == 2) pl.fold_us = by_rate.fold_us;
  return pl;
}

// Weight-grad by windows of dHW (rz_window.h): used when hashed_weight is too large for one
// LDS image and the contraction over M is short, so that the K*N global atomics of the scatter
// kernel would dominate.
struct WindowPlan {
  bool use;
  int window;    // elements of dHW per workgroup
  int windows;   // workgroups
  long long tiles;   // W tiles (entries of the offset table the kernel scans)
  size_t pack_bytes; // X and dY as fragments (workspace that the call can do without)
};
static constexpr int kWindowFloats = 25600;   // LDS floats a workgroup can hold next to its staging

// Hashed tiles that the window kernel serves: 32 to 256 rows, 32 to 128 columns.  Its unit of work is 32
// rows by min(BN, 64) columns of a tile; a tile has window_units of them, unit u = strip * parts + part
// starting at off + window_unit_start and spanning window_unit_span elements of hashed_weight.
static inline bool window_tile_supported(int BK, int BN) {
  return (BN == 32 || BN == 64 || BN == 128) && (BK == 32 || BK == 64 || BK == 128 || BK == 256);
}
static inline int window_unit_cols(int BN) { return BN < 64 ? BN : 64; }
static inline int window_units(int BK, int BN) { return (BK / 32) * (BN / window_unit_cols(BN)); }
static inline int window_unit_span(int BN) { return 31 * BN + window_unit_cols(BN); }
static inline long long window_unit_start(int BN, int u) {
  const int parts = BN / window_unit_cols(BN);
  return (long long)(u / parts) * (32 * BN) + (long long)(u % parts) * window_unit_cols(BN);
}

// Size and number of the windows for a hashed_weight of H elements (a function of H alone: a
// layer plan built once per layer holds the strip lists of exactly these windows).
static inline void window_geometry(int H, int* window, int* windows) {
  // one workgroup per compute unit when the windows can be that large, else whole rounds
  const long long rounds = ((long long)H + (long long)kWindowFloats * kComputeUnits - 1) /
                           ((long long)kWindowFloats * kComputeUnits);
  long long w = (((long long)H + rounds * kComputeUnits - 1) / (rounds * kComputeUnits) + 3) & ~3LL;
  if (w < 1024) w = 1024;                        // tiny windows would each redo most tiles
  *window = (int)w;
  *windows = (int)(((long long)H + w - 1) / w);
}

// Images of a window that a workgroup keeps in LDS, a power of two up to its sixteen wavefronts.  With a small window nearly every
// unit meets the one before it in the list, and the chain of adds takes most of the time; with images a unit waits for those of
// its own image only (bf16, windows of 4096: M = 16, K = 2048, N = 8192 35.6 -> 20 us, M = 64, K = N = 4096 39.4 -> 24.7;
// windows of 1024: M = 32, K = N = 2048 37 -> 15.5).  A function of the window alone: the packed form, which has no staging area, would have
// room for half as many again, but the order of the sums, and with it the bits of dHW, would then depend on the workspace that the caller has.
static inline int window_images(int window) {
  int n = 1;
  while (n < 16 && 2 * n * window <= kWindowFloats) n *= 2;
  return n;
}

// Bytes of X and dY as fragments (window_pack_kernel): the rows up to whole groups, the columns up to whole hashed tiles.
static inline size_t window_pack_bytes(int M, int K, int N, int BK, int BN, int elem_bytes) {
  const size_t group = elem_bytes == 4 ? 8 : 16, rows = ((size_t)M + group - 1) / group * group;
  return rows * (size_t)elem_bytes * ((size_t)((K + BK - 1) / BK) * BK + (size_t)((N + BN - 1) / BN) * BN);
}

// What the window kernel takes with its operands as fragments (with the kernel that makes them), staged, or element by element:
// microseconds on MI355X, fitted to 770 calls of drawn shapes (1 to 700 rows, 128 to 14000 columns, tiles of 32 x 64 and 64 x 64,
// K * N / H of 16 and 100) in captured graphs; the fits' error is 8 % (element by element in fp32 15 %).  A workgroup works through
// the units that meet its window, each at a fixed price and one per 32 rows of M; in 16 bits the latter grows where X and dY outgrow
// an L2 (4 MB), from which every unit reads its own rows and columns.  The adds into one place of an image go one after the
// other: K * N / H links, of the images' share each.  The greater of the two sets the time; of the smaller one a part still shows.
static inline double window_us(int M, int K, int N, int H, int BK, int BN, int elem_bytes, int window, int windows, bool packed) {
  struct Fit { double fixed, per_mb, unit, rows, misses, link, rest; };
  static const Fit fits[2][3] = {{{10.4, 2.0, 0.160, 0.040, 0.040, 2.3, 0.17}, {10.1, 0.9, 0.171, 0.063, 0.039, 1.8, 0.41}, {12.6, 3.0, 0.219, 0.178, 0.066, 3.1, 0.05}},
                                 {{11.7, 4.7, 0.050, 0.320, 0.0, 3.3, 0.40}, {12.6, 3.4, 0.083, 0.290, 0.0, 1.66, 1.0}, {13.6, 8.2, 0.0, 0.524, 0.0, 1.14, 1.0}}};
  const bool whole = K % (16 / elem_bytes) == 0 && N % (16 / elem_bytes) == 0;
  const Fit& f = fits[elem_bytes == 4][packed ? 0 : whole ? 1 : 2];
  const double tiles = (double)((K + BK - 1) / BK) * (double)((N + BN - 1) / BN);
  const double units = tiles * window_units(BK, BN) * ((double)window + window_unit_span(BN)) / (double)H;
  const double rounds = (double)((windows + kComputeUnits - 1) / kComputeUnits);
  const double chunks = M > 16 ? M / 32.0 : 0.5, mb = (double)M * ((double)K + N) * elem_bytes * 1e-6;
  const double work_us = rounds * units * (f.unit + chunks * (f.rows + (mb > 4.3 ? f.misses * (1.0 - 4.3 / mb) : 0.0)));
  const double chain_us = f.link * (double)K * N / (double)H / window_images(window);
  return f.fixed + f.per_mb * mb + (work_us > chain_us ? work_us + f.rest * chain_us : chain_us + f.rest * work_us);
}

// A second fit of the same times, over what the first one leaves out: 3300 drawn calls of 1 to 4000 rows, 64 to 16384 columns, every hashed tile that
// the kernel serves, K * N / H of 1 to 2000 (of 1500 other such calls nine tenths are within 0.69 to 1.2 of the measured time, half within
// 8 %).  Beside what the first one knows: the busiest window has a few times the square root of the mean number of units more; a unit that
// reaches beyond the window is added with checks; a handful of units leave wavefronts idle; 32-column units are about half the work,
// those of 128-column tiles, which lie further apart, more.
static inline double window_us_any_tile(int M, int K, int N, int H, int BK, int BN, int elem_bytes, int window, int windows, bool packed) {
  struct Fit { double fixed, per_mb, unit, rows, misses, link, rest, beyond, narrow_unit, narrow_rows, per_m, wide, busiest, few; };
  static const Fit fits[2][3] = {
    {{9.27, 0.80, 0.0833, 0.0266, 0.0196, 0.726, 1.25, 0.0317, 0.567, 0.715, 1.04, 0.302, 4.18, 4.33},
     {8.34, 0.0, 0.1107, 0.0454, 0.0332, 1.48, 0.418, 0.0489, 0.469, 0.774, 1.20, 0.150, 3.72, 5.43},
     {8.66, 0.37, 0.1473, 0.1136, 0.0659, 1.17, 0.499, 0.0562, 0.356, 0.723, 1.09, 0.230, 4.29, 10.2}},
    {{9.69, 1.0, 0.1080, 0.2395, 0.0122, 1.72, 0.433, 0.0286, 0.495, 0.528, 1.43, 0.200, 2.87, 2.47},
     {8.75, 0.02, 0.1604, 0.2143, 0.0108, 2.45, 0.258, 0.0317, 0.423, 0.579, 1.52, 0.163, 3.48, 6.69},
     {9.44, 0.0, 0.0768, 0.3956, 0.0370, 2.03, 0.405, 0.0662, 0.382, 0.627, 1.72, 0.147, 3.80, 7.03}}};
  const bool whole = K % (16 / elem_bytes) == 0 && N % (16 / elem_bytes) == 0, narrow = BN == 32;
  const Fit& f = fits[elem_bytes == 4][packed ? 0 : whole ? 1 : 2];
  const double span = window_unit_span(BN), all = (double)((K + BK - 1) / BK) * (double)((N + BN - 1) / BN) * window_units(BK, BN);
  const double meets = ((double)window + span) / (double)H, mean = all * (meets < 1.0 ? meets : 1.0), units = mean + f.busiest * sqrt(mean);
  const double beyond = window > span ? 2.0 * span / (window + span) : 1.0;   // the share of the units that do not lie inside the window
  const int group = elem_bytes == 4 ? 8 : 16;
  const double rounds = (double)((windows + kComputeUnits - 1) / kComputeUnits), chunks = (double)((M + group - 1) / group * group) / 32.0;
  const double mb = (double)M * ((double)K + N) * elem_bytes * 1e-6;
  const double unit = (f.unit + f.beyond * beyond) * (narrow ? f.narrow_unit : 1.0);
  const double rows = (f.rows + (mb > 4.3 ? f.misses * (1.0 - 4.3 / mb) : 0.0)) * (narrow ? f.narrow_rows : 1.0);
  const double work_us = rounds * (units * unit + sqrt(units * units + f.few * f.few) * chunks * rows) * (BN == 128 ? 1.0 + f.wide : 1.0);
  const double chain_us = f.link * (double)K * N / (double)H / window_images(window);
  return f.fixed + f.per_mb * mb + f.per_m * H * 1e-6 + (work_us > chain_us ? work_us + f.rest * chain_us : chain_us + f.rest * work_us);
}

// ... and what the fold (priced by plan_weight_grad, whose prices leave out what all of its plans share) or the atomics take on such calls,
// fitted to the same measurements: nine tenths are within 0.8 to 1.3 (fold) and 0.88 to 1.13 (atomics) of the measured time.
static inline double scatter_us(int M, int K, int N, int H, int elem_bytes, const WeightGradPlan& other) {
  const bool f32 = elem_bytes == 4;
  const double kn = (double)K * N * 1e-6, h = H * 1e-6, mb = (double)M * ((double)K + N) * elem_bytes * 1e-6;
  if (other.fold.use && other.fold.small)
    return f32 ? 3.0 + 1.28 * other.fold_us + 9.8 * h + 0.34 * kn + 0.235 * mb : 8.3 + 0.557 * other.fold_us + 2.23 * h + 1.37 * kn + 0.47 * mb;
  if (other.fold.use) return f32 ? 2.2 + 1.13 * other.fold_us + 1.2 * h + 0.13 * mb : 2.1 + 1.04 * other.fold_us + 0.9 * h + 0.08 * kn;
  const double rounds = (double)((tile_count(K, N, 128) + kComputeUnits - 1) / kComputeUnits), steps = (double)((M + 63) / 64), gmac = kn * M * 1e-3;
  return f32 ? 5.7 + 3.95 * kn + 16.5 * gmac + 1.5 * h + 0.0279 * (kn / h) + rounds * (0.55 + 0.17 * steps)
             : 8.2 + 4.14 * kn + 2.37 * gmac + 2.26 * h + 0.0107 * (kn / h) + rounds * (0.64 + 0.142 * steps);
}

// limit: bytes of workspace that the call may have.  planned: the caller holds a layer plan, so the kernel neither hashes the tile offsets nor scans
// them for its strips (some 25 us less, measured at K = N = 10240).
static inline WindowPlan plan_window(int M, int K, int N, int H, int BK, int BN, int elem_bytes, const rz_tuning& t,
                                     const WeightGradPlan& other, bool planned = false, size_t limit = (size_t)-1) {
  WindowPlan pl = {false, 0, 0, 0, 0};
  if (t.window == -1 || !window_tile_supported(BK, BN)) return pl;
  const long long tiles = (long long)((K + BK - 1) / BK) * ((N + BN - 1) / BN);
  if (tiles > (1 << 20)) return pl;              // every workgroup scans every tile's offset
  pl.tiles = tiles;
  window_geometry(H, &pl.window, &pl.windows);
  // The operands as fragments where that is faster, by more than the launch that it adds costs a host that is the bound (K = N =
  // 10240, H = 6.5 M, bf16: M = 8 55 -> 51 us, 32 59 -> 53, 128 99 -> 77, 256 180 -> 144; fp32: 32 113 -> 105, but 64 169 -> 174 and
  // 128 287 -> 318, where the matrix pipe is the bound and the staged form keeps it busier).
  double t_window = window_us(M, K, N, H, BK, BN, elem_bytes, pl.window, pl.windows, false);
  const size_t pack_bytes = window_pack_bytes(M, K, N, BK, BN, elem_bytes);
  const double packed_us = window_us(M, K, N, H, BK, BN, elem_bytes, pl.window, pl.windows, true);
  if (packed_us + 3.0 < t_window && pack_bytes <= limit && (unsigned long long)pack_bytes <= 0xffffffffULL && (size_t)tiles * sizeof(int32_t) + 512 <= limit - pack_bytes) {
    t_window = packed_us;
    pl.pack_bytes = pack_bytes;
  }
  if (!planned) t_window += 23.0;   // (the offsets hashed, every workgroup's search among them)
  // ... against what the contraction kernel's plan would take: the fold, or the atomic scatter.  Those prices leave out what is the
  // same for all of their plans: measured, on such shapes, the windowed fold takes 1.18 times its price (5 to 95 %: 1.07 to
  // 1.35), the few-tiles fold 1.7 (fp32) to 1.9 times (its longest calls less, hence 1.65), the atomics about 1.8 times.
  const double t_scatter = 0.9 * (double)K * N / 184e3 + 2.0 * M * (double)K * N / 800e6;
  const double t_other = other.fold.use ? other.fold_us * (other.fold.small ? 1.65 : 1.18) : 1.8 * t_scatter;
  // The first fits are good on average but far off for some tiles: by them alone 16-bit 256 x 128 tiles with M = 2258, K = 14448, N = 12316 took 5548 us,
  // by atomics 1069.  So the second ones must agree.  4800 drawn calls, against the window kernel without fragments and images by a rule on rates:
  // by the first fits 84 take more than 10 % longer, the worst 3.6 times, the mean is 0.926; by both 23, 1.65, 0.919; by the second alone
  // 68, 2.4, 0.914, and by it 118 take more than 10 % longer than by the first (by both: 3).
  double t_second = window_us_any_tile(M, K, N, H, BK, BN, elem_bytes, pl.window, pl.windows, pl.pack_bytes > 0);
  if (!planned) t_second += 23.0;
  pl.use = t.window == 1 || (t_window < t_other && t_second < scatter_us(M, K, N, H, elem_bytes, other));
  return pl;
}

// A layer plan: what the weight-grad of one layer needs of its hash and nothing else (it depends on
// K, N, H, the tile and the hash constants, not on M, the element type or the data), computed once
// on the host and kept by the caller in device memory.  int32 words:
//   [0, 16)   header: magic, version, K, N, H, BK, BN, hash_levels, tiles, windows, window,
//             entries, strips per tile, checksum of the hash constants (layer_plan_hash_sum),
//             fold windows, fold window
//   offsets   [tiles]           where every W tile starts in hashed_weight (index tk * tiles_n + tn)
//   start     [windows + 1]     first entry of every window of the window kernel (window_geometry)
//   list      [capacity]        the units of work (tile * units per tile + unit: 32 rows by up to 64 columns of
//                               a tile, see window_units) that meet the window, ascending
//   offs      [capacity]        ... and where each starts in hashed_weight
//   fold_start [fold windows + 1]  first entry of every window of the fold kernel (fold_geometry)
//   fold_list  [fold capacity]     the tiles that meet the window, in the order in which the fold kernel's
//                                  own search numbers them (fold_rank_order)
// The first two lists exist for the tiles the window kernel supports (windows = 0 otherwise).
static constexpr int32_t kLayerPlanMagic = 0x525a4c50, kLayerPlanVersion = 2;
static constexpr int kLayerPlanHeader = 16;
// What a plan's header says of the hash constants that its offsets were computed with (the kernels
// that read a plan compare it with their own call's constants).
__host__ __device__ static inline int32_t layer_plan_hash_sum(const HashParams& h) {
  uint32_t s = 2166136261u;
  const uint32_t v[8] = {h.R0, h.R1, h.R2, h.R3, h.R4, h.R5, h.R7, (uint32_t)h.levels};
  for (int i = 0; i < 8; i++) s = (s ^ v[i]) * 16777619u;
  return (int32_t)(s & 0x7fffffffu);
}
// header words 2..7 and 13 against a call (K, N, H, BK, BN, hash_levels, constants)
__host__ __device__ static inline bool layer_plan_matches(const int32_t* hd, int K, int N, int H, const HashParams& h) {
  return hd[0] == kLayerPlanMagic && hd[2] == K && hd[3] == N && hd[4] == H && hd[5] == h.BK && hd[6] == h.BN &&
         hd[7] == h.levels && hd[13] == layer_plan_hash_sum(h);
}
struct LayerPlanLayout {
  bool ok;
  int tiles, windows, window, strips_per_tile, strip_elems;   // (units per tile, elements a unit spans)
  long long capacity;                 // list entries reserved (an upper bound of those used)
  int fold_window, fold_windows;
  long long fold_capacity;
  size_t offsets_at, start_at, list_at, offs_at, fold_start_at, fold_list_at, words;
};
static inline LayerPlanLayout layer_plan_layout(int K, int N, int H, int BK, int BN) {
  LayerPlanLayout l = {};
  const long long tiles = (long long)((K + BK - 1) / BK) * ((N + BN - 1) / BN);
  if (tiles > (1 << 22)) return l;
  l.tiles = (int)tiles;
  auto round16 = [](size_t v) { return (v + 15) & ~(size_t)15; };
  l.offsets_at = kLayerPlanHeader;
  l.start_at = round16(l.offsets_at + (size_t)tiles);
  if (window_tile_supported(BK, BN) && tiles <= (1 << 20)) {
    window_geometry(H, &l.window, &l.windows);
    l.strips_per_tile = window_units(BK, BN);
    l.strip_elems = window_unit_span(BN);
    // a unit that spans strip_elems consecutive elements meets at most ceil(strip_elems / window) + 1 windows
    l.capacity = tiles * l.strips_per_tile * ((l.strip_elems + l.window - 1) / l.window + 1);
  }
  l.list_at = round16(l.start_at + (size_t)l.windows + 1);
  l.offs_at = round16(l.list_at + (size_t)l.capacity);
  // a tile of BK * BN consecutive elements meets at most ceil(BK * BN / window) + 1 fold windows
  fold_geometry(H, &l.fold_window, &l.fold_windows);
  l.fold_capacity = tiles * (((long long)BK * BN + l.fold_window - 1) / l.fold_window + 1);
  l.fold_start_at = round16(l.offs_at + (size_t)l.capacity);
  l.fold_list_at = round16(l.fold_start_at + (size_t)l.fold_windows + 1);
  l.words = round16(l.fold_list_at + (size_t)l.fold_capacity);
  l.ok = l.words < (1u << 30);
  return l;
}

// Forward / input-grad with few C tiles and a long contraction (skinny batches): R is cut into
// slices over blockIdx.y, every slice writes an fp32 partial result, a second kernel adds them.
struct SplitPlan {
  int tile;
  int splits;        // 1 = no split, no workspace
  int r_chunk;
  size_t workspace_bytes;
  double est_us;     // what the model expects the launch(es) to take
  int run_steps;     // > 0: in runs of that many steps of 64 (plan_runs); then `splits` is the most parts a tile has and r_chunk a run
  int run_rounds, run_groups, run_tiles;   // whole tiles of every workgroup, workgroups, tiles that are cut
};

// 16-bit forward / input-grad of at most 32 rows whose plan is the 128 tile: C tiles of 32 x 128 (see kernel_form).
// All that decides it is here, because the planner finishes, and prices, a cut by the kernel that will run: an override
// of the tile, the single-stage form or register staging (clamp = -1, rows shorter than a 16-byte piece) keeps the
// square tile.  (A cut of the 128 tile is a multiple of the form's step: slice_unit.)
static inline bool rows32_form(int tile, int I, int R, int elem_bytes, const rz_tuning& t) {
  return tile == 128 && elem_bytes == 2 && I <= 32 && R * elem_bytes >= 16 && t.tile == 0 && t.stages != 1 && t.clamp != -1;
}

// A 16-bit forward / input-grad whose plan is the 128 tile: whether pairs of tiles, 256 x 128, are faster (the square tile reads a half more from LDS per
// multiplication, which is what bounds it; a pair leaves half the compute units idle where there are few tiles).  bf16: 2048 x 4096
// over 1024 23.2 -> 20.1 us; 3001 x 1531 over 2047 49.7 -> 35.9; but 2048^3 22.8 -> 29.4 if it were taken there.
static inline bool pair_form(int tile, int I, int J, int R, int chunk, int elem_bytes, const rz_tuning& t) {
  if (tile != 128 || elem_bytes != 2 || I <= 128 || R < 8 || t.tile != 0 || t.stages == 1 || t.clamp == -1) return false;
  const int slices = chunk < R ? (R + chunk - 1) / chunk : 1;
  const double steps = (double)(((chunk < R ? chunk : R) + 63) / 64);
  return store16_us(256, 128, I, J, slices, steps) < store16_us(128, 128, I, J, slices, steps) * 0.97;
}

// Slices up to which a cut contraction is finished by its own kernel (GemmParams::finish; 0: never).  The
// slice that comes last at a tile reads the others' planes by itself, four bytes per lane and load, after
// an atomic's round trip: that pays up to four slices, where the rows of a tile are real (a batch of
// fewer rows than the tile has is finished in 3 us by a second kernel too), and with the 256 tile only
// where the planes are large.  Measured, forward, GPU-bound (finished in the kernel / second kernel):
// bf16 K = N = 10240: M = 128, 128 tile, three slices 47 / 54 us; M = 32 49 / 46; M = 1024, 256 tile 252 / 260;
// M = 128, 256 tile 104 / 93.  M = 128, K = 2048, N = 8192: 128 tile, three slices 14.7 / 20.8 us.
// M = 64, K = N = 4096: 64 tile, four slices 12.7 / 13.6; 128 tile 21.3 / 18.4.  Six slices at M = 32: 52 / 40.
// Tiles of 32 rows have few values per lane and finish up to eight slices: fp32 M = 32, K = N = 1024 in six slices of the
// 32 x 64 tile 10.5 / 8.0 us through the module (second kernel / finished in the kernel); the 16-bit 32 x 128 tile, M = 32,
// K = N = 10240 in three, 29.4 us in one kernel where a second one takes 4.8 us more.
static inline int finish_slices(int tile, int I, int J, int R, int elem_bytes, const rz_tuning& t) {
  if (rows32_form(tile, I, R, elem_bytes, t)) return finish_limit(32);
  if (I < (tile == 32 ? 32 : tile)) return 0;
  if (tile == 256 && (double)I * J * 4.0 < 16.0e6) return 0;
  return finish_limit(tile);
}

// 16-bit 256 tile: whether `steps` R steps of 64 are too few for the phase loop.  It gains 3 to 5 % per step but takes 1.1 us more around
// its steps (of which the exchange of accumulators is 0.3), with ragged tiles 2 to 3, than the loop of the other tiles.  bf16, us (other
// loop / phase loop), K = N or M = N = 4096 if not said: forward of 1 / 5 / 6 / 8 steps 11.3 / 12.5, 16.2 / 16.5, 17.8 / 17.8, 20.5 / 20.2; ragged,
// 4090 x 4000, 1 / 6 / 12 / 16 steps 14.4 / 17.2, 21.6 / 23.0, 32.0 / 31.9, 39.3 / 38.4, 2030 x 4090 (half the chip) 14.0 / 17.4, 21.4 / 23.9, 29.6 / 30.8,
// 35.1 / 35.6; weight-grad 1 / 3 / 4 steps 23.4 / 23.7, 26.2 / 26.4, 27.5 / 27.4; ragged 1 / 8 / 10 steps 25.2 / 26.7, 32.8 / 33.3, 35.0 / 35.2.
static inline bool short_loop(int op, bool full, int steps) {
  return steps <= (op == kWeightGrad ? (full ? 3 : 8) : (full ? 5 : 10));
}

// 16-bit forward / input-grad of more than 64 rows: roughly how long the call takes, in microseconds, as a sum over what its kernels do:
// rounds of workgroups take their steps and a fixed part, both longer the fuller the chip, with ragged tiles, and with rows that are not whole
// 16-byte pieces; a cut takes a fixed part and its planes, whether its own kernel finishes it or a second one.  Fitted to 54 000
// GPU-bound measurements (forward and input-grad of 2360 shapes of 65 to 32768 rows and 64 to 16384 columns, aligned and odd, every tile,
// one to twelve slices).
struct Forward16Times {
  double launch, step, step_fill, step_ragged, step_odd, round, round_ragged, round_odd, round_fill;
  double finish, finish_mb, second, second_mb, second_slice;   // us, us per MB of planes written and read, us per slice beyond eight
};
static constexpr Forward16Times kForward16Times[7] = {
  {1.978, 0.198, 0.025, 0.004, 0.051, 1.999, 1.049, 0.100, 0.240, 2.615, 0.098, 3.034, 0.209, 0.433},   // 64 tile, at most one workgroup per compute unit
  {4.458, 0.263, 0.194, 0.015, 0.068, -1.211, 0.953, 0.178, 3.756, 3.314, 0.008, 3.387, 0.080, 0.198},   // 64 tile, two per compute unit
  {2.197, 0.420, 0.088, 0.012, 0.099, 1.594, 1.426, 0.193, 1.129, 5.960, 0.102, 2.961, 0.201, 0.001},   // 128 tile of eight wavefronts
  {3.117, 0.487, 0.487, 0.009, 0.179, 1.435, 1.654, 0.849, 1.360, 10.317, 0.114, 7.999, 0.076, 0.001},   // 128 tile of four, pairs on a compute unit
  {2.550, 0.592, 0.134, 0.013, 0.164, 2.418, 1.313, 0.965, 1.519, 11.180, 0.107, 3.789, 0.197, 0.001},   // 256 x 128
  {5.198, 1.201, 0.123, 0.000, 0.144, 0.566, 1.771, 1.471, 4.903, 12.357, 0.159, 6.117, 0.143, 0.001},   // 256 tile, few steps
  {2.453, 0.966, 0.351, 0.021, 0.092, 6.473, 1.870, 1.543, 0.819, 8.326, 0.187, 4.928, 0.118, 0.001},   // 256 tile
};
static inline double forward16_us(int rows, int cols, int I, int J, int R, int slices, int steps, bool finished) {
  const long long wgs = (long long)((I + rows - 1) / rows) * ((J + cols - 1) / cols) * slices;
  const bool full = I % rows == 0 && J % cols == 0 && R % (rows == 64 ? 128 : 64) == 0;
  const double n = steps, ragged = full ? 0.0 : 1.0, odd = (R % 8 != 0 || J % 8 != 0) ? 1.0 : 0.0;
  const long long per = rows == 64 && wgs > kComputeUnits ? 2 * kComputeUnits : kComputeUnits;
  double rounds = (double)((wgs + per - 1) / per), fill = (double)wgs / (rounds * per);
  int which = cols == 256 ? (short_loop(kForward, full, steps) ? 5 : 6) : rows == 256 ? 4 : rows == 64 ? (wgs <= kComputeUnits ? 0 : 1) : 2;
  if (which == 2 && wgs > kComputeUnits * 3 / 2) {   // (a compute unit's last workgroup without a partner takes 0.62 of a pair's time)
    which = 3;
    const long long pairs = wgs / (2 * kComputeUnits), rest = wgs - pairs * 2 * kComputeUnits;
    rounds = (double)pairs + (rest == 0 ? 0.0 : rest > kComputeUnits ? 1.0 : 0.62);
    fill = 1.0;
  }
  const Forward16Times& c = kForward16Times[which];
  const double us = c.launch + rounds * (n * (c.step + c.step_fill * fill + c.step_ragged * ragged + c.step_odd * odd) +
                                         c.round + c.round_ragged * ragged + c.round_odd * odd + c.round_fill * fill);
  if (slices == 1) return us;
  const double mb = (double)I * J * 4.0e-6;
  return us + (finished ? c.finish + c.finish_mb * (2.0 * slices - 1.0) * mb
                        : c.second + c.second_mb * (2.0 * slices + 0.5) * mb + (slices > 8 ? c.second_slice * (slices - 8) : 0.0));
}

// (The plans take a cut as finished by its own kernel wherever finish_slices says so, whatever rz_tuning.finish: with a second kernel, by that
// override or for want of counters, a call keeps its cut, and so its bits.)
// Tile and number of slices together: the pair with the least estimated time.  A slice pays the
// fill and drain of its pipeline (about three steps), the cut pays the fp32 partial planes
// (written, read back) and the launch of the kernel that adds them.
static inline SplitPlan plan_split_by_rate(int I, int J, int R, int elem_bytes, const rz_tuning& t, int depth = 0) {
  SplitPlan best = {};
  double best_us = 0.0;
  const double peak = elem_bytes == 4 ? 149e6 : 1150e6;   // flop per microsecond of the 256 tile on a full chip
  const int tiles_of[4] = {256, 128, 64, 32};
  // (an override that asks for the 32 x 64 tile where it does not exist gets the 64 tile)
  const int forced = (t.tile == 32 && elem_bytes != 4) ? 64 : t.tile;
  for (int tile : tiles_of) {
    if (forced && tile != forced) continue;
    // (the 32 x 64 tile: fp32 only, and only where 64-row tiles would end in a tile at most half full —
    //  K = N = 10240: M = 96 259 -> 232 us, M = 160 428 -> 353 us, M = 288 668 -> 620 us)
    if (tile == 32 && !forced && (elem_bytes != 4 || (I > 32 && (I - 1) % 64 >= 32))) continue;
    // (depth 2: an override's number of slices that whole steps of the 16-bit 64 tile cannot make may be cut at
    //  half of one: the bounds-checked form takes those)
    const int TR = slice_unit(tile, elem_bytes) / (depth == 2 && tile == 64 && elem_bytes == 2 ? 2 : 1);
    const long long tiles = tile_count(I, J, tile);
    const int r_steps = (R + TR - 1) / TR;
    const double useful = (double)I * (double)J / ((double)tiles * tile * tile_cols(tile));
    // fp32 staged directly (complete tiles, or ragged ones with rows of 16 bytes and more): see tile_rate;
    // a workgroup's fill and drain cost about 2, 8 and 12 steps of 128 bytes for the tiles of 256, 128
    // and 64 / 32 x 64 (4096^3: 941, 986, 1016 us; M = 4096, K = N = 1024: 128 tile 76 us, 64 tile 82 us;
    // 1024^3: 64 tile 23.8 us, 128 tile cut in four 35 us).  The bounds-checked form, which only shapes
    // with shorter rows or an override still take, keeps the older pricing.
    const bool whole = I % tile == 0 && J % tile_cols(tile) == 0 && R % TR == 0;
    const bool direct = elem_bytes == 4 && (whole || (t.clamp != -1 && R * elem_bytes >= 16));
    const double lo64 = whole ? 0.67 : 0.60;
    const double fill = !direct ? 2.0 : tile == 256 ? 2.0 : tile == 128 ? 8.0 : 12.0;
    double whole_us = 0.0;
    for (int want = 1; want <= 16; want++) {
      if (want > 1 && t.split == -1) break;
      // (a kernel of a dozen microseconds is not worth cutting: the second launch and the short loops
      //  cost what the idle compute units would have gained — fp32, M = 32 and 96, K = N = 1024: 13 us
      //  whole, 15 us cut in eight or four)
      if (want > 1 && direct && whole_us <= 16.0 && t.split <= 0) break;
      const int steps_per = (r_steps + want - 1) / want;
      const int slices = (r_steps + steps_per - 1) / steps_per;
      if (slices != want) continue;                           // (the same cut as a smaller `want`)
      if (t.split > 0 && slices != t.split) continue;         // (an override asks for exactly that many slices)
      if (slices > 1 && steps_per * (TR * elem_bytes / 128) < 4 && t.split <= 0) break;   // slices of a few steps are all fill and drain
      const double steps = (double)steps_per * (TR * elem_bytes / 128);
      const double rate = peak * tile_rate((double)tiles * slices, tile, elem_bytes, lo64, direct || elem_bytes == 2) * useful * steps / (steps + fill);
      double us = 2.0 * (double)I * (double)J * (double)R / rate + 4.0;
      // (16-bit, more than 64 rows: by the fitted times of the kernels; a slice's planes as fitted with them)
      const bool fitted = elem_bytes == 2 && I > 64;
      if (fitted) {
        const bool pair = pair_form(tile, I, J, R, slices > 1 ? steps_per * TR : R, elem_bytes, t);
        us = store16_us(pair ? 256 : tile, tile, I, J, slices, (double)steps_per * (TR / 64.0));
      }
      // (up to finish_slices the kernel finishes its own tiles: every plane is written, all but one are read
      //  back by the finishing workgroups, and no second kernel is launched — worth a couple of microseconds
      //  and a plane; fp32, M = 16384, K = 512, N = 1024 input-grad, planes of 33 MB: the 256 tile in two
      //  slices 155 us against the whole 128 tile's 136)
      const bool finished = slices > 1 && slices <= finish_slices(tile, I, J, R, elem_bytes, t);
      if (slices > 1 && fitted) us += finished ? (2.0 * slices - 1.0) * (double)I * J * 4.0 / 8.0e6 + 3.5 : (2.0 * slices * (double)I * J * 4.0 + (double)I * J * elem_bytes) / 7.0e6 + 0.5;
      else if (finished) us += (2.0 * slices - 1.0) * (double)I * J * 4.0 / 4.0e6 + 2.0;
      else if (slices > 1) us += (2.0 * slices * (double)I * J * 4.0 + (double)I * J * elem_bytes) / 4.0e6 + (direct ? 3.0 : 4.0);
      else whole_us = us;
      // (near ties go to the larger tile and the fewer slices, which come first)
      if (best.tile == 0 || us < best_us * 0.97) {
        best.tile = tile;
        best.splits = slices;
        best.r_chunk = steps_per * TR;
        best_us = us;
      }
    }
  }
  // (16-bit: a problem that some tile does whole in a dozen microseconds is not cut — M = 128, K = N = 1024:
  //  64 tile whole 10.2 us; every cut, finished in the kernel or not, 12 to 16 us)
  if (elem_bytes == 2 && t.split == 0 && best.splits > 1 && depth == 0) {
    rz_tuning whole_only = t;
    whole_only.split = -1;
    const SplitPlan w = plan_split_by_rate(I, J, R, elem_bytes, whole_only, 1);
    if (w.est_us <= 14.0) return w;
  }
  if (best.tile == 0 && t.split > 0 && depth < 2) return plan_split_by_rate(I, J, R, elem_bytes, t, 2);
  if (best.tile == 0 && t.split > 0) {   // (no cut comes out at exactly that many slices: the library's own choice)
    rz_tuning free_cut = t;
    free_cut.split = 0;
    return plan_split_by_rate(I, J, R, elem_bytes, free_cut);
  }
  best.workspace_bytes = best.splits > 1 ? (size_t)best.splits * (size_t)I * (size_t)J * sizeof(float) : 0;
  best.est_us = best_us;
  return best;
}

// ... and for a 16-bit batch of more than 64 rows the plan with the least time by forward16_us, where that promises 7 % more than
// the fit's error in telling two plans apart.  (The times of the plan by rate know no ragged tiles and take a second kernel for half a
// microsecond.  Measured, 2992 calls: the plan by rate is 3.9 % from the best form on average and more than 10 % in 1 call of 6; so
// 1.2 %, 1 in 22, and 18 calls are more than 3 % slower than by rate, 431 faster — M = 192, K = 3712, N = 1152 forward 15.1 -> 10.3 us, four slices
// for eight; M = 101, K = 2233, N = 1012 15.2 -> 10.8, four for one.  Without the 7 %: 0.7 %, but 102 are slower; in a long training pass
// near ties fall as the plan by rate has them: M = 1024, K = N = 10240 in three slices 658 us, whole 671.)
static inline SplitPlan plan_split_by_slices(int I, int J, int R, int elem_bytes, const rz_tuning& t) {
  const SplitPlan by_rate = plan_split_by_rate(I, J, R, elem_bytes, t);
  if (elem_bytes != 2 || I <= 64 || R < 8 || t.tile != 0 || t.split != 0 || t.stages == 1 || t.clamp == -1) return by_rate;
  auto time_of = [&](int tile, int slices, int chunk) {
    const bool pair = pair_form(tile, I, J, R, slices > 1 ? chunk : R, elem_bytes, t);
    const bool finished = slices > 1 && slices <= finish_slices(tile, I, J, R, elem_bytes, t);
    return forward16_us(pair ? 256 : tile, tile, I, J, R, slices, chunk / 64, finished);
  };
  SplitPlan best = by_rate;
  double best_us = 0.0;
  const int tiles_of[3] = {256, 128, 64};
  for (int tile : tiles_of) {
    const int TR = slice_unit(tile, elem_bytes), r_steps = (R + TR - 1) / TR;
    for (int slices = 1; slices <= 16; slices++) {
      const int chunk = (r_steps + slices - 1) / slices * TR;
      if (((r_steps * TR + chunk - 1) / chunk) != slices) continue;   // (the same cut as fewer slices)
      if (slices > 1 && chunk < 4 * 64) break;   // slices of a few steps are all fill and drain
      const double us = time_of(tile, slices, chunk);
      if (best_us == 0.0 || us < best_us * 0.97) {   // (near ties go to the larger tile and the fewer slices)
        best.tile = tile;
        best.splits = slices;
        best.r_chunk = chunk;
        best_us = us;
      }
    }
  }
  const int unit = slice_unit(by_rate.tile, elem_bytes);
  const double by_rate_us = time_of(by_rate.tile, by_rate.splits, by_rate.splits > 1 ? by_rate.r_chunk : (R + unit - 1) / unit * unit);
  if (best_us >= 0.93 * by_rate_us) return by_rate;
  best.workspace_bytes = best.splits > 1 ? (size_t)best.splits * (size_t)I * (size_t)J * sizeof(float) : 0;
  best.est_us = best_us;
  return best;
}

// 16-bit forward / input-grad in runs of equal length (GemmKernel::run_all), C tiles of 256 x cols: what fills whole rounds of the compute
// units is left whole, and the steps of the tiles that remain are dealt out evenly.  tile = 0: no such cut.  A tile has
// at most as many parts as the kernel adds up.  Of the lengths of a run from an even share to a quarter more, the one with the least
// time by what forward16_us was fitted to: steps, a fixed part for every tile and piece, planes written and read (a longer run may leave
// the tiles' ends in fewer pieces).  The 256 tile's runs are 4 % faster than that says, those of 256 x 128 up to 8 % slower.
static constexpr size_t kRunAlign = 16;   // (the planes are read and written two floats at a time, whatever address the workspace has)
static inline SplitPlan plan_runs(int I, int J, int R, int cols) {
  SplitPlan best = {};
  const long long tiles = (long long)((I + 255) / 256) * ((J + cols - 1) / cols);
  const long long rounds = tiles / kComputeUnits, rest = tiles - rounds * kComputeUnits;
  const int steps = (R + 63) / 64;
  if (rest == 0 || rounds > 0x7fff || rest * steps > 0x3fffffff) return best;
  const Forward16Times& c = kForward16Times[cols == 256 ? 6 : 4];
  const bool full = I % 256 == 0 && J % cols == 0 && R % 64 == 0, odd = R % 8 != 0 || J % 8 != 0;
  const double step = c.step + c.step_fill + (full ? 0.0 : c.step_ragged) + (odd ? c.step_odd : 0.0);
  const double fixed = c.round + c.round_fill + (full ? 0.0 : c.round_ragged) + (odd ? c.round_odd : 0.0);
  const double mb = 256.0 * cols * 4.0e-6, share = cols == 256 ? 0.96 : 1.08;
  const int even = (int)((rest * steps + kComputeUnits - 1) / kComputeUnits);
  for (int L = even < 8 ? 8 : even; L < steps && L <= even + even / 4; L++) {
    const int F = steps / L, r = steps - F * L;
    const bool ends_cut = r != 0 && rest * r > L && L % r != 0;   // (a cut lies inside an end)
    const int parts = F + (r == 0 ? 0 : ends_cut ? 2 : 1);        // the most of a tile
    if (parts > kFinishSlices) continue;
    const long long end_runs = (rest * r + L - 1) / L, groups = rest * F + end_runs;
    if (groups > kComputeUnits) continue;
    const double pieces_all = (double)(rest * (F + (r != 0 ? 1 : 0)) + (ends_cut ? end_runs - 1 : 0));
    const double most = r == 0 ? 1.0 : rest * r <= L ? (double)rest : 1.0 + (L + r - 2) / r;
    const double pieces = 0.5 * (most + pieces_all / groups);
    const double us = share * (c.launch + (double)rounds * (steps * step + fixed) + L * step + pieces * fixed + c.finish +
                               c.finish_mb * (2.0 * pieces_all - (double)rest) * mb);
    if (best.tile != 0 && us >= best.est_us) continue;
    best.tile = cols;
    best.splits = parts;
    best.r_chunk = L * 64;
    best.run_steps = L;
    best.run_rounds = (int)rounds;
    best.run_groups = rounds > 0 ? kComputeUnits : (int)groups;
    best.run_tiles = (int)rest;
    best.est_us = us;
  }
  if (best.tile != 0) best.workspace_bytes = (size_t)best.splits * (size_t)best.run_tiles * 256 * (size_t)cols * sizeof(float) + kRunAlign;
  return best;
}
static inline SplitPlan plan_split(int I, int J, int R, int elem_bytes, const rz_tuning& t) {
  SplitPlan best = plan_split_by_slices(I, J, R, elem_bytes, t);
  if (elem_bytes != 2 || I <= 64 || R < 8 || t.tile != 0 || t.split != 0 || t.stages == 1 || t.clamp == -1) return best;
  const SplitPlan wide = plan_runs(I, J, R, 256), pair = plan_runs(I, J, R, 128);
  // the plan by slices, by the same times; runs have to promise 5 %.  bf16 / fp16, by slices or whole / in runs, us: M = 1024, K = N = 10240 forward
  // 194 / 177, input-grad 191 / 178; M = 5031, 4002 <- 6371 296 / 230; M = 8864, 9146 -> 934 222 / 165; M = 3744, 9622 <- 9701 698 / 609;
  // M = 1286, 9678 -> 16359 432 / 369.  Taken for 3 of 100 drawn calls of more than 64 rows, those with a long R and a last round that is far from full: on 20 of them 0.91
  // times the time in the mean, at most 0.99.
  const bool finished = best.splits > 1 && best.splits <= finish_slices(best.tile, I, J, R, elem_bytes, t);
  const int unit = slice_unit(best.tile, elem_bytes), chunk = best.splits > 1 ? best.r_chunk : (R + unit - 1) / unit * unit;
  const bool pairs = pair_form(best.tile, I, J, R, best.splits > 1 ? chunk : R, elem_bytes, t);
  const double us = forward16_us(pairs ? 256 : best.tile, best.tile, I, J, R, best.splits, chunk / 64, finished);
  const SplitPlan& runs = pair.tile == 0 || (wide.tile != 0 && wide.est_us <= pair.est_us) ? wide : pair;
  // (nor for planes of more than twice what the call reads and writes, unless slices take as much: M = 653, K = 11012 <- 6869 would have 104 MB
  //  beside 23 MB of dY and dX.  Of the plans in runs 7 % are left out by that, all of short batches.)
  const size_t most = 2 * (size_t)elem_bytes * (size_t)I * ((size_t)J + (size_t)R);
  if (runs.workspace_bytes > (best.workspace_bytes > most ? best.workspace_bytes : most) + kRunAlign) return best;
  return runs.tile != 0 && runs.est_us < 0.95 * us ? runs : best;
}

// Which instantiation of the contraction kernel runs a launch: C tile, wavefronts, LDS stages,
// whether every tile and step is complete (no bounds checks), whether a ragged shape still
// takes direct staging with edge pieces fetched from inside the operands, and the contracted
// elements per step that follow from those.  One function decides for the launch and for
// rz_plan_query.
struct KernelForm {
  int tile, rows, cols, waves, stages;   // tile: the planner's code; rows x cols: the C tile of the kernel that serves it
  bool full, clamp;
  bool short_loop;   // 16-bit 256 tile: the loop for a few R steps
  int step;
};

// (image: a weight-grad whose workgroups hold an image of dHW in LDS)
static inline KernelForm kernel_form(int op, int I, int J, int R, int chunk, int tile, long long workgroups,
                                     int elem_bytes, const rz_tuning& t, bool image = false) {
  KernelForm f;
  f.tile = tile;
  f.rows = tile;
  f.cols = tile_cols(tile);
  f.stages = (tile == 128 && t.stages == 1) ? 1 : 2;
  // 128 tile: with about one workgroup per compute unit, eight wavefronts (two per SIMD, 64 x 32
  // each) hide latency better than four of 64 x 64; with more workgroups resident the
  // four-wavefront form does less LDS traffic per flop
  // 16-bit, eight wavefronts, directly staged: four stages of 128 bytes of R (128 KB).  With two of 256 bytes, in as
  // much LDS, the loads of a step were issued when the last ones had landed, so that between two barriers nothing was in
  // flight for a while; now three steps are at any time (M = 128, K = N = 10240 in three slices, forward and input-grad:
  // 44.7 -> 42.3 and 45.2 -> 41.0 us; M = 3001, K = 2047, N = 1531 input-grad 42.0 -> 40.4 us; 2048^3 as before, 22.5)
  // 64 tile: four wavefronts; fp32 forward / input-grad take eight (two groups that share every R
  // step: a second wavefront per SIMD keeps the MFMA pipe fed while the first waits for LDS)
  // (32-bit: every two-stage form stages directly; 16-bit too)
  const bool direct_capable = f.stages == 2;
  // 64 tile, 16-bit: sixteen wavefronts in four groups that share every 256-byte step — a problem of few
  // tiles leaves most compute units idle and the others waiting for memory, and four wavefronts cannot keep
  // enough loads in flight.  Up to one workgroup per compute unit, four LDS stages (128 KB in flight); beyond
  // that, two, so that two workgroups share a compute unit.
  const bool many64 = tile == 64 && elem_bytes == 2;
  const int waves128 = f.stages == 1 ? 4 : (workgroups <= kComputeUnits * 3 / 2 ? 8 : 4);
  const int step_plain = elem_bytes == 4 ? slice_unit(tile, elem_bytes, op == kWeightGrad) : 128 / elem_bytes;
  const int step_direct = (direct_capable && elem_bytes == 2 && many64) ? 256 / elem_bytes : step_plain;
  f.full = (I % tile == 0) && (J % tile_cols(tile) == 0) && (R % step_direct == 0) && (chunk % step_direct == 0);
  // a plain operand's rows must hold at least one 16-byte piece (a piece that straddles the end of a
  // row is handled in the kernel; a row shorter than a piece is not)
  const int vec = 16 / elem_bytes;
  const bool pieces_ok = (op == kWeightGrad ? (I >= vec && J >= vec) : R >= vec) && (chunk >= R || chunk % step_direct == 0);
  f.clamp = !f.full && direct_capable && pieces_ok && t.clamp != -1;
  f.step = (f.full || f.clamp) ? step_direct : step_plain;
  // (fp32 weight-grad on the 64 tile: in two groups, as forward and input-grad, for at most one workgroup per compute unit and a long loop, or an image, which
  //  more wavefronts clear and store.  With more workgroups, the four-wavefront ones that share a unit hide as much, and adding the groups up costs.  124 drawn
  //  calls, eight wavefronts in place of four, times the time: at most 256 workgroups of 512 rows and more 0.95 to 0.99, of fewer 1.01 to 1.04, of a few rows
  //  and an image 0.98 to 0.99 (M = 3, K = N = 192, a pass 18.2 / 17.8 us); up to 512 workgroups 1.02 to 1.09, up to 1024 1.02 to 1.04, beyond 1.00 to 1.02.)
  const bool two_groups = workgroups <= kComputeUnits && (image || (chunk < R ? chunk : R) >= 512);
  f.waves = tile == 256 ? 8
            : tile == 32 ? 4
            : tile == 64 ? ((many64 && (f.full || f.clamp)) ? 16 : (elem_bytes == 4 && (op != kWeightGrad || (two_groups && (f.full || f.clamp)))) ? 8 : 4)
                         : waves128;
  if (tile == 128 && f.waves == 8 && elem_bytes == 2 && (f.full || f.clamp)) f.stages = 4;
  if (f.waves == 16) f.stages = workgroups <= kComputeUnits ? 4 : 2;
  // 16-bit forward / input-grad on the planner's 128 tile, a batch of at most 32 rows (decoding): C tiles of 32 x 128.
  // The 128 rows of the square tile would stage the batch four times over beside every piece of W; without them three
  // LDS stages fit, twice as many bytes of W are in flight, and no padded rows are multiplied or stored, so that the
  // kernel can finish a cut itself (K = N = 10240, H = 6.5 M bf16, three slices: M = 1 43.5 -> 28.3 us, M = 32 42.0 -> 29.4 us,
  // 7.1 TB/s of W from beyond the L2s).  33 to 64 rows: two such tiles would read W twice; the 64 tile takes those.
  if (op != kWeightGrad && rows32_form(tile, I, R, elem_bytes, t)) {
    f.rows = 32;
    f.waves = 8;
    f.stages = 3;
    f.step = 128;
    f.full = I == 32 && J % 128 == 0 && R % 128 == 0 && chunk % 128 == 0;
    f.clamp = !f.full;
  }
  // 16-bit forward / input-grad on the planner's 128 tile: two tiles of one column by one workgroup, where that is the faster
  if (op != kWeightGrad && f.rows == 128 && pair_form(tile, I, J, R, chunk, elem_bytes, t)) {
    f.rows = 256;
    f.waves = 8;
    f.stages = 3;
    f.full = I % 256 == 0 && J % 128 == 0 && R % 64 == 0 && chunk % 64 == 0;
    f.clamp = !f.full;
  }
  f.short_loop = elem_bytes == 2 && tile == 256 && (f.full || f.clamp) && short_loop(op, f.full, ((chunk < R ? chunk : R) + 63) / 64);
  return f;
}

// An input-grad planned in runs, beside a weight-grad on the same tile in one launch: its tiles whole, since what they leave idle the
// weight-grad's workgroups fill and no planes are needed.  tile = 0: in runs, as by itself.  By the times that forward16_us was fitted to:
// the launch takes the sum of what its workgroups take, spread over the compute units, and half a workgroup of the op whose
// workgroups come last, but no less than the longest.  (M = 1024, K = N = 10240 bf16: 181 + 199 us in runs and apart, 347 in one launch.)
static inline SplitPlan backward_whole_tiles(int M, int K, int N, const SplitPlan& sp, const WeightGradPlan& plan) {
  SplitPlan whole = {};
  if (sp.run_steps == 0 || sp.tile != 256 || plan.tile != 256) return whole;
  const Forward16Times& c = kForward16Times[6];
  const double step = c.step + c.step_fill, fixed = c.round + c.round_fill;
  const double ig_us = (double)((N + 63) / 64) * step + fixed, wg_us = (double)((plan.r_chunk + 63) / 64) * step + fixed;
  const double ig_wgs = (double)tile_count(M, K, 256), wg_wgs = (double)plan.workgroups;
  const double spread = (ig_wgs * ig_us + wg_wgs * wg_us) / kComputeUnits + 0.5 * (ig_us < wg_us ? ig_us : wg_us);
  const double longest = ig_us > wg_us ? ig_us : wg_us, together = c.launch + (spread > longest ? spread : longest);
  const double apart = sp.est_us + c.launch + (double)(((long long)plan.workgroups + kComputeUnits - 1) / kComputeUnits) * wg_us;
  if (together >= 0.97 * apart) return whole;
  whole.tile = 256;
  whole.splits = 1;
  whole.r_chunk = N;
  whole.est_us = together;
  return whole;
}

// Input-grad and weight-grad of one backward pass in one launch (rz_backward_kernel): which pair of kernels, kApart where the two
// have no launch in common.
enum BackwardPair { kApart = 0, k64With64, k64With128, kPairWith128, kPairWith256, k256With256, k256With128, k128With128 };
struct BackwardForm {
  int pair;
  bool full;      // both without bounds checks (else both with)
  int stages;     // of the 16-bit 64 tiles
  bool wg_first;  // whose workgroups come first in the grid: those that take longer
};
static inline long long f_tiles(const KernelForm& f, int I, int J) {
  return (long long)((I + f.rows - 1) / f.rows) * ((J + f.cols - 1) / f.cols);
}
// When the last of n1 workgroups of d1 each, then n2 of d2, is done, each on the compute unit that is free first: the first op's last round leaves
// `late` units a workgroup longer.
static inline double list_schedule(long long n1, double d1, long long n2, double d2) {
  const long long rounds1 = n1 / kComputeUnits, late = n1 - rounds1 * kComputeUnits;
  const double from_a = (double)rounds1 * d1, from_b = from_a + d1;
  double end = late > 0 ? from_b : from_a;
  for (long long done_a = 0, done_b = 0; done_a * (kComputeUnits - late) + done_b * late < n2;) {
    const double next_a = from_a + (double)(done_a + 1) * d2, next_b = from_b + (double)(done_b + 1) * d2;
    if (late == 0 || next_a <= next_b) done_a++;
    else done_b++;
    const double last = late == 0 || next_a <= next_b ? next_a : next_b;
    end = last > end ? last : end;
  }
  return end;
}

// runs_us: sp are whole tiles in place of runs, which take so long by themselves (0: sp is how the input-grad goes by itself).
static inline BackwardForm backward_form(int M, int K, int N, int H, const SplitPlan& sp, const WeightGradPlan& plan, bool with_dbias,
                                         int elem_bytes, const rz_tuning& t, double runs_us = 0.0) {
  BackwardForm b = {kApart, false, 2, false};
  if (!with_dbias || sp.run_steps > 0 || t.tile != 0 || t.stages == 1 || t.clamp == -1 || (long long)H * 4 > 0x7fffffffLL) return b;
  const long long ig_wgs = tile_count(M, K, sp.tile) * sp.splits;
  const KernelForm i = kernel_form(kInputGrad, M, K, N, sp.splits > 1 ? sp.r_chunk : N, sp.tile, ig_wgs, elem_bytes, t);
  const KernelForm w = kernel_form(kWeightGrad, K, N, M, plan.r_chunk, plan.tile, plan.workgroups, elem_bytes, t, plan.image_pitch > 0);
  if (!(i.full || i.clamp) || !(w.full || w.clamp) || i.short_loop || w.short_loop) return b;
  const bool pair = i.rows == 256 && i.cols == 128;
  if (i.rows != i.cols && !pair) return b;
  b.full = i.full && w.full;
  if (i.rows == 64 && w.tile == 64) {
    // (fp32: by eight wavefronts here, see kernel_form; many workgroups of a short loop lose more by that than a boundary)
    if (elem_bytes == 4 && plan.workgroups > 2 * kComputeUnits && (plan.r_chunk < M ? plan.r_chunk : M) < 384) return b;
    b.pair = k64With64;
    b.stages = elem_bytes == 2 && ig_wgs + plan.workgroups <= kComputeUnits ? 4 : 2;
  } else if (elem_bytes == 2 && i.rows == 64 && w.tile == 128 && w.waves == 8) {
    // (the 128 tile by sixteen wavefronts of 32 x 32 here: a third more LDS traffic, for a few steps)
    if (ig_wgs <= kComputeUnits && plan.r_chunk <= 2048) b.pair = k64With128;
  } else if (elem_bytes == 2 && pair && w.tile == 128 && w.waves == 8) {
    b.pair = kPairWith128;
  } else if (elem_bytes == 2 && pair && w.tile == 256) {
    b.pair = kPairWith256;
  } else if (elem_bytes == 2 && i.rows == 256 && w.tile == 256) {
    b.pair = k256With256;
  } else if (elem_bytes == 2 && i.rows == 256 && w.tile == 128 && w.waves == 8) {
    b.pair = k256With128;
  } else if (elem_bytes == 2 && i.rows == 128 && i.waves == 8 && w.tile == 128 && w.waves == 8) {
    b.pair = k128With128;
  }
  if (b.pair == kApart) return b;
  if (b.pair == k64With64) {   // (several workgroups of each on a compute unit: those of the longer loop first)
    const int ig_loop = sp.splits > 1 ? sp.r_chunk : N, wg_loop = plan.r_chunk < M ? plan.r_chunk : M;
    b.wg_first = plan.r_chunk > ig_loop;
    // (an image of dHW that leaves a compute unit room for one workgroup, the input-grad's as well)
    const size_t image_bytes = plan.image_pitch > 0 ? (size_t)plan.image_pitch * sizeof(float) + (16 + 65) * sizeof(int) : 0;
    const bool one_each = image_bytes > 80 * 1024, two_each = !one_each && 3 * image_bytes > 160 * 1024;
    if (elem_bytes == 2) {
      // An input-grad of at most one workgroup a unit has four stages by itself; beside a weight-grad that fills the units twice over anyway it
      // would only lose them (M = 3968, K = 256, N = 2688 35.1 apart, 36.2 us).  One of more than three to two units, of a long loop, would lose its
      // neighbour to an image (bf16 M = 9856, K = 192, N = 2688, 129 KB, 462 of them: 117 / 122; fp16 M = 5664, N = 2560, 267: 99 / 91).
      if (ig_wgs <= kComputeUnits && ig_wgs + plan.workgroups > 2 * kComputeUnits && N >= 1024) b.pair = kApart;
      if (one_each && ig_wgs > 3 * kComputeUnits / 2 && N >= 1024) b.pair = kApart;
      return b;
    }
    // fp32, in rows of the contracted dimension at 0.02 us on a compute unit, with a fixed part: the two ops one after the other, each in rounds (of
    // four-wavefront workgroups with an image more than two may share a unit, so that their last round counts by its share), against a list schedule.
    // Apart there is a boundary more.  Together the weight-grad's workgroups have eight wavefronts, which costs 3 % (6.5 % if an image also takes an
    // input-grad's neighbour), but gains 3 % where an image leaves room for two workgroups, and beyond two workgroups a unit the second op's come to lie as
    // they fall, which costs a quarter of one.
    // Fitted to 503 drawn calls: of those that it joins 15 are slower than apart by more than 1 % (at most 9 %), the others up to 33 % faster; 18 that it does
    // not join would be 3 to 9 % faster.  Joined wherever the kernels match, 97 were slower by 1 to 11 %.  Apart / together, us: M = 50, 1920 -> 192
    // 25.6 / 19.3; M = 384, 3008 -> 832 (282 and 611 workgroups) 66.2 / 51.3; but M = 1984, 320 -> 3008 (465 and 235 workgroups) 88.5 / 97.6,
    // M = 6688, 192 -> 12672 with an image of 97 KB 665 / 742.
    const double di = ig_loop + 100.0, dw = wg_loop + 130.0, n_w = (double)plan.workgroups;
    double rounds_w = (double)((plan.workgroups + kComputeUnits - 1) / kComputeUnits);
    if (plan.image_pitch > 0 && !two_each && plan.workgroups > 2 * kComputeUnits && n_w / kComputeUnits + 0.25 < rounds_w) rounds_w = n_w / kComputeUnits + 0.25;
    const double apart = (double)((ig_wgs + kComputeUnits - 1) / kComputeUnits) * di + rounds_w * dw;
    const double together = b.wg_first ? list_schedule(plan.workgroups, dw, ig_wgs, di) : list_schedule(ig_wgs, di, plan.workgroups, dw);
    const double loose = ig_wgs + plan.workgroups > 2 * kComputeUnits ? 0.25 * (b.wg_first ? di : dw) : 0.0;
    const double larger = (one_each && ig_wgs > kComputeUnits ? 0.065 : two_each ? -0.03 : 0.03) * apart;
    if ((apart - together - loose - larger) * 0.02 + 5.0 <= 0.0) b.pair = kApart;
    return b;
  }
  // One workgroup on a compute unit: by what the two kernels and the common one take.  A workgroup takes its steps of 64 and a fixed part
  // (forward16_us), the steps longer the fuller the chip; in the common launch the compute units that one op leaves idle
  // take workgroups of the other, and all of them run at a full chip's pace.  (Two ops of 153 and 162 workgroups, bf16 M = 4288, K = 2304, N = 4544, are 315
  // for 256 units: 211 us, apart 197.)
  auto times = [&](const KernelForm& f, bool wg, int chunk, int R, double fill) {
    const Forward16Times& c = kForward16Times[f.rows == 256 ? (f.cols == 256 ? 6 : 4) : f.rows == 128 ? 2 : 0];
    return ((chunk < R ? chunk : R) + 63) / 64 * (c.step + c.step_fill * fill) * (wg && f.rows == 128 ? 1.15 : 1.0) + c.round + c.round_fill * fill;
  };
  const long long n_i = f_tiles(i, M, K) * sp.splits, n_w = plan.workgroups;
  auto alone = [&](const KernelForm& f, bool wg, int chunk, int R, long long n) {
    const double rounds = (double)((n + kComputeUnits - 1) / kComputeUnits);
    return rounds * times(f, wg, chunk, R, (double)n / (rounds * kComputeUnits));
  };
  const int ig_chunk = sp.splits > 1 ? sp.r_chunk : N;
  const double full = n_i + n_w >= kComputeUnits ? 1.0 : (double)(n_i + n_w) / kComputeUnits;
  const double d_i = times(i, false, ig_chunk, N, full), d_w = times(w, true, plan.r_chunk, M, full);
  b.wg_first = d_w > d_i;
  const double d1 = b.wg_first ? d_w : d_i, d2 = b.wg_first ? d_i : d_w;
  const long long n1 = b.wg_first ? n_w : n_i, n2 = b.wg_first ? n_i : n_w;
  const double end = list_schedule(n1, d1, n2, d2);
  // What the two lose side by side: about 2 % of a launch that shares nothing else (M = 8192, K = 4096, N = 16384, whose ops fill whole rounds, a pass
  // 2316 us apart, 2349 in one launch), and 15 % of one of complete 128 tiles: bf16 M = 14336, K = 128, N = 6912 110 / 124, fp16 M = 16128, K = 256,
  // N = 2816 82 / 95; of 108 drawn passes 56 of the 61 that this leaves apart are slower in one launch, by up to 15 %, and 42 of the 47 that it joins
  // faster, by up to 26 % (bf16 M = 1408, K = 1920, N = 2816, 165 and 330 workgroups, 84 / 69), the others slower by at most 6 %.  (Why is not known: the
  // L2s miss as often, 2.2 and 2.3 million requests a pass of the second.)
  // And where both ops fill whole rounds there is the boundary alone to gain, nothing if X and dY, which both ops read, are more than the L2s hold (32 MB
  // in all): M = 4096, K = 512, N = 1024 61.8 us a pass apart, 59.0 in one launch, M = 8192 60.8 and 59.1; M = 16384 70.2 and 69.9, and 1 us slower where
  // the host is as slow; of 24 drawn ones none gains more than 2.3 %.  (Nearly whole rounds gain: 96 drawn passes on other tiles 0.97 in the mean.)
  // (A complete op beside a ragged one takes the checks too, which is not priced: 150 such drawn passes 0.94 in the mean, the slowest 1.03.)
  const double boundary_us = 4.0, mixing = b.pair == k128With128 && b.full ? 1.15 : 1.02;
  if (n_i % kComputeUnits == 0 && n_w % kComputeUnits == 0 && (double)M * ((double)K + N) * elem_bytes > 32.0e6) b.pair = kApart;
  const double ig_alone = runs_us > 0.0 ? runs_us - kForward16Times[6].launch : alone(i, false, ig_chunk, N, n_i);
  if (end * mixing > (ig_alone + alone(w, true, plan.r_chunk, M, n_w)) + boundary_us) b.pair = kApart;
  return b;
}

// An input-grad beside which the fragments of a windowed weight-grad are made (rz_input_grad_pack_kernel); groups = 0: by a kernel of their own, which takes
// 4 to 5 us of which 1 to 2 are work.  16-bit; fp32's tiles share compute units, so that none is idle.
struct PackForm {
  int groups;           // workgroups that make them, behind those of the input-grad
  long long fragments;
  int rows;             // of the input-grad's C tile, which tells its kernel
  bool full;
};
// whole_pieces: X and dY lie at, and their rows are multiples of, 16 bytes.
static inline PackForm pack_form(int M, int K, int N, int BK, int BN, bool whole_pieces, const SplitPlan& sp, int elem_bytes, const rz_tuning& t) {
  PackForm f = {};
  if (elem_bytes != 2 || !whole_pieces || K % 8 != 0 || N % 8 != 0 || sp.run_steps > 0 || t.tile != 0 || t.stages == 1 || t.clamp == -1) return f;
  const int chunk = sp.splits > 1 ? sp.r_chunk : N;
  const KernelForm i = kernel_form(kInputGrad, M, K, N, chunk, sp.tile, tile_count(M, K, sp.tile) * sp.splits, elem_bytes, t);
  const bool served = (i.rows == 32 && i.cols == 128) || (i.rows == 64 && i.stages == 4) || (i.rows == 128 && i.waves == 8 && i.stages == 4) ||
                      (i.rows == 256 && i.cols == 128);
  if (!served || !(i.full || i.clamp)) return f;
  const long long idle = kComputeUnits - f_tiles(i, M, K) * sp.splits;
  const long long blocks = (long long)((K + BK - 1) / BK) * (BK / 32) + (long long)((N + BN - 1) / BN) * (BN / 32);
  f.fragments = blocks * ((M + 15) / 16);
  if (idle < 1) return f;
  // The workgroups that make them, one on each idle compute unit, must be done before the input-grad is: 0.06 us a fragment and unit.  Passes, GPU-bound, apart /
  // beside, us: bf16 K = N = 10240, H = 6.5 M, 16 idle units: M = 32 107.2 / 104.6, 128 152.0 / 150.2, 200 228.0 / 225.3; M = 96 5008 x 7008, 56 of them,
  // 91.7 / 88.1; M = 152 3008 x 5008 65.2 / 62.4; M = 128 3072 x 6144, 64 of them, 57.2 / 54.3.  (Element by element in these workgroups, 0.19 us a fragment, M = 128 took 181.)
  const double pack_us = 3.0 + 0.06 * (double)f.fragments / (double)idle;
  if (pack_us > sp.est_us) return f;
  const long long most = (f.fragments + i.waves - 1) / i.waves;
  f.groups = (int)(idle < most ? idle : most);
  f.rows = i.rows;
  f.full = i.full;
  return f;
}
hipError_t launch_backward_f32(GemmParams ig, const SplitPlan* split, GemmParams wg, const WeightGradPlan* plan, const BackwardForm& form, hipStream_t stream);
hipError_t launch_backward_bf16(GemmParams ig, const SplitPlan* split, GemmParams wg, const WeightGradPlan* plan, const BackwardForm& form, hipStream_t stream);
hipError_t launch_backward_f16(GemmParams ig, const SplitPlan* split, GemmParams wg, const WeightGradPlan* plan, const BackwardForm& form, hipStream_t stream);

// Fill in the tiling fields of `p` and enqueue the kernel of one op and element type on `stream`; weight-grad
// takes its plan (tile, split of M, scatter mode) from `plan`, the others ignore it.
// (forward / input-grad take tile and split from `split`, or pick a tile and do not split).
hipError_t launch_forward_f32(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split, const rz_tuning& tuning, hipStream_t stream);
hipError_t launch_input_grad_f32(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split, const rz_tuning& tuning, hipStream_t stream);
hipError_t launch_weight_grad_f32(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split, const rz_tuning& tuning, hipStream_t stream);
hipError_t launch_forward_bf16(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split, const rz_tuning& tuning, hipStream_t stream);
hipError_t launch_input_grad_bf16(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split, const rz_tuning& tuning, hipStream_t stream);
hipError_t launch_weight_grad_bf16(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split, const rz_tuning& tuning, hipStream_t stream);
hipError_t launch_forward_f16(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split, const rz_tuning& tuning, hipStream_t stream);
hipError_t launch_input_grad_f16(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split, const rz_tuning& tuning, hipStream_t stream);
hipError_t launch_weight_grad_f16(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split, const rz_tuning& tuning, hipStream_t stream);

struct WindowParams;
hipError_t launch_input_grad_pack_bf16(const GemmParams& ig, const SplitPlan* split, const WindowParams& w, const PackForm& form, hipStream_t stream);
hipError_t launch_input_grad_pack_f16(const GemmParams& ig, const SplitPlan* split, const WindowParams& w, const PackForm& form, hipStream_t stream);
// Enqueues the windowed weight-grad kernel; p.window and the tile grid must come from plan_window.
hipError_t launch_window_f32(const WindowParams& p, int windows, hipStream_t stream);
hipError_t launch_window_bf16(const WindowParams& p, int windows, hipStream_t stream);
hipError_t launch_window_f16(const WindowParams& p, int windows, hipStream_t stream);

}  // namespace rz
