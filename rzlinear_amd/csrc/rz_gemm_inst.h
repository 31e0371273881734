// Body shared by the per-dtype translation units: tile choice + launch.
#pragma once

#include <atomic>

#include "rz_gemm.h"
#include "rz_launch.h"
#include "rz_window.h"

namespace rz {

// The fields of p that the launch of kernel K fills in, its grid and its LDS bytes.
template <typename K, typename T, int OP, int TI, int TJ, bool COLSUM>
static hipError_t prepare_one(GemmParams& p, const WeightGradPlan* plan, const SplitPlan* split, dim3* grid, size_t* smem) {
  p.tiles_i = (p.I + TI - 1) / TI;
  p.tiles_j = (p.J + TJ - 1) / TJ;
  const long long tiles = (long long)p.tiles_i * p.tiles_j;
  if (tiles <= 0 || tiles > 0x7fffffffLL) return hipErrorInvalidValue;
  int splits = 1;
  const int r_steps = (p.R + K::TR - 1) / K::TR;
  if (OP == kWeightGrad) {
    if (plan == nullptr || plan->tile != TI) return hipErrorInvalidValue;
    splits = plan->splits;
    p.r_chunk = plan->r_chunk;
    p.image_pitch = plan->image_pitch;
    if ((size_t)p.image_pitch * sizeof(float) > kMaxImageBytes) return hipErrorInvalidValue;
    // exactly one target: the tile-by-tile output, or an image (LDS mode: partial images) to scatter into
    if (plan->fold.use != (p.tiles_out != nullptr) || (p.tiles_out == nullptr) == (p.scatter == nullptr))
      return hipErrorInvalidValue;
    if (plan->fold.use && p.image_pitch > 0) return hipErrorInvalidValue;
    if (COLSUM) {
      if (p.colsum == nullptr || plan->colsum_pitch != p.tiles_j * TJ ||
          plan->colsum_rows != plan->splits * p.tiles_i)
        return hipErrorInvalidValue;
      p.colsum_pitch = plan->colsum_pitch;
    }
  } else if (split != nullptr && split->splits > 1) {
    constexpr int kPlanTile = TI != TJ && TJ == 128 ? 128 : TI;   // (the C tiles of 32 x 128 and 256 x 128 serve plans of the 128 tile)
    if (split->tile != kPlanTile || p.partial == nullptr) return hipErrorInvalidValue;
    splits = split->splits;
    p.r_chunk = split->r_chunk;
    // a slice must begin on a step boundary: the offset table of a step assumes that the step
    // lies inside one hashed tile or covers whole ones
    if (p.r_chunk % K::TR != 0) return hipErrorInvalidValue;
    // (the kernel that finishes its own tiles holds the other slices' values in registers)
    if (p.finish != nullptr && splits > finish_limit(TI)) return hipErrorInvalidValue;
  } else {
    p.r_chunk = r_steps * K::TR;
    p.partial = nullptr;
    p.finish = nullptr;
  }
  *smem = sizeof(typename K::Smem);
  static_assert(sizeof(typename K::Smem) <= 160 * 1024, "tile does not fit the 160 KB LDS of a compute unit");
  if (OP == kWeightGrad && p.image_pitch > 0) {
    // the dHW image and the scatter's offset table behind it may need more than the stages
    const size_t need = (size_t)p.image_pitch * sizeof(float) + (K::kOffEntries + K::kTurnEntries) * sizeof(int);
    if (need > *smem) *smem = need;
  }
  *grid = dim3((unsigned)tiles, (unsigned)splits, 1);
  return hipSuccess;
}

template <typename T, int OP, int TI, int TJ, int WI, int WJ, int NSTAGE, bool FULL, bool COLSUM, bool CLAMP = false,
          int WK = 1, bool SHORT = false>
static hipError_t launch_one(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split,
                             hipStream_t stream) {
  static std::atomic<uint64_t> lds_limit_raised{0};
  typedef GemmKernel<T, OP, TI, TJ, WI, WJ, NSTAGE, FULL, COLSUM, CLAMP, WK, SHORT> K;
  dim3 grid;
  size_t smem;
  hipError_t e = prepare_one<K, T, OP, TI, TJ, COLSUM>(p, plan, split, &grid, &smem);
  if (e != hipSuccess) return e;
  auto kernel = rz_gemm_kernel<T, OP, TI, TJ, WI, WJ, NSTAGE, FULL, COLSUM, CLAMP, WK, SHORT>;
  if (smem > 64 * 1024) {
    e = raise_lds_limit(reinterpret_cast<const void*>(kernel), lds_limit_raised);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kernel, grid, dim3(K::kThreads), smem, stream, p);
  return hipGetLastError();
}

// FULL kernels carry no bounds checks: every tile and every R step must be complete.  Ragged
// shapes: the directly staged forms (all but the single-stage one) still
// stage directly, with edge pieces fetched from inside the operands (CLAMP); everything else takes
// the bounds-checked kernel.
template <typename T, int OP, int TILE, int WI, int WJ, int NSTAGE, bool COLSUM = false, int WK = 1, int TILE_J = TILE>
static hipError_t launch_tile(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split,
                              const KernelForm& form, hipStream_t stream) {
  // (the form was derived on the host from the same rules that select the instantiation here:
  //  refuse to launch if the two ever disagree about the step length)
  // A directly staged load addresses the hashed operand by a 32-bit byte offset from its first
  // element: an fp32 hashed_weight of 4 GB and more takes the bounds-checked kernel, whose loads
  // carry full pointers (the step is the same for both fp32 forms).
  const bool far = sizeof(T) == 4 && OP != kWeightGrad &&
                   ((unsigned long long)p.h.range + (unsigned long long)p.h.BK * (unsigned long long)p.h.BN) * sizeof(T) > 0xffffffffull;
  if constexpr (sizeof(T) == 4) if (far) {
    if (form.step != GemmKernel<T, OP, TILE, TILE_J, WI, WJ, NSTAGE, false>::TR) return hipErrorInvalidValue;
    return launch_one<T, OP, TILE, TILE_J, WI, WJ, NSTAGE, false, COLSUM, false, WK>(p, plan, split, stream);
  }
  // (the 64 tile of four wavefronts but for fp32 weight-grad, and the 16-bit 128 tile of eight with two stages, serve rows shorter than a 16-byte piece only)
  // (16-bit 256 tile, a few R steps)
  if constexpr (sizeof(T) == 2 && TILE == 256 && TILE_J == 256) if (form.short_loop) {
    if (form.step != GemmKernel<T, OP, TILE, TILE_J, WI, WJ, NSTAGE, true, false, false, WK, true>::TR) return hipErrorInvalidValue;
    if (form.full) return launch_one<T, OP, TILE, TILE_J, WI, WJ, NSTAGE, true, COLSUM, false, WK, true>(p, plan, split, stream);
    if (form.clamp) return launch_one<T, OP, TILE, TILE_J, WI, WJ, NSTAGE, false, COLSUM, true, WK, true>(p, plan, split, stream);
    return hipErrorInvalidValue;
  }
  constexpr bool kCheckedOnly = WK == 1 && ((TILE == 64 && !(sizeof(T) == 4 && OP == kWeightGrad)) || (sizeof(T) == 2 && TILE == 128 && WI * WJ == 8 && NSTAGE == 2));
  if constexpr (!kCheckedOnly) if (form.full) {
    if (form.step != GemmKernel<T, OP, TILE, TILE_J, WI, WJ, NSTAGE, true>::TR) return hipErrorInvalidValue;
    return launch_one<T, OP, TILE, TILE_J, WI, WJ, NSTAGE, true, COLSUM, false, WK>(p, plan, split, stream);
  }
  constexpr bool kDirectOnly = WI * WJ * WK == 16 || (sizeof(T) == 2 && NSTAGE >= 3);
  if constexpr (NSTAGE >= 2 && !kCheckedOnly) {
    if (form.clamp) {
      if (form.step != GemmKernel<T, OP, TILE, TILE_J, WI, WJ, NSTAGE, false, false, true, WK>::TR) return hipErrorInvalidValue;
      return launch_one<T, OP, TILE, TILE_J, WI, WJ, NSTAGE, false, COLSUM, true, WK>(p, plan, split, stream);
    }
  }
  if constexpr (kDirectOnly) {
    return hipErrorInvalidValue;
  } else {
    if (form.full || form.clamp || form.step != GemmKernel<T, OP, TILE, TILE_J, WI, WJ, NSTAGE, false>::TR) return hipErrorInvalidValue;
    return launch_one<T, OP, TILE, TILE_J, WI, WJ, NSTAGE, false, COLSUM, false, WK>(p, plan, split, stream);
  }
}

template <typename T, int OP, int TILE, int WI, int WJ, int NSTAGE, int WK = 1>
static hipError_t launch_op(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split,
                            const KernelForm& form, hipStream_t stream) {
  if constexpr (OP == kWeightGrad) {
    // with a column-sum target the kernel also produces the bias gradient's partial sums
    if (p.colsum != nullptr) return launch_tile<T, OP, TILE, WI, WJ, NSTAGE, true, WK>(p, plan, split, form, stream);
    return launch_tile<T, OP, TILE, WI, WJ, NSTAGE, false, WK>(p, plan, split, form, stream);
  } else {
    return launch_tile<T, OP, TILE, WI, WJ, NSTAGE, false, WK>(p, plan, split, form, stream);
  }
}

// Tile shapes (all two LDS stages, software pipelined unless noted):
//   256: 256 x 256, eight wavefronts of 128 x 64, one workgroup per compute unit (16-bit: a loop of its own, except for a few R steps)
//   128: 128 x 128, four wavefronts of 64 x 64 (up to two workgroups per compute unit) or
//        eight of 64 x 32 when there is about one workgroup per compute unit (16-bit: four LDS stages); tuning.stages = 1
//        selects a single-stage form that leans on several workgroups per compute unit
//        instead of a pipeline (tuning aid)
//        16-bit forward / input-grad: 256 x 128, eight wavefronts of 64 x 64, three LDS stages, where pairs are faster
//    64:  64 x  64, for problems with few tiles: 16-bit sixteen wavefronts of 32 x 32 in four groups that
//        share every R step between them; fp32 eight, in two such groups; weight-grad of many short loops, and rows shorter than a 16-byte piece, four
//        16-bit forward / input-grad of at most 32 rows: 32 x 128 (eight wavefronts of 32 x 32 in two groups
//        that share every R step, three LDS stages)
//    32:  32 x  64 (fp32 forward / input-grad whose rows would leave a 64-row tile at most half full): four wavefronts of 32 x 32 in two such groups
// 16-bit forward / input-grad in runs (plan_runs), and without counters the kernel that adds the parts up.
template <typename T, int OP, int TJ, int WI, int WJ, int NSTAGE, bool FULL>
static hipError_t launch_runs_form(const GemmParams& p, const SplitPlan& plan, hipStream_t stream) {
  typedef GemmKernel<T, OP, 256, TJ, WI, WJ, NSTAGE, FULL, false, !FULL> K;
  static std::atomic<uint64_t> lds_limit_raised{0}, lds_limit_raised_finish{0};
  auto kernel = rz_gemm_runs_kernel<T, OP, 256, TJ, WI, WJ, NSTAGE, FULL, !FULL, false>;
  auto finish = rz_gemm_runs_kernel<T, OP, 256, TJ, WI, WJ, NSTAGE, FULL, !FULL, true>;
  const size_t smem = sizeof(typename K::Smem);
  hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(kernel), lds_limit_raised);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3((unsigned)plan.run_groups), dim3(K::kThreads), smem, stream, p);
  e = hipGetLastError();
  if (e != hipSuccess || p.finish != nullptr) return e;
  e = raise_lds_limit(reinterpret_cast<const void*>(finish), lds_limit_raised_finish);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(finish, dim3((unsigned)plan.run_tiles), dim3(K::kThreads), smem, stream, p);
  return hipGetLastError();
}

template <typename T, int OP, int TJ, int WI, int WJ, int NSTAGE>
static hipError_t launch_runs(GemmParams p, const SplitPlan& plan, hipStream_t stream) {
  p.tiles_i = (p.I + 255) / 256;
  p.tiles_j = (p.J + TJ - 1) / TJ;
  p.run_steps = plan.run_steps;
  p.run_rounds = plan.run_rounds;
  p.run_groups = plan.run_groups;
  if (p.partial == nullptr || plan.splits > kFinishSlices || plan.run_tiles < 1 || plan.run_tiles > kComputeUnits ||
      (long long)plan.run_rounds * plan.run_groups + plan.run_tiles != (long long)p.tiles_i * p.tiles_j)
    return hipErrorInvalidValue;
  if (p.I % 256 == 0 && p.J % TJ == 0 && p.R % 64 == 0) return launch_runs_form<T, OP, TJ, WI, WJ, NSTAGE, true>(p, plan, stream);
  return launch_runs_form<T, OP, TJ, WI, WJ, NSTAGE, false>(p, plan, stream);
}

template <typename T, int OP>
static hipError_t launch_gemm_t(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split,
                                const rz_tuning& tuning, hipStream_t stream) {
  if constexpr (sizeof(T) == 2 && OP != kWeightGrad) if (split != nullptr && split->run_steps > 0) {
    if (split->tile == 256) return launch_runs<T, OP, 256, 2, 4, 2>(p, *split, stream);
    return launch_runs<T, OP, 128, 4, 2, 3>(p, *split, stream);
  }
  const bool wg = OP == kWeightGrad && plan != nullptr;
  const bool cut = !wg && split != nullptr && split->splits > 1;
  const int tile = wg ? plan->tile : (split != nullptr ? split->tile : pick_tile(p.I, p.J, (int)sizeof(T), tuning));
  const int chunk = wg ? plan->r_chunk : (cut ? split->r_chunk : p.R);
  const long long workgroups = wg ? plan->workgroups : tile_count(p.I, p.J, tile) * (cut ? split->splits : 1);
  const KernelForm form = kernel_form(OP, p.I, p.J, p.R, chunk, tile, workgroups, (int)sizeof(T), tuning, wg && plan->image_pitch > 0);
  if constexpr (sizeof(T) == 2 && OP != kWeightGrad) {
    if (form.rows == 32 && form.cols == 128) return launch_tile<T, OP, 32, 1, 4, 3, false, 2, 128>(p, plan, split, form, stream);
  }
  if constexpr (sizeof(T) == 2 && OP != kWeightGrad) {
    if (form.rows == 256 && form.cols == 128) return launch_tile<T, OP, 256, 4, 2, 3, false, 1, 128>(p, plan, split, form, stream);
  }
  if (form.rows != form.tile || form.cols != tile_cols(form.tile)) return hipErrorInvalidValue;
  switch (form.tile * 1000 + form.waves * 10 + form.stages) {
    case 256082: return launch_op<T, OP, 256, 2, 4, 2>(p, plan, split, form, stream);
    case 64042:
      if constexpr (sizeof(T) == 2 || OP == kWeightGrad) return launch_op<T, OP, 64, 2, 2, 2>(p, plan, split, form, stream);
      return hipErrorInvalidValue;
    case 64164:   // 16-bit, at most one workgroup per compute unit: four groups of four wavefronts share every R step
      if constexpr (sizeof(T) == 2) return launch_op<T, OP, 64, 2, 2, 4, 4>(p, plan, split, form, stream);
      return hipErrorInvalidValue;
    case 64162:   // ... more of them: two LDS stages
      if constexpr (sizeof(T) == 2) return launch_op<T, OP, 64, 2, 2, 2, 4>(p, plan, split, form, stream);
      return hipErrorInvalidValue;
    case 64082:   // fp32: two groups of four wavefronts share every R step
      if constexpr (sizeof(T) == 4) return launch_op<T, OP, 64, 2, 2, 2, 2>(p, plan, split, form, stream);
      return hipErrorInvalidValue;
    case 32042:   // fp32 forward / input-grad, rows in 32s: 32 x 64, two groups of two wavefronts
      if constexpr (sizeof(T) == 4 && OP != kWeightGrad) return launch_tile<T, OP, 32, 1, 2, 2, false, 2, 64>(p, plan, split, form, stream);
      return hipErrorInvalidValue;
    case 128041: return launch_op<T, OP, 128, 2, 2, 1>(p, plan, split, form, stream);
    case 128082: return launch_op<T, OP, 128, 2, 4, 2>(p, plan, split, form, stream);
    case 128084:
      if constexpr (sizeof(T) == 2) return launch_op<T, OP, 128, 2, 4, 4>(p, plan, split, form, stream);
      return hipErrorInvalidValue;
    case 128042: return launch_op<T, OP, 128, 2, 2, 2>(p, plan, split, form, stream);
    default: return hipErrorInvalidValue;
  }
}

// The two kernels of a backward pass in one launch (with column sums: there is none without a bias gradient).  What a boundary between two launches costs a GPU
// that is waiting for it is 4 to 6 us, and the host a launch; where neither op fills the chip their workgroups run side by side as well.  GPU-bound, with what
// finishes dHW (apart / in one launch, us): bf16 M = 78, K = 752, N = 133 17.2 / 11.4; M = 160, K = 448, N = 1216 22.6 / 15.0; M = 6016, K = 3200, N = 1600
// 156 / 135; fp16 M = 3663, K = 13603, N = 1370 360 / 294; fp32 M = 50, K = 1920, N = 192 25.6 / 19.3; fp32 1024^3 through the module, forward included,
// 68.8 / 63.6.  Where it is not faster: backward_form.
template <typename T, int TI, int TJ, int WI, int WJ, int IG_STAGES, int WK, int TILE, int WG_WI, int WG_WJ, int WG_STAGES, int WG_WK, bool FULL>
static hipError_t launch_backward_form(GemmParams ig, const SplitPlan* split, GemmParams wg, const WeightGradPlan* plan, bool wg_first,
                                       hipStream_t stream) {
  static std::atomic<uint64_t> lds_limit_raised{0};
  typedef GemmKernel<T, kInputGrad, TI, TJ, WI, WJ, IG_STAGES, FULL, false, !FULL, WK> IG;
  typedef GemmKernel<T, kWeightGrad, TILE, TILE, WG_WI, WG_WJ, WG_STAGES, FULL, true, !FULL, WG_WK> WG;
  dim3 ig_grid, wg_grid;
  size_t ig_smem, smem;
  hipError_t e = prepare_one<IG, T, kInputGrad, TI, TJ, false>(ig, nullptr, split, &ig_grid, &ig_smem);
  if (e == hipSuccess) e = prepare_one<WG, T, kWeightGrad, TILE, TILE, true>(wg, plan, nullptr, &wg_grid, &smem);
  if (e != hipSuccess) return e;
  if (ig_smem > smem) smem = ig_smem;
  const long long groups = (long long)ig_grid.x * ig_grid.y + (long long)wg_grid.x * wg_grid.y;
  if (groups > 0x7fffffffLL) return hipErrorInvalidValue;
  auto kernel = rz_backward_kernel<IG, WG>;
  if (smem > 64 * 1024) {
    e = raise_lds_limit(reinterpret_cast<const void*>(kernel), lds_limit_raised);
    if (e != hipSuccess) return e;
  }
  const BackwardGrid g = {(int)ig_grid.x, (int)ig_grid.y, (int)wg_grid.x, (int)wg_grid.y, wg_first ? 1 : 0};
  hipLaunchKernelGGL(kernel, dim3((unsigned)groups), dim3(IG::kThreads), smem, stream, ig, wg, g);
  return hipGetLastError();
}

template <typename T, int TI, int TJ, int WI, int WJ, int IG_STAGES, int WK, int TILE, int WG_WI, int WG_WJ, int WG_STAGES, int WG_WK>
static hipError_t launch_backward_pair(const GemmParams& ig, const SplitPlan* split, const GemmParams& wg, const WeightGradPlan* plan,
                                       const BackwardForm& form, hipStream_t stream) {
  if (form.full) return launch_backward_form<T, TI, TJ, WI, WJ, IG_STAGES, WK, TILE, WG_WI, WG_WJ, WG_STAGES, WG_WK, true>(ig, split, wg, plan, form.wg_first, stream);
  return launch_backward_form<T, TI, TJ, WI, WJ, IG_STAGES, WK, TILE, WG_WI, WG_WJ, WG_STAGES, WG_WK, false>(ig, split, wg, plan, form.wg_first, stream);
}

template <typename T>
static hipError_t launch_backward_t(const GemmParams& ig, const SplitPlan* split, const GemmParams& wg, const WeightGradPlan* plan,
                                    const BackwardForm& form, hipStream_t stream) {
  if constexpr (sizeof(T) == 4) {
    if (form.pair == k64With64) return launch_backward_pair<T, 64, 64, 2, 2, 2, 2, 64, 2, 2, 2, 2>(ig, split, wg, plan, form, stream);
  } else {
    switch (form.pair) {
      case k64With64:
        if (form.stages == 4) return launch_backward_pair<T, 64, 64, 2, 2, 4, 4, 64, 2, 2, 4, 4>(ig, split, wg, plan, form, stream);
        return launch_backward_pair<T, 64, 64, 2, 2, 2, 4, 64, 2, 2, 2, 4>(ig, split, wg, plan, form, stream);
      case k64With128: return launch_backward_pair<T, 64, 64, 2, 2, 4, 4, 128, 4, 4, 4, 1>(ig, split, wg, plan, form, stream);
      case kPairWith128: return launch_backward_pair<T, 256, 128, 4, 2, 3, 1, 128, 2, 4, 4, 1>(ig, split, wg, plan, form, stream);
      case kPairWith256: return launch_backward_pair<T, 256, 128, 4, 2, 3, 1, 256, 2, 4, 2, 1>(ig, split, wg, plan, form, stream);
      case k256With256: return launch_backward_pair<T, 256, 256, 2, 4, 2, 1, 256, 2, 4, 2, 1>(ig, split, wg, plan, form, stream);
      case k256With128: return launch_backward_pair<T, 256, 256, 2, 4, 2, 1, 128, 2, 4, 4, 1>(ig, split, wg, plan, form, stream);
      case k128With128: return launch_backward_pair<T, 128, 128, 2, 4, 4, 1, 128, 2, 4, 4, 1>(ig, split, wg, plan, form, stream);
      default: break;
    }
  }
  return hipErrorInvalidValue;
}

// What the kernels that make the fragments take; returns how many there are.  (Blocks of 32 columns up to whole hashed tiles: every unit of
// every tile has its fragments, see window_pack_bytes.)
template <typename T>
static long long pack_params(const WindowParams& w, PackParams* pk) {
  constexpr int kRows = sizeof(T) == 4 ? 8 : 16;
  const long long blocks_x = (long long)w.tiles_k * (w.h.BK / 32), blocks_y = (long long)w.tiles_n * (w.h.BN / 32);
  const long long ngroups = ((long long)w.M + kRows - 1) / kRows;
  *pk = {w.X, w.dY, w.packed_x, w.packed_y, w.M, w.K, w.N, (int)blocks_x, (int)blocks_y, (int)ngroups, w.ldx, w.lddy};
  return (blocks_x + blocks_y) * ngroups;
}

// An input-grad and, in the same launch, the fragments of the weight-grad behind it (pack_groups).
template <typename T, int TI, int TJ, int WI, int WJ, int STAGES, int WK, bool FULL>
static hipError_t launch_pack_form(GemmParams ig, const SplitPlan* split, const PackParams& pk, int groups, hipStream_t stream) {
  static std::atomic<uint64_t> lds_limit_raised{0};
  typedef GemmKernel<T, kInputGrad, TI, TJ, WI, WJ, STAGES, FULL, false, !FULL, WK> IG;
  dim3 grid;
  size_t smem;
  hipError_t e = prepare_one<IG, T, kInputGrad, TI, TJ, false>(ig, nullptr, split, &grid, &smem);
  if (e != hipSuccess) return e;
  auto kernel = rz_input_grad_pack_kernel<T, IG>;
  if (smem > 64 * 1024) {
    e = raise_lds_limit(reinterpret_cast<const void*>(kernel), lds_limit_raised);
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kernel, dim3(grid.x * grid.y + (unsigned)groups), dim3(IG::kThreads), smem, stream, ig, pk, (int)grid.x, (int)grid.y);
  return hipGetLastError();
}

template <typename T, int TI, int TJ, int WI, int WJ, int STAGES, int WK>
static hipError_t launch_pack_tile(const GemmParams& ig, const SplitPlan* split, const PackParams& pk, const PackForm& form, hipStream_t stream) {
  if (form.full) return launch_pack_form<T, TI, TJ, WI, WJ, STAGES, WK, true>(ig, split, pk, form.groups, stream);
  return launch_pack_form<T, TI, TJ, WI, WJ, STAGES, WK, false>(ig, split, pk, form.groups, stream);
}

template <typename T>
static hipError_t launch_input_grad_pack_t(const GemmParams& ig, const SplitPlan* split, const WindowParams& w, const PackForm& form,
                                           hipStream_t stream) {
  PackParams pk;
  if (w.packed_x == nullptr || w.packed_y == nullptr || pack_params<T>(w, &pk) != form.fragments) return hipErrorInvalidValue;
  switch (form.rows) {
    case 32: return launch_pack_tile<T, 32, 128, 1, 4, 3, 2>(ig, split, pk, form, stream);
    case 64: return launch_pack_tile<T, 64, 64, 2, 2, 4, 4>(ig, split, pk, form, stream);
    case 128: return launch_pack_tile<T, 128, 128, 2, 4, 4, 1>(ig, split, pk, form, stream);
    case 256: return launch_pack_tile<T, 256, 128, 4, 2, 3, 1>(ig, split, pk, form, stream);
    default: return hipErrorInvalidValue;
  }
}

template <typename T, int TBN, int OPERANDS, bool WHOLE>
static hipError_t launch_window_whole(WindowParams p, int windows, hipStream_t stream) {
  typedef WindowKernel<T, TBN, OPERANDS, WHOLE> K;
  static_assert(K::kFixedBytes + sizeof(float) * kWindowFloats <= 160 * 1024, "the images of a window do not fit the LDS");
  if (p.window < 4 || p.window > kWindowFloats || (p.window & 3) || windows < 1) return hipErrorInvalidValue;
  if ((long long)windows * p.window < p.H) return hipErrorInvalidValue;
  if (p.h.BN != TBN || !window_tile_supported(p.h.BK, p.h.BN)) return hipErrorInvalidValue;
  auto kernel = rz_window_kernel<T, TBN, OPERANDS, WHOLE>;
  p.images = window_images(p.window);
  const size_t smem = K::kFixedBytes + sizeof(float) * (size_t)p.window * p.images;
  static std::atomic<uint64_t> lds_limit_raised{0};
  if (smem > 64 * 1024) {
    hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(kernel), lds_limit_raised);
    if (e != hipSuccess) return e;
  }
  if (p.windows != windows) return hipErrorInvalidValue;
  const int bias_blocks = p.dbias != nullptr ? (p.N + kWindowBiasCols - 1) / kWindowBiasCols : 0;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(windows + bias_blocks)), dim3(K::kThreads), smem, stream, p);
  return hipGetLastError();
}

template <typename T, int TBN, int OPERANDS>
static hipError_t launch_window_form(const WindowParams& p, int windows, hipStream_t stream) {
  if constexpr (OPERANDS == kPacked)
    if (p.K % p.h.BK == 0 && p.N % TBN == 0) return launch_window_whole<T, TBN, OPERANDS, true>(p, windows, stream);
  return launch_window_whole<T, TBN, OPERANDS, false>(p, windows, stream);
}

// With room for them the operands are laid out as fragments first; else, where their rows hold whole 16-byte pieces, they go
// through the staged form.
template <typename T, int TBN>
static hipError_t launch_window_one(const WindowParams& p, int windows, hipStream_t stream) {
  constexpr int kVec = 16 / (int)sizeof(T);
  if (p.packed_x != nullptr && p.packed_y != nullptr) {
    if (!p.packed) {
      PackParams pk;
      const long long wgs = (pack_params<T>(p, &pk) + 3) / 4;
      if (wgs > 0x1fffffffLL) return hipErrorInvalidValue;
      hipLaunchKernelGGL(window_pack_kernel<T>, dim3((unsigned)wgs), dim3(256), 0, stream, pk);
    }
    hipError_t e = hipGetLastError();
    return e != hipSuccess ? e : launch_window_form<T, TBN, kPacked>(p, windows, stream);
  }
  // (the staged form keeps the byte offsets of a lane's pieces, up to sixteen rows, in 32-bit registers)
  if (p.K % kVec == 0 && p.N % kVec == 0 && p.ldx < (1 << 25) && p.lddy < (1 << 25))
    return launch_window_form<T, TBN, kStaged>(p, windows, stream);
  return launch_window_form<T, TBN, kByElement>(p, windows, stream);
}

template <typename T>
static hipError_t launch_window_t(const WindowParams& p, int windows, hipStream_t stream) {
  if (p.h.BN == 64) return launch_window_one<T, 64>(p, windows, stream);
  if (p.h.BN == 32) return launch_window_one<T, 32>(p, windows, stream);
  if (p.h.BN == 128) return launch_window_one<T, 128>(p, windows, stream);
  return hipErrorInvalidValue;
}

}  // namespace rz
