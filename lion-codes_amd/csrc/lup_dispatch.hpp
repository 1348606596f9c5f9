// lup_dispatch.hpp -- launch tables filled by the per-shard instantiation
// units (lup_inst.hip compiled once per kernel variant and shard).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lup_class.hpp"
#include "lup_kernel.hpp"

namespace lufqhe {

// Kernel variants compiled into the library.
//   0: CROUT_REF pivots, fused FP64 arithmetic (production default)
//   1: ABS pivots, fused FP64 arithmetic
//   2: CROUT_REF pivots, the reference's own formulas (bit-exact parity mode)
constexpr int kNumVariants = 3;
constexpr int variant_policy(int v) { return v == 1 ? POLICY_ABS : POLICY_CROUT_REF; }
constexpr int variant_arith(int v) { return v == 2 ? ARITH_REF : ARITH_FUSED; }
inline int variant_of(int policy, int arith) {
  if (policy == POLICY_CROUT_REF && arith == ARITH_FUSED) return 0;
  if (policy == POLICY_ABS && arith == ARITH_FUSED) return 1;
  if (policy == POLICY_CROUT_REF && arith == ARITH_REF) return 2;
  return -1;
}

constexpr int kMaxN = 64;

// Launch shape of one (variant, n) kernel: `lanes` lanes per matrix split into
// `lane_cols` lane-columns, WPB waves per workgroup.  The kernel is compiled
// for exactly one shape.
struct KernelShape {
  int lanes;
  int lane_cols;
  int waves_per_block;
  int min_waves;  // waves per SIMD the register allocation allows at least
  bool panel;     // lup_panel_kernel, else lup_det_kernel
};

// Launches the (variant, n) kernel on `blocks` workgroups.
using BatchLaunch = hipError_t (*)(const BatchArgs&, int64_t blocks,
                                   hipStream_t stream);

struct KernelEntry {
  BatchLaunch launch;
  KernelShape shape;
  const void* kernel;  // for occupancy queries
};

// g_kernels[variant][n][shape]: the fused variants carry every candidate
// shape of candidate_shape(); the reference-arithmetic variant only shape 0.
extern KernelEntry g_kernels[kNumVariants][kMaxN + 1][kMaxShapes];

// Shape chosen per (variant, n); 0 until the autotuner's table is applied.  A
// choice other than the default (the table's) is pinned: it runs uniform
// batches of every size.
int selected_shape(int variant, int n);
bool shape_pinned(int variant, int n);

// Class kernels (lup_class.hpp), one per fused variant (0: CROUT_REF, 1: ABS)
// and size class, filled by lup_class_inst.hip.
using ClassLaunch = hipError_t (*)(const ClassArgs&, int64_t blocks, hipStream_t stream);
constexpr int kClassVariants = 2;
extern ClassLaunch g_class[kClassVariants][kClasses];

// Uniform batches that leave SIMDs idle are bound by one matrix's latency.
// They run the panel kernel with one matrix per wave (n = 17..32: the pivot
// row by v_readlane instead of LDS, and half the row slots) or two waves per
// matrix (n >= 49: the trailing columns split between them).  Measured, us a
// launch, against the selected shape: n = 17 9.1 / 13.5, n = 24 11.3 / 20.7,
// n = 32 15.1 / 18.3, n = 56 29.2 / 36.1, n = 64 34.9 / 42.2 at 48 matrices;
// n = 32 17.2 / 19.5 at 1024 and 23.5 / 22.4 at 2048; n = 64 35.4 / 42.6 at 256 and
// 48.7 / 44.1 at 512.  At n = 33..48 two waves gained at most 9% and lost at
// 512 matrices.  n <= 16 has no such route.  Measured there, us a call back to
// back, {8,1,1} / {16,1,1} / panel kernel with one / two matrices per wave: n =
// 16 13.0 / 10.4 / 10.4 / 10.3 at 2 matrices, 13.1 / 10.4 / 10.6 / 10.4 at 1000,
// 14.7 / 14.1 / 18.1 / 13.5 at 4096, 17.0 / 18.5 / 31.0 / 19.6 at 8192; n =
// 8..12 10.1 to 10.9 with any of them up to 4096, which is the host's time of a
// call (the kernels take 6.5 to 9.7, the panel ones 4.9 to 7.3 up to 1000).
constexpr int small_waves(int n) { return n < 17 ? 0 : n <= 32 ? 1 : n <= 48 ? 0 : 2; }
constexpr bool small_batch(int n, int64_t count, int cus) {
  return count <= (n <= 32 ? 4 : 1) * (int64_t)cus;
}
constexpr int64_t kSmallMost = 4 * 256;  // no larger batch is small on this architecture
using SmallLaunch = hipError_t (*)(const BatchArgs&, hipStream_t stream);
extern SmallLaunch g_small[kClassVariants][kMaxN + 1];

// Whether a launch of `blocks` one-wave workgroups fills the device's wave
// slots at two waves per SIMD.  From there on a size's own kernel wins, below
// it a launch shared with other sizes of the class: with all of a batch of one
// size the class kernels take 2-5% longer (n <= 32), 5-7% (n = 36..48), 6-15%
// (n = 57..64) and only at n = 52 and 56 no longer, but 32768 matrices of n =
// 10..40 in 31 launches on four streams took 298 us and in shared ones 238.
constexpr bool fills_device(int64_t blocks, int cus) { return blocks >= (int64_t)cus * 8; }

// One class launch being put together: the buckets of its class, added
// largest n first.
struct ClassBatch {
  static constexpr int64_t kMostTasks = (int64_t{1} << 26) - 1;  // 64 threads each: a grid holds 2^32
  int cls = 0;
  int64_t tasks = 0;
  ClassArgs ca{};

  // A size that shares with no other runs its own kernel: the class kernel
  // takes longer for it (graph replay of one size, us, class | own: 1000 x
  // n = 24 26.0 | 25.1, 1900 x n = 57 101 | 93, 1900 x n = 64 115 | 109) and
  // there is no launch to save.
  bool alone() const { return ca.nbuckets == 1; }

  // Matrices first .. first+count-1 of the index tables have side n: how many
  // of them the launch takes (whole tasks, up to its grid's limit).
  int64_t add(int n, int64_t first, int64_t count) {
    const int g = class_group(n);
    const int64_t room = (kMostTasks - tasks) * g;
    if (count > room) count = room;
    if (count <= 0) return 0;
    const int b = ca.nbuckets++;
    ca.n[b] = n;
    ca.task[b] = (int32_t)tasks;
    ca.first[b] = first;
    ca.count[b] = count;
    tasks += (count + g - 1) / g;
    return count;
  }
  hipError_t launch(int variant, const BatchArgs& args, hipStream_t s) const {
    ClassArgs a = ca;
    a.args = args;
    return g_class[variant][cls](a, tasks, s);
  }
};

}  // namespace lufqhe
