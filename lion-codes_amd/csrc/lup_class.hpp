// lup_class.hpp -- one launch for a range of sizes (mixed batches, serving).
//
// The sizes are cut into classes of similar register demand.  A class kernel
// holds every size of its class, and its grid is the tasks of all the
// class's buckets, largest n first: a workgroup finds its bucket from its
// index and runs that size's code (det_task or panel_task, the code of the
// per-size kernels, so the bits are the same).  One launch takes the place of
// one per size for sizes too few to fill the device by themselves: no kernel
// waits for the tail of the one before it on its stream, and the small sizes
// fill the end of the large ones.
//
// The cuts lie where the per-size kernels change occupancy, since a class
// kernel has the register allocation of its largest size: n <= 8 leaves
// three waves per SIMD, 9..16, 17..32 and 33..56 two, 57..64 one.
#pragma once

#include "lup_kernel.hpp"
#include "lup_panel.hpp"

namespace lufqhe {

constexpr int kClasses = 5;
constexpr int kClassLo[kClasses] = {1, 9, 17, 33, 57};
constexpr int kClassHi[kClasses] = {8, 16, 32, 56, 64};
constexpr int kClassOcc[kClasses] = {3, 2, 2, 2, 1};
constexpr int kMaxClassSizes = 24;

constexpr int size_class(int n) {
  int c = 0;
  while (c + 1 < kClasses && n > kClassHi[c]) ++c;
  return c;
}

// The tile each size runs with inside its class kernel: the shapes the
// autotuner chose on MI355X.  Fixed at compile time; any shape gives the
// same bits.
constexpr ShapeLC class_shape(int n) {
  if (n <= 8) return {4, 1, 1, false};
  if (n <= 16) return {8, 1, 1, false};
  if (n <= 24 && n != 23) return {16, 2, 2, false};
  if (n <= 32) return {32, 4, 2, true};
  return {64, 4, 2, true};
}
constexpr int class_group(int n) { return 64 / class_shape(n).lanes; }  // matrices per task

constexpr int class_task_lds(int n) {
  const ShapeLC s = class_shape(n);
  return s.panel ? panel_lds(n, 64 / s.lanes, 1) : (64 / s.lanes) * group_lds(n, s.lanes, s.lane_cols);
}
constexpr int class_lds(int lo, int hi) {
  int m = 0;
  for (int n = lo; n <= hi; ++n) m = class_task_lds(n) > m ? class_task_lds(n) : m;
  return m;
}

// A class launch: the arguments its buckets share, and per bucket its size,
// its first task and its matrices' place in the index tables (args.offs,
// args.out_idx and args.perm_offs, each given).
struct ClassArgs {
  BatchArgs args;
  int32_t nbuckets;
  int32_t n[kMaxClassSizes];
  int32_t task[kMaxClassSizes];
  int64_t first[kMaxClassSizes];
  int64_t count[kMaxClassSizes];
};

template <int LO, int HI, int POLICY>
__device__ __forceinline__ void class_dispatch(int n, const BatchArgs& args, int64_t task,
                                               double2* __restrict__ lds, int lane) {
  if constexpr (LO == HI) {
    constexpr ShapeLC s = class_shape(LO);
    // a lane id of this size's own, so that nothing computed from it is
    // shared with the other sizes and held from the dispatch on
    asm volatile("" : "+v"(lane));
    if constexpr (s.panel)
      panel_task<LO, 64 / s.lanes, 1, POLICY>(args, task, lds, lane, 0);
    else
      det_task<LO, s.lanes, s.lane_cols, POLICY, ARITH_FUSED>(args, task, lds, lane);
  } else {
    constexpr int MID = (LO + HI) / 2;
    if (n <= MID)
      class_dispatch<LO, MID, POLICY>(n, args, task, lds, lane);
    else
      class_dispatch<MID + 1, HI, POLICY>(n, args, task, lds, lane);
  }
}

template <int CLASS, int POLICY>
__global__ void __launch_bounds__(64, kClassOcc[CLASS]) lup_class_kernel(ClassArgs ca) {
  constexpr int LO = kClassLo[CLASS], HI = kClassHi[CLASS];
  static_assert(HI - LO + 1 <= kMaxClassSizes, "sizes of a class");
  __shared__ double2 lds[class_lds(LO, HI)];
  // the last bucket that starts at or before this task
  const int t = (int)blockIdx.x;
  int b = 0;
#pragma unroll
  for (int step = 16; step > 0; step >>= 1)
    if (b + step < ca.nbuckets && t >= ca.task[b + step]) b += step;
  BatchArgs a = ca.args;
  const int64_t first = ca.first[b];
  a.count = ca.count[b];
  a.ld = ca.n[b];
  a.offs += first;
  a.out_idx += first;
  if (a.perm_offs) a.perm_offs += first;
  class_dispatch<LO, HI, POLICY>(ca.n[b], a, t - ca.task[b], lds, (int)(threadIdx.x & 63));
}

}  // namespace lufqhe
