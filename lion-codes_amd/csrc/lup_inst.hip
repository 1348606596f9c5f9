// lup_inst.hip -- explicit kernel instantiations for one variant and one
// shard of the sizes n = 1..64 (n % LUFQHE_SHARDS == LUFQHE_SHARD).  The
// build compiles this file once per (variant, shard) so the 192 fully
// unrolled kernels compile in parallel; each object registers its kernels in
// g_kernels at load time.
#include <utility>

#include "lup_dispatch.hpp"
#include "lup_kernel.hpp"
#include "lup_panel.hpp"

#if !defined(LUFQHE_VARIANT) || !defined(LUFQHE_SHARD) || !defined(LUFQHE_SHARDS)
#error "compile with -DLUFQHE_VARIANT=v -DLUFQHE_SHARD=s -DLUFQHE_SHARDS=k"
#endif

namespace lufqhe {
namespace {

constexpr int kPolicy = variant_policy(LUFQHE_VARIANT);
constexpr int kArith = variant_arith(LUFQHE_VARIANT);
// One wave per workgroup: measured 3-11% faster than 2 or 4 on MI355X
// (finer-grained placement of the waves as others finish).
constexpr int kWavesPerBlock = 1;

template <int N, int SH>
constexpr ShapeLC shape_of() {
  return kArith == ARITH_FUSED ? candidate_shape(N, SH) : reference_shape(N);
}

template <int N, int SH>
constexpr auto kernel_of() {
  constexpr ShapeLC sh = shape_of<N, SH>();
  if constexpr (sh.panel)
    return &lup_panel_kernel<N, 64 / sh.lanes, 1, kPolicy, sh.waves>;
  else
    return &lup_det_kernel<N, sh.lanes, sh.lane_cols, kPolicy, kArith, kWavesPerBlock, sh.waves>;
}

template <int N, int SH>
hipError_t launch(const BatchArgs& args, int64_t blocks, hipStream_t stream) {
  hipLaunchKernelGGL((kernel_of<N, SH>()), dim3((unsigned)blocks), dim3(64 * kWavesPerBlock), 0,
                     stream, args);
  return hipGetLastError();
}

template <int N, int SH>
void register_shape() {
  constexpr ShapeLC sh = shape_of<N, SH>();
  // reference arithmetic is a parity mode: only one shape is built
  if constexpr (sh.lanes > 0 && (kArith == ARITH_FUSED || SH == 0)) {
    static_assert(!sh.panel || (sh.lanes == 64 / panel_groups(N) && sh.lane_cols == 4),
                  "the panel kernel's geometry");
    KernelEntry& e = g_kernels[LUFQHE_VARIANT][N][SH];
    e.launch = &launch<N, SH>;
    e.shape = KernelShape{sh.lanes, sh.lane_cols, kWavesPerBlock, sh.waves, sh.panel};
    e.kernel = reinterpret_cast<const void*>(kernel_of<N, SH>());
  }
}

// The kernel of a small batch (small_batch in lup_dispatch.hpp).
template <int N>
hipError_t launch_small(const BatchArgs& args, hipStream_t stream) {
  constexpr int H = small_waves(N);
  hipLaunchKernelGGL((lup_panel_kernel<N, 1, H, kPolicy, 2>), dim3((unsigned)args.count),
                     dim3(64 * H), 0, stream, args);
  return hipGetLastError();
}

template <int N>
void register_one() {
  if constexpr (N % LUFQHE_SHARDS == LUFQHE_SHARD) {
    if constexpr (kArith == ARITH_FUSED && small_waves(N) > 0)
      g_small[LUFQHE_VARIANT][N] = &launch_small<N>;
    register_shape<N, 0>();
    register_shape<N, 1>();
    register_shape<N, 2>();
    register_shape<N, 3>();
  }
}

template <int... I>
void register_all(std::integer_sequence<int, I...>) {
  (register_one<I + 1>(), ...);
}

struct Registrar {
  Registrar() { register_all(std::make_integer_sequence<int, kMaxN>{}); }
};
Registrar registrar;

}  // namespace
}  // namespace lufqhe
