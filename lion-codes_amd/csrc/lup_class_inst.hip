// lup_class_inst.hip -- one class kernel (lup_class.hpp) for one fused
// variant.  The build compiles this file once per (variant, class), so the
// class kernels -- each holding the fully unrolled code of up to 24 sizes --
// compile in parallel; each object registers its kernel in g_class at load
// time.
#include "lup_class.hpp"
#include "lup_dispatch.hpp"

#if !defined(LUFQHE_VARIANT) || !defined(LUFQHE_CLASS)
#error "compile with -DLUFQHE_VARIANT=v (0 or 1) -DLUFQHE_CLASS=c"
#endif

namespace lufqhe {
namespace {

constexpr int kPolicy = variant_policy(LUFQHE_VARIANT);
static_assert(variant_arith(LUFQHE_VARIANT) == ARITH_FUSED, "class kernels are fused only");

hipError_t launch(const ClassArgs& ca, int64_t blocks, hipStream_t stream) {
  hipLaunchKernelGGL((lup_class_kernel<LUFQHE_CLASS, kPolicy>), dim3((unsigned)blocks), dim3(64),
                     0, stream, ca);
  return hipGetLastError();
}

struct Registrar {
  Registrar() { g_class[LUFQHE_VARIANT][LUFQHE_CLASS] = &launch; }
};
Registrar registrar;

}  // namespace
}  // namespace lufqhe
