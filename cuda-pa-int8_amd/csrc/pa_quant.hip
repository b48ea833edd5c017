// Launcher of the INT8 quantize + paged-cache write for one scale mode and input
// type (the kernel and its semantics are in pa_write_kernel.hpp).  Compiled
// once per variant with -DPA_QUANT_GIVEN=0/1 (per-token scales, or one given
// scale per tensor) and -DPA_QUANT_BF16=0/1.
#include "pa_internal.hpp"
#include "pa_write_kernel.hpp"

#if !defined(PA_QUANT_GIVEN) || !defined(PA_QUANT_BF16)
#error "PA_QUANT_GIVEN and PA_QUANT_BF16 must be defined"
#endif

namespace pa {

template <>
hipError_t launch_quant_write_i8<PA_QUANT_GIVEN, PA_QUANT_BF16>(const WriteLaunch& l) {
  constexpr WriteMode kMode = PA_QUANT_GIVEN ? WriteMode::kGivenScale : WriteMode::kTokenScale;
  switch (l.head_dim) {
#define PA_CASE(D) \
  case D: return launch_write<D, kMode, PA_QUANT_BF16>(l);
    PA_FOR_EACH_HEAD_DIM(PA_CASE)
#undef PA_CASE
    default: return hipErrorInvalidValue;
  }
}

}  // namespace pa
