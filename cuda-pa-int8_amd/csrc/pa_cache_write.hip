// Launcher of the fp16 paged-cache write: no quantization, only the placement
// (the kernel and its semantics are in pa_write_kernel.hpp).
#include "pa_internal.hpp"
#include "pa_write_kernel.hpp"

namespace pa {

hipError_t launch_cache_write_f16(const WriteLaunch& l) {
  switch (l.head_dim) {
#define PA_CASE(D) \
  case D: return launch_write<D, WriteMode::kF16, false>(l);
    PA_FOR_EACH_HEAD_DIM(PA_CASE)
#undef PA_CASE
    default: return hipErrorInvalidValue;
  }
}

}  // namespace pa
