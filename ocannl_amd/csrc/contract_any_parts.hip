// Contractions of any extents and strides: instances that multiply an fp32 operand in bf16 parts.
#include <hip/hip_runtime.h>

#include "contract_any_f32.hpp"

namespace ocannl {

hipError_t launch_any_parts(int bm, int bn, bool a_bf16, bool b_bf16, bool akc, bool bkc, dim3 grid, const OcnAnyDesc& d, const void* qp, const void* pp,
                            hipStream_t s) {
  return any_f32_shape<true>(bm, bn, a_bf16, b_bf16, akc, bkc, grid, d, *static_cast<const AnyBatch*>(qp), *static_cast<const AnyPtrs*>(pp), s);
}

}  // namespace ocannl
