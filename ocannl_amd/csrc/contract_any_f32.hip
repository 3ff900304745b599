// Contractions of any extents and strides: instances with an fp32 operand that multiply it as it is, and the choice between
// these and those that multiply its bf16 parts (contract_any_parts.hip).
#include <hip/hip_runtime.h>

#include "contract_any_f32.hpp"

namespace ocannl {

// contract_any_parts.hip
hipError_t launch_any_parts(int bm, int bn, bool a_bf16, bool b_bf16, bool akc, bool bkc, dim3 grid, const OcnAnyDesc& d, const void* qp, const void* pp,
                            hipStream_t s);

hipError_t launch_any_f32(int bm, int bn, bool parts, bool a_bf16, bool b_bf16, bool akc, bool bkc, dim3 grid, const OcnAnyDesc& d, const void* qp,
                          const void* pp, hipStream_t s) {
  if (parts) return launch_any_parts(bm, bn, a_bf16, b_bf16, akc, bkc, grid, d, qp, pp, s);
  return any_f32_shape<false>(bm, bn, a_bf16, b_bf16, akc, bkc, grid, d, *static_cast<const AnyBatch*>(qp), *static_cast<const AnyPtrs*>(pp), s);
}

}  // namespace ocannl
