// Contractions of any extents and strides: instances with an fp32 operand (exact products, fp32 matrix cores).
#include <hip/hip_runtime.h>

#include "contract_any.hpp"

namespace ocannl {

hipError_t launch_any_f32(int bm, int bn, bool a_bf16, bool b_bf16, bool akc, bool bkc, dim3 grid, const OcnAnyDesc& d, const void* qp, const void* pp,
                          hipStream_t s) {
  const AnyBatch& q = *static_cast<const AnyBatch*>(qp);
  const AnyPtrs& p = *static_cast<const AnyPtrs*>(pp);
  if (a_bf16) return launch_layout<64, 64, true, false>(akc, bkc, grid, d, q, p, s);
  if (b_bf16) return launch_layout<64, 64, false, true>(akc, bkc, grid, d, q, p, s);
  if (bn == 32) return launch_layout<128, 32, false, false>(akc, bkc, grid, d, q, p, s);
  if (bm == 32) return launch_layout<32, 128, false, false>(akc, bkc, grid, d, q, p, s);
  if (bm == 128) return launch_layout<128, 128, false, false>(akc, bkc, grid, d, q, p, s);
  return launch_layout<64, 64, false, false>(akc, bkc, grid, d, q, p, s);
}

}  // namespace ocannl
