// The direct-to-LDS contraction kernel (gemm_dtl.hpp) for chains: several operand pairs into one C, in a translation unit of
// its own so that it compiles beside gemm_dtl.hip.
#include <hip/hip_runtime.h>

#include "gemm.hpp"
#include "gemm_common.hpp"
#include "gemm_dtl.hpp"

namespace ocannl {

hipError_t launch_gemm_dtl_chain(int bm, int bn, int bk, int ns, bool akc, bool bkc, const GemmArgs& a, hipStream_t s, hipEvent_t ev) {
  if (bm == 128 && bn == 128 && bk == 64 && ns == 5) return launch_dtl_steps<128, 128, 64, 5, true>(akc, bkc, a, s, ev);
  if (bm == 128 && bn == 128 && bk == 32 && ns == 4) return launch_dtl_steps<128, 128, 32, 4, true>(akc, bkc, a, s, ev);
  return hipErrorInvalidValue;
}

}  // namespace ocannl
