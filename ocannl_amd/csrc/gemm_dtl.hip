// Instances of the direct-to-LDS contraction kernel (gemm_dtl.hpp), in a translation unit of their own
// so that they compile beside the register-staged kernels of gemm.hip.
#include <hip/hip_runtime.h>

#include "gemm.hpp"
#include "gemm_common.hpp"
#include "gemm_dtl.hpp"

namespace ocannl {
hipError_t launch_gemm_dtl(int bm, int bn, int bk, int ns, bool akc, bool bkc, const GemmArgs& a, hipStream_t s, hipEvent_t ev) {
  if (bm == 256 && bn == 256 && bk == 32 && ns == 4) return launch_dtl_steps<256, 256, 32, 4, false>(akc, bkc, a, s, ev);
  if (bm == 128 && bn == 64 && bk == 32 && ns == 4) return launch_dtl_steps<128, 64, 32, 4, false>(akc, bkc, a, s, ev);
  if (bm == 128 && bn == 128 && bk == 64 && ns == 5) return launch_dtl_steps<128, 128, 64, 5, false>(akc, bkc, a, s, ev);
  if (bm == 128 && bn == 128 && bk == 32 && ns == 4) return launch_dtl_steps<128, 128, 32, 4, false>(akc, bkc, a, s, ev);
  // (two steps of K, which is all the pipeline itself: no turn of its loop)
  if (bm == 128 && bn == 128 && bk == 32 && ns == 3 && a.K == 64 && a.splits == 1) return launch_dtl_layout<128, 128, 32, 3, false, false>(akc, bkc, a, s, ev);
  return hipErrorInvalidValue;
}

}  // namespace ocannl
