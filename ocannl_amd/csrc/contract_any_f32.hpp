// The instance of the contraction tile for any shape that a tile with an fp32 operand takes.
#pragma once
#include "contract_any.hpp"

namespace ocannl {
namespace {

template <bool PARTS>
hipError_t any_f32_shape(int bm, int bn, bool a_bf16, bool b_bf16, bool akc, bool bkc, dim3 grid, const OcnAnyDesc& d, const AnyBatch& q,
                         const AnyPtrs& p, hipStream_t s) {
  if (a_bf16) return launch_layout<64, 64, true, false, PARTS>(akc, bkc, grid, d, q, p, s);
  if (b_bf16) return launch_layout<64, 64, false, true, PARTS>(akc, bkc, grid, d, q, p, s);
  if (bn == 32) return launch_layout<128, 32, false, false, PARTS>(akc, bkc, grid, d, q, p, s);
  if (bm == 32) return launch_layout<32, 128, false, false, PARTS>(akc, bkc, grid, d, q, p, s);
  if (bm == 128) return launch_layout<128, 128, false, false, PARTS>(akc, bkc, grid, d, q, p, s);
  return launch_layout<64, 64, false, false, PARTS>(akc, bkc, grid, d, q, p, s);
}

}  // namespace
}  // namespace ocannl
