// Launch interface of the hand-written CDNA4 MFMA contraction kernels (gemm.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "plan.hpp"

namespace ocannl {

// Device-side view of one strided-batched contraction.
struct GemmArgs {
  const void* a;
  const void* b;
  void* c;
  int64_t M, N, K;
  int64_t a_row, a_k, b_row, b_k, c_row;   // element strides; C is unit-stride along N
  int nbatch;
  int64_t batch_ext[3];
  int64_t a_batch[3], b_batch[3], c_batch[3];
  int accumulate;    // beta = 1
  int c_is_bf16;
  int xcd_m;         // tile-grid rows of the XCD partition (set by launch_gemm; 0: none)
  int member_xcds;   // > 0: every member of a grouped launch keeps to this many XCDs of its own (set by launch_gemm)
  int splits;        // split-K factor (set by launch_gemm)
  float* ws;         // split-K workspace [batch][split][M][N] (set by launch_gemm)
  // One launch may cover up to four independent contractions of identical shapes, strides and
  // precisions: member g > 0 uses a_more / b_more / c_more[g - 1], and the grid's z axis is
  // member * batches + batch.
  int ngroups;       // >= 1
  // A chain `c =+ a_p * b_p` into the same C (bf16 operands): K runs over a / b, then over
  // a_more[p - 1] / b_more[p - 1].  Never together with ngroups > 1.
  int npairs;        // >= 1
  int batches;       // product of batch_ext (set by launch_gemm)
  const void* a_more[3];
  const void* b_more[3];
  void* c_more[3];
  // When not null: a bf16 tensor of C's shape that receives the rounded result at the same element
  // offsets (C must be fp32).  It feeds later bf16 contractions that read C.
  void* c2;
  void* c2_more[3];
  // Epilogue fusion (bf16 C, no accumulation, no K split): when `bias` is not null the stored value is
  // bf16(bf16(acc) + bias[n]) (bias: bf16, indexed by the column); when `relu_out` is not null, relu of
  // the stored value also goes to that tensor at the same element offsets; with `relu_c` set the stored
  // value itself is the relu (C is the only tensor written).
  const void* bias;
  void* relu_out;
  int relu_c;
};

// Picks the kernel instance for the operand precisions / layouts and launches it on `stream`.
// Returns hipErrorInvalidValue for a combination the planner should not have produced.
// `workspace` must hold gemm_workspace_bytes(desc) bytes (may be null when that is 0).
// `after_main`, when not null, is recorded on the stream right after the contraction kernel itself
// (before the split-K reduction, if one follows), for per-kernel timing.
hipError_t launch_gemm(const GemmDesc& desc, const GemmArgs& args, void* workspace, hipStream_t stream,
                       hipEvent_t after_main = nullptr);

// Bytes of split-K workspace this contraction needs (0 when K is not split).
size_t gemm_workspace_bytes(const GemmDesc& desc);

// Direct-to-LDS kernel with one sub-step a step: is the number of K steps of a split (a whole number each) beyond the last
// ns - 1 odd?  It runs them in pairs.
constexpr bool dtl_odd(int64_t bk, int64_t ns, int64_t K, int64_t splits, int64_t pairs) { return bk == 32 && (K / bk / splits * pairs - (ns - 1)) % 2 != 0; }

// Name of the instance launch_gemm would pick (for kernel_info and profiles).
const char* gemm_kernel_name(const GemmDesc& desc);

// Is this contraction, which the kernels of gemm.hip could take, faster as one of any shape (contract_any.hip)?  `room`:
// bytes of workspace that keep the routine's scratch within what ocannl_hip_routine_run_static_scratch has.
bool gemm_prefers_any(const GemmDesc& desc, uint64_t room);
// Makes it one of any shape: extents and strides as digits.
void as_any_shape(GemmDesc& desc);

// Least K at which an fp32 operand of a contraction of any shape is multiplied in bf16 parts, and the same where no compute
// unit has a second tile: below, what parts save is less than what they cost, a vote on whether to multiply again (260 x 132
// x 16 4.4 us as fp32, 5.2 in parts).  2001 x 2001 x 130 (1024 tiles) 22 to 25 us as fp32, 20 to 21 in parts; 1023 x 1023 (256) x 130
// 8.6 to 9.5 and 8.8 to 9.8, x 198 10.6 to 11.9 and 10.5 to 11.7, x 300 13.8 to 16.1 and 12.2 to 13.8.
constexpr int64_t kPartsFrom = 129, kPartsFromAlone = 193;

// contract_any.hip: the same for contractions with `desc.any` set (launch_gemm and its siblings forward to these).
// Do the extents and the element offsets within one batch entry fit the 32-bit arithmetic of contract_any.h?
bool contract_any_fits(const GemmDesc& desc);
// Elements of C, padding included, that a compute unit works on per k in staged tiles, with the workgroups dealt out evenly and K split as
// it would be; `alone`: no unit gets a second workgroup.
int64_t contract_any_area(const GemmDesc& desc, bool& alone);
// Is it few enough tiles for contract_direct.hip?
bool contract_any_direct(const GemmDesc& desc);
// One whose K splits would take more workspace than `room` goes unsplit to the tiles of contract_direct.hip, if they are few
// enough.
void contract_any_settle(GemmDesc& desc, uint64_t room);
hipError_t launch_contract_any(const GemmDesc& desc, const GemmArgs& args, void* workspace, hipStream_t stream, hipEvent_t after_main);
size_t contract_any_workspace_bytes(const GemmDesc& desc);
const char* contract_any_name(const GemmDesc& desc);

}  // namespace ocannl
