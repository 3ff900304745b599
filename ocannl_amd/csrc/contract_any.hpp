// Kernel template and launch of the contraction tile for any extents and strides (contract_any.h); instances for bf16
// operands in contract_any.hip, with an fp32 operand in contract_any_f32.hip.
#pragma once
#include <hip/hip_runtime.h>

#include "contract_any.h"
#include "gemm.hpp"

namespace ocannl {
namespace {

struct AnyBatch {
  int nbatch, batches, members;
  int ext[3];
  long a[3], b[3], c[3];      // element strides of the batch digits
};
struct AnyPtrs {
  const void* a[4];
  const void* b[4];
  void* c[4];
  void* c2[4];
  int pairs;                  // a chain into one C (contract_direct.hip only): operands a[i], b[i] in turn
  float* ws;
  OcnAnyEpilogue ep;
};

// K steps in flight ahead (ocn_any_tile): three gained nothing (1777 x 771 x 1001 in bf16, forward and both gradients: 56.3
// us with two, 58.2 with three)
constexpr int kAnyDepth = 2;

// Batch entry z of the launch -> operands.
__device__ __forceinline__ void any_operands(const OcnAnyDesc& d, const AnyBatch& q, const AnyPtrs& p, int z, const void*& a, const void*& b, void*& c,
                                             void*& c2) {
  const int g = q.members > 1 ? z / q.batches : 0;
  int r = z - g * q.batches;
  long ao = 0, bo = 0, co = 0;
  if (q.nbatch > 2) { const int i = r % q.ext[2]; r /= q.ext[2]; ao += i * q.a[2]; bo += i * q.b[2]; co += i * q.c[2]; }
  if (q.nbatch > 1) { const int i = r % q.ext[1]; r /= q.ext[1]; ao += i * q.a[1]; bo += i * q.b[1]; co += i * q.c[1]; }
  if (q.nbatch > 0) { ao += r * q.a[0]; bo += r * q.b[0]; co += r * q.c[0]; }
  a = g == 0 ? p.a[0] : g == 1 ? p.a[1] : g == 2 ? p.a[2] : p.a[3];
  b = g == 0 ? p.b[0] : g == 1 ? p.b[1] : g == 2 ? p.b[2] : p.b[3];
  c = g == 0 ? p.c[0] : g == 1 ? p.c[1] : g == 2 ? p.c[2] : p.c[3];
  c2 = g == 0 ? p.c2[0] : g == 1 ? p.c2[1] : g == 2 ? p.c2[2] : p.c2[3];
  a = static_cast<const char*>(a) + ao * (d.a.bf16 ? 2 : 4);
  b = static_cast<const char*>(b) + bo * (d.b.bf16 ? 2 : 4);
  c = static_cast<char*>(c) + co * (d.c_bf16 ? 2 : 4);
  if (c2) c2 = static_cast<char*>(c2) + co * 2;
}

// Grid: x = tiles of all batch entries, padded to a multiple of eight and dealt so that each XCD (workgroup
// ids go round robin) walks a contiguous range of them -- neighbouring tiles share panels through its L2;
// y = K splits.
template <int BM, int BN, bool A_KC, bool B_KC, bool ABF, bool BBF, bool PARTS>
__device__ __forceinline__ void any_body(const OcnAnyDesc& d, const AnyBatch& q, const AnyPtrs& p) {
  extern __shared__ __align__(16) unsigned char smem_any[];
  const int per = gridDim.x / 8, tiles = d.tiles_m * d.tiles_n;
  const int t = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  const int z = t / tiles, r = t - z * tiles;
  if (z >= q.batches * q.members) return;
  const void *a, *b;
  void *c, *c2;
  any_operands(d, q, p, z, a, b, c, c2);
  float* const ws = d.splits > 1 ? p.ws + (long)z * d.splits * d.M * d.N : nullptr;
  ocn_any_tile<BM, BN, A_KC, B_KC, ABF, BBF, false, kAnyDepth, PARTS>(d, a, b, c, c2, ws, p.ep, r / d.tiles_n, r % d.tiles_n, (int)blockIdx.y, 0, 0, smem_any);
}

template <int BM, int BN, bool A_KC, bool B_KC>
__global__ void __launch_bounds__(256) gemm_bf16_kernel_any(const OcnAnyDesc d, const AnyBatch q, const AnyPtrs p) {
  any_body<BM, BN, A_KC, B_KC, true, true, false>(d, q, p);
}
template <int BM, int BN, bool A_KC, bool B_KC, bool ABF, bool BBF, bool PARTS>
__global__ void __launch_bounds__(256) gemm_f32_kernel_any(const OcnAnyDesc d, const AnyBatch q, const AnyPtrs p) {
  any_body<BM, BN, A_KC, B_KC, ABF, BBF, PARTS>(d, q, p);
}

template <int BM, int BN, bool A_KC, bool B_KC, bool ABF, bool BBF, bool PARTS>
hipError_t go(dim3 grid, const OcnAnyDesc& d, const AnyBatch& q, const AnyPtrs& p, hipStream_t s) {
  constexpr int smem = ocn_any_smem<BM, BN, A_KC, B_KC, ABF, BBF, PARTS>();
  void (*kernel)(OcnAnyDesc, AnyBatch, AnyPtrs);
  if constexpr (ABF && BBF) kernel = gemm_bf16_kernel_any<BM, BN, A_KC, B_KC>;
  else kernel = gemm_f32_kernel_any<BM, BN, A_KC, B_KC, ABF, BBF, PARTS>;
  if (smem > 65536) {
    static thread_local bool configured = false;
    if (!configured) {
      hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
      if (e != hipSuccess) return e;
      configured = true;
    }
  }
  hipLaunchKernelGGL(kernel, grid, dim3(256), smem, s, d, q, p);
  return hipGetLastError();
}

template <int BM, int BN, bool ABF, bool BBF, bool PARTS>
hipError_t launch_layout(bool akc, bool bkc, dim3 grid, const OcnAnyDesc& d, const AnyBatch& q, const AnyPtrs& p, hipStream_t s) {
  if (akc && bkc) return go<BM, BN, true, true, ABF, BBF, PARTS>(grid, d, q, p, s);
  if (akc) return go<BM, BN, true, false, ABF, BBF, PARTS>(grid, d, q, p, s);
  if (bkc) return go<BM, BN, false, true, ABF, BBF, PARTS>(grid, d, q, p, s);
  return go<BM, BN, false, false, ABF, BBF, PARTS>(grid, d, q, p, s);
}

struct AnyShape { int bm, bn, splits; bool parts, direct; };

}  // namespace

// contract_any_f32.hip
hipError_t launch_any_f32(int bm, int bn, bool parts, bool a_bf16, bool b_bf16, bool akc, bool bkc, dim3 grid, const OcnAnyDesc& d, const void* q, const void* p,
                          hipStream_t s);
// contract_direct.hip: 32 x 32 tiles of regular operands
hipError_t launch_direct(bool akc, bool bkc, dim3 grid, const OcnAnyDesc& d, const void* q, const void* p, hipStream_t s);

}  // namespace ocannl
