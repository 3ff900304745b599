// fp32 contractions on the bf16 matrix cores: both operands fp32, products as good as fp32 ones.
//
// An fp32 value is the sum of three bf16 values (8 significant bits each: hi, then mid and lo of what is left,
// rounded to nearest), exactly.  Of the nine products of two such sums the six largest make up the product of the
// values to 2^-24 of its size at most (the three left out: mid lo, lo mid, lo lo), and the matrix cores sum sixteen k
// of one of them in one rounding: the sum over K goes through 6 K / 16 roundings where v_mfma_f32_32x32x2_f32
// goes through K.  Measured against fp64 (2-norm), uniform values: K = 16: 3.2e-8 (fp32 instructions 7.3e-8),
// 64: 1.1e-7 (1.4e-7), 1024: 4.7e-7 (5.6e-7), 4096: 1.00e-6 (1.18e-6); positive values, K = 4096: 5.3e-7 (8.4e-7);
// values spread over e^(3 sigma): 7.0e-7 (1.41e-6).
//
// Both operands are taken 2^23 times as large and the sums 2^-46 times: no part of any fp32 value, subnormal ones included, is
// then a subnormal bf16, next to which the matrix cores keep fewer bits of a product.  What that does not cover is
// multiplied again with fp32 instructions, tile by tile: results that are not finite -- an infinity has no remainder, and
// sums from 2^81 on and values from 2^104 on overflow.  That pass hides nothing: 4096 x 4096 x 4096 with such a value in
// every tile 1.62 ms, 0.63 without one, 1.04 where all tiles ran on fp32 instructions.
//
// What bounds it: the matrix cores: 8192 x 4096 x 4096 in 1.36 ms is 1.21 PFLOP/s of bf16 products, 202 TFLOP/s of fp32
// ones; they are busy in 62 % of the cycles, a loop of their instruction alone sustains 1.76 PFLOP/s on normally distributed
// operands and a library's bf16 product of 8192^3 1.48; with v_mfma_f32_32x32x2_f32, which this replaces, 2.12 ms,
// 82 % of what that instruction can do.  One operand row-contiguous 1.38 (2.18), both, 4096 x 4096 x 8192: 1.36 (2.16);
// 2048 x 2048 x 2048 on 128 x 128 tiles 120 us (174).  A step moves 48 KB into LDS and 96 KB of fragments out of it in
// the 3072 cycles of its products, and splits 32 values a thread in about 210 vector instructions: room enough beside
// the products, so the tile converts its values itself and no pass over the operands does.
// Four wavefronts of 128 x 128, one to a SIMD; eight of 128 x 64 read more fragments: forward and both gradients of the
// first product 3.83 ms against 3.75.
#include <hip/hip_runtime.h>

#include "gemm.hpp"
#include "gemm_common.hpp"

namespace ocannl {
namespace {

constexpr int kSK = 16;          // k of a step: one matrix instruction per product
constexpr float kScale = 0x1p23f, kUnscale = 0x1p-46f;

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// ROWS x kSK tile of one operand by T threads, in chunks of four along whichever of k and the row is contiguous.  Rows
// and k past the end are read at the last one: those rows' results are not stored, and the k count as zero.
//   split: three planes of bf16; KC: [row][k], 32 bytes a row, the 16-byte halves of row r exchanged where r / 8 is odd
//   (the fragment reads of 16 consecutive rows then touch all banks); else [k][row], 16-byte piece c of k-line kl at
//   c ^ (kl % 4) * 4 (the four k-lines of a transposing read lie in four different groups of banks).
//   whole: fp32, KC: [row][k] padded by 16 bytes, else [k][row] padded by 32.
template <int ROWS, bool KC, int T>
struct F32Stage {
  static constexpr int kChunks = ROWS * kSK / 4 / T, kPerLine = KC ? kSK / 4 : ROWS / 4, kLines = T / kPerLine;
  static constexpr int kStride = KC ? kSK : ROWS, kPlane = ROWS * kSK;                                       // bf16
  static constexpr int kWholeStride = KC ? kSK + 4 : ROWS + 8, kWhole = (KC ? ROWS : kSK) * kWholeStride;   // floats
  static_assert(kChunks * T * 4 == ROWS * kSK && T % kPerLine == 0 && kLines % (KC ? 16 : 4) == 0, "whole chunks, one swizzle term per thread");
  f32x4 regs[kChunks];
  const float* at[KC ? kChunks : 1];   // rows of this thread's chunks, at k = 0
  int k;                               // first chunk's k in step 0
  int put;                             // and its place in a plane

  __device__ __forceinline__ void init(const float* base, long ld, long row0, long rows, int tid) {
    const int line = tid / kPerLine, c = tid % kPerLine;
    if constexpr (KC) {
#pragma unroll
      for (int j = 0; j < kChunks; ++j) {
        const long r = row0 + line + j * kLines;
        at[j] = base + (r < rows ? r : rows - 1) * ld;
      }
      k = c * 4;
      put = line * kStride + ((c >> 1) ^ (line >> 3 & 1)) * 8 + (c & 1) * 4;
    } else {
      const long r = row0 + c * 4;
      at[0] = base + (r < rows ? r : rows - 4);
      k = line;
      put = line * kStride + ((c >> 1) ^ (line & 3) << 2) * 8 + (c & 1) * 4;
    }
  }
  // chunk j of the step that starts at k0, of K
  template <int J>
  __device__ __forceinline__ void load(long ld, int k0, int K) {
    if constexpr (KC) { const int x = k0 + k, last = K - 4; regs[J] = *reinterpret_cast<const f32x4*>(at[J] + (x < last ? x : last)); }
    else { const int x = k0 + k + J * kLines, last = K - 1; regs[J] = *reinterpret_cast<const f32x4*>(at[0] + (x < last ? x : last) * ld); }
  }
  // the same, for the chunks in registers: k past the end count as zero
  __device__ __forceinline__ void clip(int k0, int K) {
#pragma unroll
    for (int j = 0; j < kChunks; ++j)
      if (k0 + k + (KC ? 0 : j * kLines) >= K) regs[j] = f32x4{0, 0, 0, 0};
  }
  // part P of chunk J goes to its plane and what is left of the value stays
  template <int J, int P>
  __device__ __forceinline__ void store(unsigned short* lds) {
    f32x4& r = regs[J];
    if constexpr (P == 0) {
#pragma unroll
      for (int q = 0; q < 4; ++q) r[q] *= kScale;
    }
    const u32x2 p = u32x2{pack2(r.x, r.y), pack2(r.z, r.w)};
    if constexpr (P < 2)
      r = f32x4{r.x - __uint_as_float(p.x << 16), r.y - __uint_as_float(p.x & 0xFFFF0000u), r.z - __uint_as_float(p.y << 16), r.w - __uint_as_float(p.y & 0xFFFF0000u)};
    *reinterpret_cast<u32x2*>(lds + P * kPlane + put + J * kLines * kStride) = p;
  }
  __device__ __forceinline__ void store_whole(float* lds, int tid) const {
#pragma unroll
    for (int j = 0; j < kChunks; ++j)
      *reinterpret_cast<f32x4*>(lds + (tid / kPerLine + j * kLines) * kWholeStride + (tid % kPerLine) * 4) = regs[j];
  }
  // lane's offset of a fragment, and the fragment of part P, 32 rows from w0 + 32 BLK (w0: a multiple of 64)
  static __device__ __forceinline__ int lane_frag(int lane, int w0) {
    if constexpr (KC) return (w0 + (lane & 31)) * kStride + ((lane >> 5) ^ (lane >> 3 & 1)) * 8;
    const int kl = (lane >> 5) * 8 + (lane >> 2 & 3);
    return kl * kStride + ((w0 + (lane >> 4 & 1) * 16 + (lane & 3) * 4) ^ (lane >> 2 & 3) << 5);
  }
  template <int P, int BLK>
  static __device__ __forceinline__ bf16x8 fragment(const unsigned short* lds, int frag) {
    if constexpr (KC) return *reinterpret_cast<const bf16x8*>(lds + P * kPlane + frag + BLK * 32 * kStride);
    else return tr_fragment(lds + P * kPlane + (frag ^ BLK << 5), kStride);
  }
  static __device__ __forceinline__ f32x4 whole_fragment(const float* lds, int row, int k, int lane) {
    if constexpr (KC) return *reinterpret_cast<const f32x4*>(lds + (row + (lane & 31)) * kWholeStride + k + (lane >> 5) * 4);
    else {
      const float* const p = lds + (k + (lane >> 5) * 4) * kWholeStride + row + (lane & 31);
      return f32x4{p[0], p[kWholeStride], p[2 * kWholeStride], p[3 * kWholeStride]};
    }
  }
};

constexpr int kSNS = 3;          // stages in LDS

// Orders LDS only: fetches stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int BM, int BN>
constexpr size_t f32_smem() { return (size_t)kSNS * 3 * (BM + BN) * kSK * sizeof(unsigned short); }

// GM x GN wavefronts, one per SIMD (256 x 256 tiles) or two workgroups of them on a compute unit.  Step s: multiplies stage s, whose first fragments the step before has read; splits
// the values of step s + 2 into their stage and asks for those of s + 3.  These are placed between the matrix instructions
// by hand, a few vector instructions to each, and pinned there.
template <int BM, int BN, int GM, int GN, bool A_KC, bool B_KC>
__global__ void __launch_bounds__(64 * GM * GN) __attribute__((amdgpu_waves_per_eu(BM * BN / (GM * GN) > 8192 ? 1 : 2, BM * BN / (GM * GN) > 8192 ? 1 : 2)))
gemm_f32_kernel(const GemmArgs g) {
  constexpr int T = 64 * GM * GN, WM = BM / GM, WN = BN / GN, TM = WM / 32, TN = WN / 32;
  using SA = F32Stage<BM, A_KC, T>;
  using SB = F32Stage<BN, B_KC, T>;
  constexpr int kStage = 3 * (SA::kPlane + SB::kPlane);
  static_assert((SA::kWhole + SB::kWhole) * 4 <= kSNS * kStage * 2 && GM * GN * 32 * (TN * 32 + 4) * 4 <= kSNS * kStage * 2, "LDS of the other phases");
  extern __shared__ __align__(16) unsigned short smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave / GN) * WM, wn0 = (wave % GN) * WN;
  const long tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
  long tmi, tni, wg, zz;
  int nx;
  place_workgroup(g, wg, zz, nx);
  tile_of_block(wg, tiles_m, tiles_n, g.xcd_m, nx, tmi, tni);
  const long m0 = tmi * BM, n0 = tni * BN;
  long ao, bo, co;
  const void *abase, *bbase;
  void *cbase, *c2base;
  decode_batch(g, decode_group(g, zz, abase, bbase, cbase, c2base), ao, bo, co);
  const long lda = A_KC ? g.a_row : g.a_k, ldb = B_KC ? g.b_row : g.b_k;

  // split-K: blockIdx.y owns a contiguous range of K steps
  const long all_steps = (g.K + kSK - 1) / kSK;
  const long per_split = (all_steps + g.splits - 1) / g.splits;
  const long kbeg = (long)blockIdx.y * per_split * kSK;
  const int K = (int)((kbeg + per_split * kSK < g.K ? kbeg + per_split * kSK : g.K) - kbeg);
  const int ksteps = K > 0 ? (K + kSK - 1) / kSK : 0;
  const float* const A = static_cast<const float*>(abase) + ao + (A_KC ? kbeg : kbeg * lda);
  const float* const B = static_cast<const float*>(bbase) + bo + (B_KC ? kbeg : kbeg * ldb);

  f32x16 acc[TM][TN];
  auto clear = [&]() OCN_LAMBDA_INLINE {
    static_for<TM>([&](auto ic) OCN_LAMBDA_INLINE {
      static_for<TN>([&](auto jc) OCN_LAMBDA_INLINE {
        static_for<16>([&](auto ec) OCN_LAMBDA_INLINE { acc[decltype(ic)::value][decltype(jc)::value][decltype(ec)::value] = 0.0f; });
      });
    });
  };
  clear();
  SA sa;
  SB sb;
  sa.init(A, lda, m0, g.M, tid);
  sb.init(B, ldb, n0, g.N, tid);
  // chunks of both operands, A's first
  constexpr int kChunks = SA::kChunks + SB::kChunks;
  auto load = [&](auto cc, int k0) OCN_LAMBDA_INLINE {
    constexpr int c = decltype(cc)::value;
    if constexpr (c < SA::kChunks) sa.template load<c>(lda, k0, K);
    else sb.template load<c - SA::kChunks>(ldb, k0, K);
  };
  auto load_all = [&](int k0) OCN_LAMBDA_INLINE { static_for<kChunks>([&](auto cc) OCN_LAMBDA_INLINE { load(cc, k0); }); };
  auto store = [&](auto cc, auto pc, unsigned short* to) OCN_LAMBDA_INLINE {
    constexpr int c = decltype(cc)::value, p = decltype(pc)::value;
    if constexpr (c < SA::kChunks) sa.template store<c, p>(to);
    else sb.template store<c - SA::kChunks, p>(to + 3 * SA::kPlane);
  };
  auto store_all = [&](int k0, unsigned short* to) OCN_LAMBDA_INLINE {
    if (k0 + kSK > K) { sa.clip(k0, K); sb.clip(k0, K); }
    static_for<kChunks * 3>([&](auto uc) OCN_LAMBDA_INLINE {
      store(std::integral_constant<int, decltype(uc)::value / 3>{}, std::integral_constant<int, decltype(uc)::value % 3>{}, to);
    });
  };
  const int a_frag = SA::lane_frag(lane, wm0), b_frag = SB::lane_frag(lane, wn0);
  bf16x8 af[2][3], bf[2][3][TN];   // [i % 2], [step % 2]
  auto read_a = [&](const unsigned short* st, auto ic) OCN_LAMBDA_INLINE {
    constexpr int i = decltype(ic)::value;
    static_for<3>([&](auto pc) OCN_LAMBDA_INLINE { af[i % 2][decltype(pc)::value] = SA::template fragment<decltype(pc)::value, i>(st, a_frag); });
  };
  auto read_b = [&](const unsigned short* st, auto par) OCN_LAMBDA_INLINE {
    static_for<3 * TN>([&](auto rc) OCN_LAMBDA_INLINE {
      constexpr int p = decltype(rc)::value / TN, j = decltype(rc)::value % TN;
      bf[decltype(par)::value][p][j] = SB::template fragment<p, j>(st + 3 * SA::kPlane, b_frag);
    });
  };
  static_assert(TM % 2 == 0, "the first block of the next step goes to the registers of block TM");
  // `st`, `nx`, `to`: stages of this step, the next and the one after
  auto step = [&](int ks, const unsigned short* st, const unsigned short* nx, unsigned short* to, auto par) OCN_LAMBDA_INLINE {
    constexpr int cur = decltype(par)::value, kPer = 6 * TN, kAll = TM * kPer, kUnits = kChunks * 3;
    if ((ks + 2) * kSK + kSK > K) { sa.clip((ks + 2) * kSK, K); sb.clip((ks + 2) * kSK, K); }
    __builtin_amdgcn_sched_barrier(0);
    static_for<kAll>([&](auto mc) OCN_LAMBDA_INLINE {
      constexpr int m = decltype(mc)::value, i = m / kPer, q = m % kPer / TN, j = m % TN;
      // small products first
      constexpr int pa = q == 1 ? 2 : q == 2 || q == 4 ? 1 : 0, pb = q == 0 ? 2 : q == 2 || q == 3 ? 1 : 0;
      if constexpr (m % kPer == 0) {
        if constexpr (i + 1 < TM) read_a(st, std::integral_constant<int, i + 1>{});
        else { read_a(nx, std::integral_constant<int, 0>{}); read_b(nx, std::integral_constant<int, 1 - cur>{}); }
      }
      static_for<kUnits>([&](auto uc) OCN_LAMBDA_INLINE {
        constexpr int u = decltype(uc)::value, c = u / 3;
        if constexpr (u * kAll / kUnits == m) {
          store(std::integral_constant<int, c>{}, std::integral_constant<int, u % 3>{}, to);
          if constexpr (u % 3 == 2) load(std::integral_constant<int, c>{}, (ks + 3) * kSK);
        }
      });
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i % 2][pa], bf[cur][pb][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    });
    lds_barrier();
  };
  if (ksteps > 0) {
    load_all(0);
    store_all(0, smem);
    load_all(kSK);
    store_all(kSK, smem + kStage);
    load_all(2 * kSK);
    lds_barrier();
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    read_a(smem, P0{});
    read_b(smem, P0{});
    unsigned short *s0 = smem, *s1 = smem + kStage, *s2 = smem + 2 * kStage;
    auto turn = [&]() OCN_LAMBDA_INLINE { unsigned short* const t = s0; s0 = s1; s1 = s2; s2 = t; };
    int ks = 0;
    for (; ks + 1 < ksteps; ks += 2) {
      step(ks, s0, s1, s2, P0{});
      turn();
      step(ks + 1, s0, s1, s2, P1{});
      turn();
    }
    if (ks < ksteps) step(ks, s0, s1, s2, P0{});
  }

  float nan = 0.0f;
  static_for<TM>([&](auto ic) OCN_LAMBDA_INLINE {
    static_for<TN>([&](auto jc) OCN_LAMBDA_INLINE {
      static_for<16>([&](auto ec) OCN_LAMBDA_INLINE {
        nan = __builtin_fmaf(acc[decltype(ic)::value][decltype(jc)::value][decltype(ec)::value], 0.0f, nan);
      });
    });
  });
  float unscale = kUnscale;
  if (__syncthreads_or(nan != nan)) {
    unscale = 1.0f;
    clear();
    float* const as = reinterpret_cast<float*>(smem);
    float* const bs = as + SA::kWhole;
#pragma unroll 1
    for (int ks = 0; ks < ksteps; ++ks) {
      load_all(ks * kSK);
      sa.clip(ks * kSK, K);
      sb.clip(ks * kSK, K);
      __syncthreads();
      sa.store_whole(as, tid);
      sb.store_whole(bs, tid);
      __syncthreads();
      // v_mfma_f32_32x32x2_f32: instruction q of four multiplies k = q (lanes 0-31) and k = 4 + q (lanes 32-63)
#pragma unroll
      for (int kk = 0; kk < kSK; kk += 8) {
        f32x4 wa[TM], wb[TN];
        static_for<TM>([&](auto ic) OCN_LAMBDA_INLINE { wa[decltype(ic)::value] = SA::whole_fragment(as, wm0 + decltype(ic)::value * 32, kk, lane); });
        static_for<TN>([&](auto jc) OCN_LAMBDA_INLINE { wb[decltype(jc)::value] = SB::whole_fragment(bs, wn0 + decltype(jc)::value * 32, kk, lane); });
        static_for<4>([&](auto qc) OCN_LAMBDA_INLINE {
          static_for<TM>([&](auto ic) OCN_LAMBDA_INLINE {
            static_for<TN>([&](auto jc) OCN_LAMBDA_INLINE {
              constexpr int q = decltype(qc)::value, i = decltype(ic)::value, j = decltype(jc)::value;
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(wa[i][q], wb[j][q], acc[i][j], 0, 0, 0);
            });
          });
        });
      }
    }
    __syncthreads();
  }
  auto rows = [&](auto ic, f32x16 (&row)[TN]) OCN_LAMBDA_INLINE -> f32x16 (&)[TN] {
    static_for<TN>([&](auto jc) OCN_LAMBDA_INLINE {
      constexpr int i = decltype(ic)::value, j = decltype(jc)::value;
      asm volatile("" : "+a"(acc[i][j]));   // (in accumulation registers until here)
      static_for<16>([&](auto ec) OCN_LAMBDA_INLINE { row[j][decltype(ec)::value] = acc[i][j][decltype(ec)::value] * unscale; });
    });
    return row;
  };
  epilogue<TM, TN>(g, cbase, c2base, rows, m0 + wm0, n0 + wn0, co, lane, reinterpret_cast<float*>(smem) + wave * 32 * (TN * 32 + 4));
}

template <int BM, int BN, int GM, int GN, bool A_KC, bool B_KC>
hipError_t go(const GemmArgs& a, hipStream_t s, hipEvent_t ev) {
  return launch(gemm_f32_kernel<BM, BN, GM, GN, A_KC, B_KC>, f32_smem<BM, BN>(), BM, BN, a, s, ev, 64 * GM * GN);
}
template <int BM, int BN, int GM, int GN>
hipError_t go_layout(bool akc, bool bkc, const GemmArgs& a, hipStream_t s, hipEvent_t ev) {
  if (akc && bkc) return go<BM, BN, GM, GN, true, true>(a, s, ev);
  if (akc) return go<BM, BN, GM, GN, true, false>(a, s, ev);
  if (bkc) return go<BM, BN, GM, GN, false, true>(a, s, ev);
  return go<BM, BN, GM, GN, false, false>(a, s, ev);
}

}  // namespace

hipError_t launch_gemm_f32(bool big, bool akc, bool bkc, const GemmArgs& a, hipStream_t s, hipEvent_t ev) {
  return big ? go_layout<256, 256, 2, 2>(akc, bkc, a, s, ev) : go_layout<128, 128, 2, 2>(akc, bkc, a, s, ev);
}

}  // namespace ocannl
