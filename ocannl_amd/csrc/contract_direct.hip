// Contractions of any extents and strides whose tiles are few: latency is what bounds them, so nothing stands between a
// load and the matrix instruction that takes it.  A workgroup owns 32 x 32 cells of C and its four wavefronts share K:
// wavefront w takes every fourth step of 32 k and reads its operands straight into the registers of
// v_mfma_f32_16x16x32_bf16 -- no LDS and no barrier in the loop, two or three steps in flight -- and the four partial tiles
// meet in LDS once, where rows of C come out 32 lanes wide.
//
//   k-contiguous operand: lane l holds row l % 16 of each block of 16 rows and k = 8 (l / 16) .. + 7 of the step: 16
//     bytes of bf16 (32 of fp32), four lanes to 64 (128) consecutive bytes.
//   row-contiguous operand: lane l holds rows 2 (l % 16) and the next at each of those eight k, that is row l % 16 of the
//     two blocks {even rows} and {odd rows}: 16 lanes read consecutive bytes, and no transposition is left to do but
//     pairing the halves of bf16 words.
//
// An fp32 operand is multiplied as the sum of three bf16 values (see contract_any.h); tiles that this does not cover, those
// with subnormal values of a bf16 operand beside it among them, are multiplied again with v_mfma_f32_16x16x4_f32, whose k =
// j, 8 + j, 16 + j, 24 + j are what the lanes hold at place j (594 x 320 x 320 10.3 -> 14.3 us).
//
// 594 x 320 (190 tiles) by K, tile with LDS stages before -> now: fp32 10.4 + 0.011 us a k -> 5 + 0.0065; bf16 with a
// row-contiguous operand 4.5 + 0.005 -> 4.2 + 0.003.  A transformer step of 594 rows with 320 to 1280 channels and mixed
// products 528 -> 475 us.  Tiles of 64 x 64 in this form take 1.5 us more to start and to meet; eight wavefronts instead of
// four gained nothing (K = 1001 bf16 7.1 -> 7.4 us, fp32 11.2 -> 11.3).  Chains of three products into one C, 594 x 320 x 320 each:
// 24.9 us on fifteen 128 x 128 tiles, 11.0 here.
#include <hip/hip_runtime.h>

#include "contract_any.hpp"

namespace ocannl {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Subnormal values of a bf16 operand beside one in parts: the least 2 |bits| - 1 of each half of its words (zero: the largest).
// Three instructions a word, where scaling the operand would take five: 2 % of a launch instead of 4 (a batch of five 180 x 26
// x 870 8.0 us without either, 8.6, 8.9).
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned watch(unsigned least, unsigned w) {
  const u16x2 twice = __builtin_bit_cast(u16x2, w) * (unsigned short)2;
  return __builtin_bit_cast(unsigned, __builtin_elementwise_min(__builtin_bit_cast(u16x2, least), (u16x2)(twice - (unsigned short)1)));
}
__device__ __forceinline__ bool subnormal(unsigned least) { return (least & 0xFFFFu) < 0xFFu || least >> 16 < 0xFFu; }

// One operand of a wavefront's step.
constexpr int R = 2;              // blocks of 16 rows of a tile
constexpr int kDirectWaves = 4;   // wavefronts that share K

template <bool KC, bool BF>
struct DirectOperand {
  // KC: 8 k of R rows; else R rows at 8 k.  bf16: words of two k or of two rows
  static constexpr int kWords = KC ? (BF ? 4 : 8) : (BF ? R / 2 : R);   // per row (KC) or per k
  struct Set { unsigned w[KC ? R : 8][kWords]; };
  int off[KC ? R : 1];
  int shift;        // !KC: rows by which the chunk starts early
  unsigned least;   // of watch()

  __device__ __forceinline__ void init(const OcnAnyOperand& o, const OcnDigits& dr, int row0, int rows, int lane) {
    shift = 0;
    least = ~0u;
    if constexpr (KC) {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int r = row0 + i * 16 + (lane & 15);
        off[i] = ocn_digit_off(ocn_digits(dr, r < rows ? r : rows - 1), o.row);
      }
    } else {
      const int r = row0 + (lane & 15) * R, at = r + R <= rows ? r : rows - R;
      off[0] = ocn_digit_off(ocn_digits(dr, at), o.row);
      shift = r - at < R ? r - at : R;
    }
  }
  template <int N>
  static __device__ __forceinline__ void fetch(unsigned (&w)[N], const void* p, long element) {
    __builtin_memcpy(w, static_cast<const char*>(p) + element * (BF ? 2 : 4), N * 4);
  }
  template <bool K1>
  static __device__ __forceinline__ int koff(const OcnAnyDesc& d, const OcnAnyOperand& o, int k) {
    if constexpr (K1) return KC ? k : k * o.k[2];
    else return ocn_digit_off(ocn_digits(d.dk, k), o.k);
  }
  // the step that starts at k0.  TAIL: k may pass kend; such a step is completed by tail()
  template <bool TAIL, bool K1>
  __device__ __forceinline__ void load(Set& s, const OcnAnyDesc& d, const OcnAnyOperand& o, const void* p, int k0, int kend, int lane) const {
    const int k = k0 + (lane >> 4) * 8;
    if constexpr (KC) {
      constexpr int V = BF ? 8 : 4;
#pragma unroll
      for (int h = 0; h < 8 / V; ++h) {
        int at = k + h * V;
        if (TAIL && at + V > kend) at = kend - V;
        const int ko = koff<K1>(d, o, at);
#pragma unroll
        for (int i = 0; i < R; ++i) fetch(*reinterpret_cast<unsigned(*)[4]>(&s.w[i][h * 4]), p, (long)off[i] + ko);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int at = TAIL && k + j >= kend ? kend - 1 : k + j;
        fetch(s.w[j], p, (long)off[0] + koff<K1>(d, o, at));
      }
    }
  }
  // N words down by n elements, zeros from above
  template <int N>
  static __device__ __forceinline__ void down(unsigned* w, int n) {
    const int words = BF ? n >> 1 : n, half = BF ? (n & 1) * 16 : 0;
    unsigned t[N + 1];
#pragma unroll
    for (int q = 0; q <= N; ++q) {
      t[q] = 0;
#pragma unroll
      for (int e = q; e < N; ++e) t[q] = e == q + words ? w[e] : t[q];
    }
#pragma unroll
    for (int q = 0; q < N; ++q) w[q] = BF ? __funnelshift_r(t[q], t[q + 1], half) : t[q];
  }
  // rows past the end: those of the chunk that exist go where they belong
  __device__ __forceinline__ void edge(Set& s) const {
    if constexpr (!KC) {
#pragma unroll
      for (int j = 0; j < 8; ++j) down<kWords>(s.w[j], shift);
    }
  }
  // k past the end count as zero
  __device__ __forceinline__ void tail(Set& s, int k0, int kend, int lane) const {
    const int k = k0 + (lane >> 4) * 8;
    if constexpr (KC) {
      constexpr int V = BF ? 8 : 4;
#pragma unroll
      for (int h = 0; h < 8 / V; ++h) {
        const int past = k + h * V + V - kend, n = past < 0 ? 0 : past < V ? past : V;
#pragma unroll
        for (int i = 0; i < R; ++i) down<4>(&s.w[i][h * 4], n);
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (k + j >= kend)
#pragma unroll
          for (int q = 0; q < kWords; ++q) s.w[j][q] = 0;
    }
  }
  // fp32: value j of block b
  static __device__ __forceinline__ float value(const Set& s, int b, int j) {
    if constexpr (!BF) return __uint_as_float(KC ? s.w[b][j] : s.w[j][b]);
    else {
      const unsigned x = KC ? s.w[b][j / 2] : s.w[j][b / 2];
      return (KC ? j & 1 : b & 1) ? __uint_as_float(x & 0xFFFF0000u) : __uint_as_float(x << 16);
    }
  }
  // block b as matrix operands: its bf16 values (WATCH: beside an operand in parts), or the three parts of its fp32 values
  template <bool WATCH>
  __device__ __forceinline__ void fragments(const Set& s, int b, bf16x8 (&f)[BF ? 1 : 3]) {
    unsigned u[4];
    if constexpr (BF) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        u[q] = KC ? s.w[b][q] : __builtin_amdgcn_perm(s.w[2 * q + 1][b / 2], s.w[2 * q][b / 2], b & 1 ? 0x07060302u : 0x05040100u);
        if constexpr (WATCH) least = watch(least, u[q]);
      }
      f[0] = __builtin_bit_cast(bf16x8, u);
    } else {
      float r[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) r[j] = value(s, b, j) * kOcnScale;
#pragma unroll
      for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          u[q] = ocn_bf16_pair(r[2 * q], r[2 * q + 1]);
          if (p < 2) { r[2 * q] -= __uint_as_float(u[q] << 16); r[2 * q + 1] -= __uint_as_float(u[q] & 0xFFFF0000u); }
        }
        f[p] = __builtin_bit_cast(bf16x8, u);
      }
    }
  }
};

constexpr int kDirectTile = 16 * R, kDirectStride = kDirectTile + 4;   // floats of a row of partial sums

// Grid as in any_body (contract_any.hpp).
// PF: steps in flight; CHAIN: several operand pairs into one C (bf16 operands).
template <int W, bool A_KC, bool B_KC, bool ABF, bool BBF, int PF, bool CHAIN>
__device__ __forceinline__ void direct_body(const OcnAnyDesc& d, const AnyBatch& q, const AnyPtrs& p) {
  constexpr bool F32 = !(ABF && BBF);
  constexpr int BT = kDirectTile, LS = kDirectStride;
  using OA = DirectOperand<A_KC, ABF>;
  using OB = DirectOperand<B_KC, BBF>;
  extern __shared__ __align__(16) float smem_direct[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int per = gridDim.x / 8, tiles = d.tiles_m * d.tiles_n;
  const int t = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  const int z = t / tiles, r = t - z * tiles;
  if (z >= q.batches * q.members) return;
  const void *a, *b;
  void *c, *c2;
  any_operands(d, q, p, z, a, b, c, c2);
  const int m0 = r / d.tiles_n * BT, n0 = r % d.tiles_n * BT;
  const int steps = (d.K + 31) / 32, per_split = (steps + d.splits - 1) / d.splits;
  const int kbeg = (int)blockIdx.y * per_split * 32;
  const int kend = kbeg + per_split * 32 < d.K ? kbeg + per_split * 32 : d.K;
  const int full = kend > kbeg ? (kend - kbeg) / 32 : 0;
  const int mine = (full - wave + W - 1) / W;                               // full steps of this wavefront (<= 0: none)
  const bool last = kend > kbeg + full * 32 && full % W == wave;            // and the partial one
  const bool edge_a = !A_KC && m0 + BT > d.M, edge_b = !B_KC && n0 + BT > d.N;

  OA oa;
  OB ob;
  oa.init(d.a, d.dm, m0, d.M, lane);
  ob.init(d.b, d.dn, n0, d.N, lane);
  f32x4 acc[R][R];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < R; ++j) acc[i][j] = f32x4{0, 0, 0, 0};
  };
  auto multiply = [&](typename OA::Set& x, typename OB::Set& y, auto exact) __attribute__((always_inline)) {
    if (edge_a) oa.edge(x);
    if (edge_b) ob.edge(y);
    if constexpr (decltype(exact)::value) {
#pragma unroll
      for (int k = 0; k < 8; ++k)
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
          for (int j = 0; j < R; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(OA::value(x, i, k), OB::value(y, j, k), acc[i][j], 0, 0, 0);
    } else {
      constexpr int NA = ABF ? 1 : 3, NB = BBF ? 1 : 3;
      bf16x8 fb[R][NB];
#pragma unroll
      for (int j = 0; j < R; ++j) ob.template fragments<F32>(y, j, fb[j]);
#pragma unroll
      for (int i = 0; i < R; ++i) {
        bf16x8 fa[NA];
        oa.template fragments<F32>(x, i, fa);
#pragma unroll
        for (int s = NA == 1 && NB == 1 ? 0 : 2; s >= 0; --s)       // small products first
#pragma unroll
          for (int pa = 0; pa < NA; ++pa) {
            if (s - pa < 0 || s - pa >= NB) continue;
#pragma unroll
            for (int j = 0; j < R; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[pa], fb[j][s - pa], acc[i][j], 0, 0, 0);
          }
      }
    }
  };
  const void *pa = a, *pb = b;
  auto load = [&](typename OA::Set& x, typename OB::Set& y, int step, auto tail, auto single) __attribute__((always_inline)) {
    constexpr bool T = decltype(tail)::value, K1 = decltype(single)::value;
    oa.template load<T, K1>(x, d, d.a, pa, kbeg + step * 32, kend, lane);
    ob.template load<T, K1>(y, d, d.b, pb, kbeg + step * 32, kend, lane);
  };
  using Yes = OcnAnyYes;
  using No = OcnAnyNo;
  auto sum = [&](auto single, auto exact) __attribute__((always_inline)) {
    typename OA::Set xa[PF], ta;
    typename OB::Set xb[PF], tb;
    auto at = [&](int s) __attribute__((always_inline)) { return wave + (s < mine ? s : mine - 1) * W; };
    if (mine > 0) {
#pragma unroll
      for (int s = 0; s < PF; ++s) load(xa[s], xb[s], at(s), No{}, single);
    }
    if (last) load(ta, tb, full, Yes{}, single);
    if (mine > 0) {
      int s = 0;
      for (; s + PF <= mine; s += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
          multiply(xa[u], xb[u], exact);
          load(xa[u], xb[u], at(s + u + PF), No{}, single);
        }
      }
#pragma unroll
      for (int u = 0; u + 1 < PF; ++u)
        if (s + u < mine) multiply(xa[u], xb[u], exact);
    }
    if (last) {
      oa.tail(ta, kbeg + full * 32, kend, lane);
      ob.tail(tb, kbeg + full * 32, kend, lane);
      multiply(ta, tb, exact);
    }
  };
  // A lane has column l % 16 of a 16 x 16 block, element e is row 4 (l / 16) + e; rows and columns of block b as in the
  // operands.  Wavefront w takes rows w BT / W .. of the sum, a lane to a column.
  constexpr int RW = BT / W, LC = BT, RL = 64 / LC;   // rows per wavefront, lanes per row, rows at once
  float v[RW / RL];
  auto reduce = [&]() __attribute__((always_inline)) {
    float* const mine_at = smem_direct + wave * BT * LS;
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int x = (lane >> 4) * 4 + e, m = A_KC ? i * 16 + x : x * R + i;
#pragma unroll
        for (int j = 0; j < R; ++j) mine_at[m * LS + (B_KC ? j * 16 + (lane & 15) : (lane & 15) * R + j)] = acc[i][j][e];
      }
    __syncthreads();
    const float* const from = smem_direct + (wave * RW + lane / LC) * LS + lane % LC;
#pragma unroll
    for (int x = 0; x < RW / RL; ++x) {
      v[x] = from[x * RL * LS];
#pragma unroll
      for (int w = 1; w < W; ++w) v[x] += from[x * RL * LS + w * BT * LS];
    }
  };

  // C's cells of this lane; what is accumulated into is asked for ahead of everything else
  const int n = n0 + lane % LC, mr = m0 + wave * RW + lane / LC;
  const bool to_ws = d.splits > 1;
  const int cn = ocn_digit_off(ocn_digits(d.dn, n < d.N ? n : d.N - 1), d.c_n);
  float* const cf = static_cast<float*>(c);
  unsigned short* const ch = static_cast<unsigned short*>(c);
  float old[RW / RL];
#pragma unroll
  for (int x = 0; x < RW / RL; ++x) old[x] = 0.0f;
  if (d.accumulate && !to_ws) {
#pragma unroll
    for (int x = 0; x < RW / RL; ++x) {
      const int m = mr + x * RL, at = ocn_digit_off(ocn_digits(d.dm, m < d.M ? m : d.M - 1), d.c_m) + cn;
      old[x] = d.c_bf16 ? __uint_as_float((unsigned)ch[at] << 16) : cf[at];
    }
  }
  clear();
  if (d.dk.n == 1) sum(Yes{}, No{}); else sum(No{}, No{});
  if constexpr (CHAIN) {
    // (at the same offsets in the tensors of every pair)
#pragma unroll 1
    for (int pair = 1; pair < p.pairs; ++pair) {
      pa = static_cast<const char*>(pair == 1 ? p.a[1] : pair == 2 ? p.a[2] : p.a[3]) + (static_cast<const char*>(a) - static_cast<const char*>(p.a[0]));
      pb = static_cast<const char*>(pair == 1 ? p.b[1] : pair == 2 ? p.b[2] : p.b[3]) + (static_cast<const char*>(b) - static_cast<const char*>(p.b[0]));
      if (d.dk.n == 1) sum(Yes{}, No{}); else sum(No{}, No{});
    }
  }
  reduce();
  if constexpr (F32) {
    float nan = 0.0f;
#pragma unroll
    for (int x = 0; x < RW / RL; ++x) nan = __builtin_fmaf(v[x], 0.0f, nan);
    if (__syncthreads_or(nan != nan || subnormal(oa.least) || subnormal(ob.least))) {
      clear();
      sum(No{}, Yes{});
      reduce();
    } else {
#pragma unroll
      for (int x = 0; x < RW / RL; ++x) v[x] *= ABF || BBF ? 1.0f / kOcnScale : kOcnUnscale;
    }
  }
  if (n >= d.N) return;
  auto to_bf16 = [](float x) __attribute__((always_inline)) { return __builtin_bit_cast(unsigned short, (__bf16)x); };
  if (to_ws) {
    float* const w = p.ws + ((long)z * d.splits + blockIdx.y) * d.M * d.N + n;
#pragma unroll
    for (int x = 0; x < RW / RL; ++x)
      if (mr + x * RL < d.M) w[(long)(mr + x * RL) * d.N] = v[x];
    return;
  }
#pragma unroll
  for (int x = 0; x < RW / RL; ++x) {
    const int m = mr + x * RL;
    if (m >= d.M) continue;
    const int at = ocn_digit_off(ocn_digits(d.dm, m), d.c_m) + cn;
    float y = v[x];
    if (d.accumulate) y += old[x];
    if (!d.c_bf16) {
      cf[at] = y;
      if (c2) static_cast<unsigned short*>(c2)[at] = to_bf16(y);
    } else {
      unsigned short h = to_bf16(y);
      if (p.ep.bias) h = to_bf16(__uint_as_float((unsigned)h << 16) + __uint_as_float((unsigned)p.ep.bias[n] << 16));
      const unsigned short relu = (h & 0x8000u) || (h & 0x7FFFu) > 0x7F80u ? (unsigned short)0 : h;   // fmaxf(0, x)
      if (p.ep.relu_from_c) *reinterpret_cast<unsigned short*>(reinterpret_cast<char*>(ch + at) + p.ep.relu_from_c) = relu;
      ch[at] = p.ep.relu_c ? relu : h;
    }
  }
}

template <bool A_KC, bool B_KC, bool ABF, bool BBF, int PF, bool CHAIN>
__global__ void __launch_bounds__(64 * kDirectWaves) gemm_bf16_kernel_any_direct(const OcnAnyDesc d, const AnyBatch q, const AnyPtrs p) {
  direct_body<kDirectWaves, A_KC, B_KC, ABF, BBF, PF, CHAIN>(d, q, p);
}
template <bool A_KC, bool B_KC, bool ABF, bool BBF, int PF, bool CHAIN>
__global__ void __launch_bounds__(64 * kDirectWaves) gemm_f32_kernel_any_direct(const OcnAnyDesc d, const AnyBatch q, const AnyPtrs p) {
  direct_body<kDirectWaves, A_KC, B_KC, ABF, BBF, PF, CHAIN>(d, q, p);
}

template <bool A_KC, bool B_KC, bool ABF, bool BBF>
hipError_t go_direct(dim3 grid, const OcnAnyDesc& d, const AnyBatch& q, const AnyPtrs& p, hipStream_t s) {
  constexpr int smem = kDirectWaves * kDirectTile * kDirectStride * 4;
  void (*kernel)(OcnAnyDesc, AnyBatch, AnyPtrs);
  if constexpr (ABF && BBF) kernel = p.pairs > 1 ? gemm_bf16_kernel_any_direct<A_KC, B_KC, ABF, BBF, 2, true> : gemm_bf16_kernel_any_direct<A_KC, B_KC, ABF, BBF, 3, false>;
  else kernel = gemm_f32_kernel_any_direct<A_KC, B_KC, ABF, BBF, 2, false>;
  hipLaunchKernelGGL(kernel, grid, dim3(64 * kDirectWaves), smem, s, d, q, p);
  return hipGetLastError();
}
template <bool ABF, bool BBF>
hipError_t direct_layout(bool akc, bool bkc, dim3 grid, const OcnAnyDesc& d, const AnyBatch& q, const AnyPtrs& p, hipStream_t s) {
  if (akc && bkc) return go_direct<true, true, ABF, BBF>(grid, d, q, p, s);
  if (akc) return go_direct<true, false, ABF, BBF>(grid, d, q, p, s);
  if (bkc) return go_direct<false, true, ABF, BBF>(grid, d, q, p, s);
  return go_direct<false, false, ABF, BBF>(grid, d, q, p, s);
}

}  // namespace

hipError_t launch_direct(bool akc, bool bkc, dim3 grid, const OcnAnyDesc& d, const void* qp, const void* pp, hipStream_t s) {
  const AnyBatch& q = *static_cast<const AnyBatch*>(qp);
  const AnyPtrs& p = *static_cast<const AnyPtrs*>(pp);
  if (d.a.bf16 && d.b.bf16) return direct_layout<true, true>(akc, bkc, grid, d, q, p, s);
  if (d.a.bf16) return direct_layout<true, false>(akc, bkc, grid, d, q, p, s);
  if (d.b.bf16) return direct_layout<false, true>(akc, bkc, grid, d, q, p, s);
  return direct_layout<false, false>(akc, bkc, grid, d, q, p, s);
}

}  // namespace ocannl
