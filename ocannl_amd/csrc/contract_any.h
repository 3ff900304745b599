// Device code of the contraction tile that takes any extents and strides:
//     C[z, m, n] (+)= sum_k A[z, m, k] * B[z, n, k]
// with m, n and k each a number of up to three digits (loop symbols of that class) and every operand's
// element offset linear in the digits.  Covers what the kernels in gemm.hip leave out: extents and strides
// that are not multiples of a vector, results with rows at any element, and convolution windows
// (x[stride * o + k] splits into digits of m and of k).  Compiled into the library (contract_any.hip, with the
// descriptor as a kernel argument) and, with a constant descriptor, into generated kernels.
//
// Operands are staged through registers into LDS in chunks of 16 bytes of compute type along whichever of
// k and the row is contiguous in memory.  A chunk that lies inside one run of the operand is ONE load at
// whatever element it starts (the vector memory path takes any element alignment); a chunk that crosses the
// end of a run or of the operand is gathered element by element.  LDS layouts and fragment reads are those
// of the register-staged kernels (gemm_common.hpp): rows padded by 16 bytes for a k-contiguous operand,
// [k][row] with ds_read_b64_tr_b16 fragments for a row-contiguous bf16 one.
//
// What bounds it: latency of a K step (load, LDS, barrier), with several workgroups per compute unit to hide it;
// address arithmetic comes next (up to two quotients per chunk and step).  As generated kernels, one thread or
// lane group per element of C, these contractions ran at the rate of scalar loads.  Measured, before -> now:
// b=1777 i=1001 o=771 bf16, forward and both gradients, 4192 -> 101 us; attention scores and their product with
// V over 197 positions, 96 heads, 438 + 569 -> 14 + 12 us; a 3 x 3 convolution of 64 x 32 x 32 positions,
// 32 -> 64 channels in fp32, forward 314 -> 66 us, weight gradient 2106 -> 94 us, input gradient (which only
// the batch and channel axes kept apart: 2048 threads) 28 500 -> 43 us.
#pragma once

template <bool C, typename A, typename B> struct ocn_if { using type = A; };
template <typename A, typename B> struct ocn_if<false, A, B> { using type = B; };

struct OcnDigits {            // x = (d0 * e1 + d1) * e2 + d2
  int n;                      // digits in use: 1 (d2 only) .. 3
  int e1, e2;                 // extents of d1 and d2
  unsigned mul1, mul2;        // quotients by e1 and e2 (see ocn_digit_div)
  int sh1, sh2;
};

struct OcnAnyOperand {
  int row[3], k[3];           // element strides of the row digits (m or n) and of the k digits
  int bf16;                   // precision in memory: bf16, else fp32
};

struct OcnAnyDesc {
  int M, N, K;
  OcnDigits dm, dn, dk;
  OcnAnyOperand a, b;
  int c_m[3], c_n[3];         // element strides of C by digit
  int c_bf16, accumulate;
  int splits, tiles_m, tiles_n;
  // Windows (the input gradient of a convolution, gathered): digit d1 of m minus digit d0 of k, and digit d2
  // of m minus digit d1 of k, are positions in A that count only inside [0, win_lim).  A tile works on the
  // positions of C of one residue (r0, r1) modulo the strides win_s: digit d1 of m is position win_s * d1 + r0
  // (of win_pos), digit d0 of k is tap win_s * d0 + r0 (of win_taps).
  int win_s[2], win_taps[2], win_lim[2], win_pos[2];
};

typedef __bf16 ocn_bf16x8 __attribute__((ext_vector_type(8)));
typedef float ocn_f32x16 __attribute__((ext_vector_type(16)));
typedef float ocn_f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int ocn_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int ocn_u32x2 __attribute__((ext_vector_type(2)));

// x / d for 0 <= x < 2^31: (hi32(x * mul) + x) >> sh with sh = ceil(log2 d), mul = floor(2^32 (2^sh - d) / d) + 1
// (division by an invariant integer through multiplication, Granlund and Montgomery 1994)
__device__ __forceinline__ int ocn_digit_div(int x, unsigned mul, int sh) {
  return (int)((__umulhi((unsigned)x, mul) + (unsigned)x) >> sh);
}
struct OcnDigitVal { int d0, d1, d2; };
__device__ __forceinline__ OcnDigitVal ocn_digits(const OcnDigits& d, int x) {
  OcnDigitVal v{0, 0, x};
  if (d.n > 1) {
    const int q = ocn_digit_div(x, d.mul2, d.sh2);
    v.d2 = x - q * d.e2;
    v.d1 = q;
    if (d.n > 2) { v.d0 = ocn_digit_div(q, d.mul1, d.sh1); v.d1 = q - v.d0 * d.e1; }
  }
  return v;
}
__device__ __forceinline__ int ocn_digit_off(const OcnDigitVal& v, const int (&s)[3]) { return v.d0 * s[0] + v.d1 * s[1] + v.d2 * s[2]; }

// ROWS x BK tile of one operand: global -> registers -> LDS, 256 threads.  F32: fp32 in LDS (bf16 sources are
// widened, exactly), chunks of 4; else bf16 in LDS, chunks of 8.  WIN: see OcnAnyDesc::win (1: this is A, 2: B).
template <int ROWS, bool KC, bool F32, int WIN>
struct OcnAnyStage {
  static constexpr int V = F32 ? 4 : 8, BK = F32 ? 32 : 64;
  static constexpr int PER = KC ? BK / V : ROWS / V;             // chunks per contiguous line
  static constexpr int CH = ROWS * BK / V / 256;                 // chunks per thread
  static constexpr int LINES = 256 / PER;                        // lines one pass of the workgroup covers
  static constexpr int PAD = F32 ? (KC ? 4 : 8) : (KC ? 8 : 32);
  static constexpr int STRIDE = (KC ? BK : ROWS) + PAD;          // LDS elements per line
  static constexpr int ELEMS = (KC ? ROWS : BK) * STRIDE;
  using Elem = typename ocn_if<F32, float, unsigned short>::type;
  union Chunk { ocn_u32x4 u; ocn_f32x4 f; unsigned short h[8]; float s[4]; };
  Chunk regs[CH];
  int off[KC ? CH : 1];       // KC: row offset of each chunk, -1 outside; else the row offset of this thread's rows
  int u0[WIN == 1 ? CH : 1], u1[WIN == 1 ? CH : 1];
  int left;                   // !KC: rows from this thread's first one that exist and lie in one run

  __device__ __forceinline__ void init(const OcnAnyOperand& o, const OcnDigits& dr, int row0, int rows, int tid) {
    if constexpr (KC) {
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const int r = row0 + tid / PER + j * LINES;
        const OcnDigitVal v = ocn_digits(dr, r);
        off[j] = r < rows ? ocn_digit_off(v, o.row) : -1;
        if constexpr (WIN == 1) { u0[j] = v.d1; u1[j] = v.d2; }
      }
    } else {
      const int r = row0 + (tid % PER) * V;
      const OcnDigitVal v = ocn_digits(dr, r);
      off[0] = ocn_digit_off(v, o.row);
      left = o.row[2] == 1 ? (dr.n > 1 ? (dr.e2 - v.d2 < rows - r ? dr.e2 - v.d2 : rows - r) : rows - r) : 0;
    }
  }

  static __device__ __forceinline__ float one(const void* p, bool bf, long i) {
    return bf ? __uint_as_float((unsigned)static_cast<const unsigned short*>(p)[i] << 16) : static_cast<const float*>(p)[i];
  }
  static __device__ __forceinline__ void whole(Chunk& c, const void* p, bool bf, long i) {
    if constexpr (!F32) __builtin_memcpy(&c.u, static_cast<const unsigned short*>(p) + i, 16);
    else if (bf) {
      ocn_u32x2 t;
      __builtin_memcpy(&t, static_cast<const unsigned short*>(p) + i, 8);
      c.f = ocn_f32x4{__uint_as_float(t.x << 16), __uint_as_float(t.x & 0xFFFF0000u), __uint_as_float(t.y << 16), __uint_as_float(t.y & 0xFFFF0000u)};
    } else __builtin_memcpy(&c.f, static_cast<const float*>(p) + i, 16);
  }
  __device__ __forceinline__ void set(Chunk& c, int i, const void* p, bool bf, long at) const {
    if constexpr (F32) c.s[i] = one(p, bf, at);
    else c.h[i] = static_cast<const unsigned short*>(p)[at];
  }
  // do the taps of k digits (d0, d1) exist; does the position of chunk j's row less those digits lie in A?
  static __device__ __forceinline__ bool tap(const OcnAnyDesc& d, const OcnDigitVal& v, int r0, int r1) {
    return d.win_s[0] * v.d0 + r0 < d.win_taps[0] && d.win_s[1] * v.d1 + r1 < d.win_taps[1];
  }
  __device__ __forceinline__ bool inside(const OcnAnyDesc& d, const OcnDigitVal& v, int j) const {
    return (unsigned)(u0[j] - v.d0) < (unsigned)d.win_lim[0] && (unsigned)(u1[j] - v.d1) < (unsigned)d.win_lim[1];
  }

  // r0, r1: residues (windows only)
  __device__ __forceinline__ void load(const OcnAnyDesc& d, const OcnAnyOperand& o, const OcnDigits& dr, const void* p, int row0, int rows, int k0,
                                       int kend, int tid, int r0, int r1) {
    const bool bf = F32 ? o.bf16 != 0 : true;
    if constexpr (KC) {
      const int k = k0 + (tid % PER) * V;
      const OcnDigitVal v = ocn_digits(d.dk, k);
      const int koff = ocn_digit_off(v, o.k);
      const bool run = o.k[2] == 1 && k + V <= kend && (d.dk.n == 1 || v.d2 + V <= d.dk.e2);
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        regs[j].u = ocn_u32x4{0, 0, 0, 0};
        if (off[j] < 0) continue;
        if (run) {
          bool there = true;
          if constexpr (WIN != 0) there = tap(d, v, r0, r1);
          if constexpr (WIN == 1) there = there && inside(d, v, j);
          if (there) whole(regs[j], p, bf, (long)off[j] + koff);
        } else {
#pragma unroll
          for (int i = 0; i < V; ++i) {
            if (k + i >= kend) continue;
            const OcnDigitVal w = ocn_digits(d.dk, k + i);
            bool there = true;
            if constexpr (WIN != 0) there = tap(d, w, r0, r1);
            if constexpr (WIN == 1) there = there && inside(d, w, j);
            if (there) set(regs[j], i, p, bf, (long)off[j] + ocn_digit_off(w, o.k));
          }
        }
      }
    } else {
      const int r = row0 + (tid % PER) * V;
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        regs[j].u = ocn_u32x4{0, 0, 0, 0};
        const int k = k0 + tid / PER + j * LINES;
        if (k >= kend) continue;
        const OcnDigitVal v = ocn_digits(d.dk, k);
        if constexpr (WIN != 0) { if (!tap(d, v, r0, r1)) continue; }
        const int koff = ocn_digit_off(v, o.k);
        if (left >= V) whole(regs[j], p, bf, (long)off[0] + koff);
        else {
#pragma unroll
          for (int i = 0; i < V; ++i)
            if (r + i < rows) set(regs[j], i, p, bf, (long)ocn_digit_off(ocn_digits(dr, r + i), o.row) + koff);
        }
      }
    }
  }
  __device__ __forceinline__ void store(Elem* lds, int tid) const {
#pragma unroll
    for (int j = 0; j < CH; ++j)
      *reinterpret_cast<ocn_u32x4*>(lds + (tid / PER + j * LINES) * STRIDE + (tid % PER) * V) = regs[j].u;
  }
};

// MFMA fragment out of a [k][row] bf16 tile; see tr_fragment in gemm_common.hpp for the lane mapping
__device__ __forceinline__ ocn_bf16x8 ocn_any_tr(const unsigned short* at_lane, int stride) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef s16x4 __attribute__((address_space(3))) * lds_ptr;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(at_lane));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(at_lane + 4 * stride));
  return __builtin_bit_cast(ocn_bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int BM, int BN, bool A_KC, bool B_KC, bool F32>
constexpr int ocn_any_smem() {
  return 2 * (OcnAnyStage<BM, A_KC, F32, 0>::ELEMS + OcnAnyStage<BN, B_KC, F32, 0>::ELEMS) * (F32 ? 4 : 2);
}

// One BM x BN tile (or, with splits, its share `split` of K) by 256 threads = 2 x 2 wavefronts (4 x 1 for tiles of 32
// columns, 1 x 4 for tiles of 32 rows).  a, b, c, c2: operands
// at the batch entry; ws: with splits, where partial sums of this entry go ([split][M][N] fp32).  c2: a bf16
// tensor of C's layout that receives the rounded fp32 result, or null.
template <int BM, int BN, bool A_KC, bool B_KC, bool F32, bool WIN>
__device__ __forceinline__ void ocn_any_tile(const OcnAnyDesc& d, const void* a, const void* b, void* c, void* c2, float* ws, int tm, int tn, int split,
                                             int r0, int r1, unsigned char* smem) {
  using SA = OcnAnyStage<BM, A_KC, F32, WIN ? 1 : 0>;
  using SB = OcnAnyStage<BN, B_KC, F32, WIN ? 2 : 0>;
  using Elem = typename SA::Elem;
  constexpr int BK = SA::BK, GN = BN == 32 ? 1 : BM == 32 ? 4 : 2, GM = 4 / GN, WM = BM / GM, WN = BN / GN, TM = WM / 32, TN = WN / 32;
  Elem* const as = reinterpret_cast<Elem*>(smem);
  Elem* const bs = as + 2 * SA::ELEMS;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave / GN) * WM, wn = (wave % GN) * WN, m0 = tm * BM, n0 = tn * BN;
  const int steps = (d.K + BK - 1) / BK, per = (steps + d.splits - 1) / d.splits;
  const int kbeg = split * per * BK;
  const int kend = kbeg + per * BK < d.K ? kbeg + per * BK : d.K;
  const int ksteps = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;

  SA sa; SB sb;
  sa.init(d.a, d.dm, m0, d.M, tid);
  sb.init(d.b, d.dn, n0, d.N, tid);
  ocn_f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  if (ksteps > 0) {
    sa.load(d, d.a, d.dm, a, m0, d.M, kbeg, kend, tid, r0, r1);
    sb.load(d, d.b, d.dn, b, n0, d.N, kbeg, kend, tid, r0, r1);
    sa.store(as, tid);
    sb.store(bs, tid);
  }
  __syncthreads();
  const int p16 = lane & 15;
  for (int ks = 0; ks < ksteps; ++ks) {
    const int cur = ks & 1;
    const bool more = ks + 1 < ksteps;
    if (more) {
      sa.load(d, d.a, d.dm, a, m0, d.M, kbeg + (ks + 1) * BK, kend, tid, r0, r1);
      sb.load(d, d.b, d.dn, b, n0, d.N, kbeg + (ks + 1) * BK, kend, tid, r0, r1);
    }
    const Elem* const ap = as + cur * SA::ELEMS;
    const Elem* const bp = bs + cur * SB::ELEMS;
    if constexpr (!F32) {
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk) {
        ocn_bf16x8 af[TM], bf[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          if constexpr (A_KC) af[i] = *reinterpret_cast<const ocn_bf16x8*>(ap + (wm + i * 32 + (lane & 31)) * SA::STRIDE + kk * 16 + (lane >> 5) * 8);
          else af[i] = ocn_any_tr(ap + ((lane >> 5) * 8 + (p16 >> 2) + kk * 16) * SA::STRIDE + ((lane >> 4) & 1) * 16 + (p16 & 3) * 4 + wm + i * 32, SA::STRIDE);
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          if constexpr (B_KC) bf[j] = *reinterpret_cast<const ocn_bf16x8*>(bp + (wn + j * 32 + (lane & 31)) * SB::STRIDE + kk * 16 + (lane >> 5) * 8);
          else bf[j] = ocn_any_tr(bp + ((lane >> 5) * 8 + (p16 >> 2) + kk * 16) * SB::STRIDE + ((lane >> 4) & 1) * 16 + (p16 & 3) * 4 + wn + j * 32, SB::STRIDE);
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
      }
    } else {
      // v_mfma_f32_32x32x2_f32: instruction q of four multiplies k = q (lanes 0-31) and k = 4 + q (lanes 32-63)
#pragma unroll
      for (int kk = 0; kk < BK / 8; ++kk) {
        ocn_f32x4 af[TM], bf[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int row = wm + i * 32 + (lane & 31), k = kk * 8 + (lane >> 5) * 4;
          if constexpr (A_KC) af[i] = *reinterpret_cast<const ocn_f32x4*>(ap + row * SA::STRIDE + k);
          else { const Elem* q = ap + k * SA::STRIDE + row; af[i] = ocn_f32x4{q[0], q[SA::STRIDE], q[2 * SA::STRIDE], q[3 * SA::STRIDE]}; }
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int row = wn + j * 32 + (lane & 31), k = kk * 8 + (lane >> 5) * 4;
          if constexpr (B_KC) bf[j] = *reinterpret_cast<const ocn_f32x4*>(bp + row * SB::STRIDE + k);
          else { const Elem* q = bp + k * SB::STRIDE + row; bf[j] = ocn_f32x4{q[0], q[SB::STRIDE], q[2 * SB::STRIDE], q[3 * SB::STRIDE]}; }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i][q], bf[j][q], acc[i][j], 0, 0, 0);
      }
    }
    if (more) {
      sa.store(as + (cur ^ 1) * SA::ELEMS, tid);
      sb.store(bs + (cur ^ 1) * SB::ELEMS, tid);
    }
    __syncthreads();
  }

  // a lane holds column lane % 32 of a 32 x 32 tile; element e is row 8 * (e / 4) + 4 * (lane / 32) + e % 4
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn + j * 32 + (lane & 31);
    if (n >= d.N) continue;
    const int cn = ocn_digit_off(ocn_digits(d.dn, n), d.c_n);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm + i * 32 + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3);
        if (m >= d.M) continue;
        float v = acc[i][j][e];
        if (d.splits > 1) { ws[((long)split * d.M + m) * d.N + n] = v; continue; }
        const OcnDigitVal md = ocn_digits(d.dm, m);
        if constexpr (WIN) { if (d.win_s[0] * md.d1 + r0 >= d.win_pos[0] || d.win_s[1] * md.d2 + r1 >= d.win_pos[1]) continue; }
        const long at = (long)ocn_digit_off(md, d.c_m) + cn;
        if (d.c_bf16) {
          unsigned short* const q = static_cast<unsigned short*>(c) + at;
          if (d.accumulate) v += __uint_as_float((unsigned)*q << 16);
          *q = __builtin_bit_cast(unsigned short, (__bf16)v);
        } else {
          float* const q = static_cast<float*>(c) + at;
          if (d.accumulate) v += *q;
          *q = v;
          if (c2) static_cast<unsigned short*>(c2)[at] = __builtin_bit_cast(unsigned short, (__bf16)v);
        }
      }
    }
  }
}
