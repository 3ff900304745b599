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
// What bounds it: latency of a K step (load, LDS, barrier), about a microsecond, with one or two workgroups per compute
// unit to hide it: matrix cores busy 4 to 5 % and about 5 TB/s out of L2 on the bf16 products of 1777 x 1001 x 771, no
// bank conflicts; in fp32, whose products take sixteen times as long, the matrix cores are busy 26 to 39 %.  Rows at odd
// elements, and the row-contiguous fp32 fragments of four reads, cost more (the last two launches of the dense layer, the
// weight gradient of the convolution).  Kernel trace, as generated kernels with one thread or lane group per element of C
// -> as tiles: the dense layer above, forward and both gradients, 4192 -> 16 + 21 + 25 us; attention scores and their
// product with V over 197 positions, 96 heads, 438 + 569 -> 12 + 9 us; a 3 x 3 convolution of 64 x 32 x 32 positions, 32 ->
// 64 channels in fp32, forward 314 -> 36 us, weight gradient 2106 -> 64 us with its summing launch, input gradient (which
// only the batch and channel axes kept apart: 2048 threads) 28 500 -> 50 us.
//
// Offsets within a batch entry are ints: contract_any_fits (contract_any.hip) says what may come here.
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
// widened, exactly), chunks of 4; else bf16 in LDS, chunks of 8.  WIN: see OcnAnyDesc (1: this is A, 2: B).
//
// A regular operand (see ocn_any_regular) is fetched without a branch, so that the loads of several steps stay in
// flight and each is waited for by count: rows past the end are clamped to the last one (their results are
// never stored), a chunk that runs past the end of its row or of K starts early and is shifted into place on the
// way to LDS, k past the end and positions outside a window are zeroed there.  Irregular operands (a run of
// memory that is not whole chunks) are gathered element by element, clamped and zeroed the same way.
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
  // what one step fetches; mask: chunks that count; an fp32 tile of a bf16 source is widened on the way to LDS (touching
  // the values any earlier would wait for them), unless it was gathered
  struct Set { Chunk c[CH]; unsigned mask; int down; };          // down: KC, elements by which the chunks start early

  int off[KC ? CH : 1];       // KC: row offset of each chunk; else the offset of this thread's rows (chunk start)
  int u0[WIN == 1 ? CH : 1], u1[WIN == 1 ? CH : 1];
  int shift;                  // !KC: elements by which the chunk starts early (0 .. V)

  __device__ __forceinline__ void init(const OcnAnyOperand& o, const OcnDigits& dr, int row0, int rows, int tid) {
    if constexpr (KC) {
      shift = 0;
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        const int r = row0 + tid / PER + j * LINES;
        const OcnDigitVal v = ocn_digits(dr, r < rows ? r : rows - 1);
        off[j] = ocn_digit_off(v, o.row);
        if constexpr (WIN == 1) { u0[j] = v.d1; u1[j] = v.d2; }
      }
    } else {
      const int r = row0 + (tid % PER) * V, at = r + V <= rows ? r : rows - V;
      off[0] = ocn_digit_off(ocn_digits(dr, at), o.row);
      shift = r - at < V ? r - at : V;
    }
  }

  static __device__ __forceinline__ float one(const void* p, bool bf, long i) {
    return bf ? __uint_as_float((unsigned)static_cast<const unsigned short*>(p)[i] << 16) : static_cast<const float*>(p)[i];
  }
  static __device__ __forceinline__ void whole(Chunk& c, const void* p, bool bf, long i) {
    if constexpr (!F32) __builtin_memcpy(&c.u, static_cast<const unsigned short*>(p) + i, 16);
    else if (bf) { ocn_u32x2 t; __builtin_memcpy(&t, static_cast<const unsigned short*>(p) + i, 8); c.u = ocn_u32x4{t.x, t.y, 0, 0}; }
    else __builtin_memcpy(&c.f, static_cast<const float*>(p) + i, 16);
  }
  static __device__ __forceinline__ void widen(Chunk& c) {
    const unsigned x = c.u.x, y = c.u.y;
    c.f = ocn_f32x4{__uint_as_float(x << 16), __uint_as_float(x & 0xFFFF0000u), __uint_as_float(y << 16), __uint_as_float(y & 0xFFFF0000u)};
  }
  // do the taps of k digits (d0, d1) exist; does the position of chunk j's row less those digits lie in A?
  static __device__ __forceinline__ bool tap(const OcnAnyDesc& d, const OcnDigitVal& v, int r0, int r1) {
    return d.win_s[0] * v.d0 + r0 < d.win_taps[0] && d.win_s[1] * v.d1 + r1 < d.win_taps[1];
  }
  __device__ __forceinline__ bool inside(const OcnAnyDesc& d, const OcnDigitVal& v, int j) const {
    return (unsigned)(u0[j] - v.d0) < (unsigned)d.win_lim[0] && (unsigned)(u1[j] - v.d1) < (unsigned)d.win_lim[1];
  }

  // a step of a regular operand; BF: the fp32 tile's source is bf16; TAIL: k may pass kend.  r0, r1: residues
  // (windows only)
  // K1: k is a single digit
  template <bool BF, bool TAIL, bool K1>
  __device__ __forceinline__ void fetch(Set& s, const OcnAnyDesc& d, const OcnAnyOperand& o, const void* p, int k0, int kend, int tid, int r0, int r1) const {
    s.mask = ~0u;
    s.down = 0;
    if constexpr (KC) {
      int k = k0 + (tid % PER) * V;
      if constexpr (TAIL) {
        const int at = k + V <= kend ? k : kend - V;
        s.down = k - at < V ? k - at : V;
        k = at;
      }
      const OcnDigitVal v = K1 ? OcnDigitVal{0, 0, k} : ocn_digits(d.dk, k);
      const int koff = K1 ? k : ocn_digit_off(v, o.k);
      bool t = true;
      if constexpr (WIN != 0) t = tap(d, v, r0, r1);
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        long at = (long)off[j] + koff;
        if constexpr (WIN != 0) {
          const bool there = WIN == 1 ? t && inside(d, v, j) : t;
          if (!there) { at = 0; s.mask &= ~(1u << j); }
        }
        whole(s.c[j], p, BF, at);
      }
    } else {
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        int k = k0 + tid / PER + j * LINES;
        if constexpr (TAIL) { if (k >= kend) { k = kend - 1; s.mask &= ~(1u << j); } }
        const OcnDigitVal v = K1 ? OcnDigitVal{0, 0, k} : ocn_digits(d.dk, k);
        long at = (long)off[0] + (K1 ? k * o.k[2] : ocn_digit_off(v, o.k));
        if constexpr (WIN != 0) { if (!tap(d, v, r0, r1)) { at = 0; s.mask &= ~(1u << j); } }
        whole(s.c[j], p, BF, at);
      }
    }
  }

  // any step of any operand, element by element
  template <bool BF>
  __device__ __forceinline__ void gather(Set& s, const OcnAnyDesc& d, const OcnAnyOperand& o, const OcnDigits& dr, const void* p, int row0, int rows,
                                         int k0, int kend, int tid, int r0, int r1) const {
    s.mask = ~0u;
    s.down = 0;
    const int kk = k0 + (KC ? (tid % PER) * V : tid / PER), rr = row0 + (tid % PER) * V;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
#pragma unroll
      for (int i = 0; i < V; ++i) {
        const int k = KC ? kk + i : kk + j * LINES, r = rr + i;
        const OcnDigitVal v = ocn_digits(d.dk, k < kend ? k : kend - 1);
        bool there = k < kend;
        if constexpr (WIN != 0) there = there && tap(d, v, r0, r1);
        if constexpr (WIN == 1 && KC) there = there && inside(d, v, j);
        long at = ocn_digit_off(v, o.k);
        if constexpr (KC) at += off[j];
        else at += ocn_digit_off(ocn_digits(dr, r < rows ? r : rows - 1), o.row);
        if (!there) at = 0;
        if constexpr (F32) { const float x = one(p, BF, at); s.c[j].s[i] = there ? x : 0.0f; }
        else { const unsigned short x = static_cast<const unsigned short*>(p)[at]; s.c[j].h[i] = there ? x : (unsigned short)0; }
      }
    }
  }

  // 16 bytes down by n elements, zeros from above
  static __device__ __forceinline__ Chunk shifted(const Chunk& raw, int n) {
    Chunk c;
    if constexpr (F32) {
#pragma unroll
      for (int q = 0; q < V; ++q) {
        float x = 0.0f;
#pragma unroll
        for (int w = q; w < V; ++w) x = w == q + n ? raw.s[w] : x;
        c.s[q] = x;
      }
    } else {
      const int w = n >> 1, h = (n & 1) * 16;   // whole words, then half a word
      const unsigned u[4] = {raw.u.x, raw.u.y, raw.u.z, raw.u.w};
      unsigned t[5];
#pragma unroll
      for (int q = 0; q < 5; ++q) {
        unsigned x = 0;
#pragma unroll
        for (int e = q; e < 4; ++e) x = e == q + w ? u[e] : x;
        t[q] = x;
      }
      c.u = ocn_u32x4{__funnelshift_r(t[0], t[1], h), __funnelshift_r(t[1], t[2], h), __funnelshift_r(t[2], t[3], h), __funnelshift_r(t[3], t[4], h)};
    }
    return c;
  }

  // `edge`: rows of the tile run past the end; TAIL: so may k
  template <bool TAIL, bool WIDEN>
  __device__ __forceinline__ void store(const Set& s, Elem* lds, int tid, bool edge) const {
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      Chunk c = s.c[j];
      if constexpr (WIDEN) widen(c);
      if constexpr (!KC) { if (edge) c = shifted(c, shift); }
      if constexpr (KC && TAIL) c = shifted(c, s.down);
      if constexpr (WIN != 0 || TAIL) { if (!(s.mask >> j & 1u)) c.u = ocn_u32x4{0, 0, 0, 0}; }
      *reinterpret_cast<ocn_u32x4*>(lds + (tid / PER + j * LINES) * STRIDE + (tid % PER) * V) = c.u;
    }
  }
};

// Whole chunks only: along k (KC) or along the rows, memory runs in multiples of a chunk.
template <bool KC, bool F32>
__device__ __forceinline__ bool ocn_any_regular(const OcnAnyOperand& o, const OcnDigits& dr, const OcnDigits& dk, int rows) {
  constexpr int V = F32 ? 4 : 8;
  if constexpr (KC) return o.k[2] == 1 && (dk.n == 1 || dk.e2 % V == 0);
  else return o.row[2] == 1 && rows >= V && (dr.n == 1 || dr.e2 % V == 0);
}

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

struct OcnAnyNo { static constexpr bool value = false; };
struct OcnAnyYes { static constexpr bool value = true; };

// Orders LDS only: fetches stay in flight across it.
__device__ __forceinline__ void ocn_any_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Folded consumers of a bf16 result (GemmArgs): a bias by column, relu into a second tensor or in place.  The second
// tensor is laid out as C and found from where C's element is, in every batch entry.
struct OcnAnyEpilogue {
  const unsigned short* bias;
  long relu_from_c;           // bytes; 0: none
  int relu_c;
};

// One BM x BN tile (or, with splits, its share `split` of K) by 256 threads = 2 x 2 wavefronts (4 x 1 for tiles of 32
// columns, 1 x 4 for tiles of 32 rows).  a, b, c, c2: operands at the batch entry; ws: with splits, where partial
// sums of this entry go ([split][M][N] fp32).  c2: a bf16 tensor of C's layout that receives the rounded fp32
// result, or null.  PF: steps of K in flight in registers ahead of the one being multiplied.
template <int BM, int BN, bool A_KC, bool B_KC, bool ABF, bool BBF, bool WIN, int PF>
__device__ __forceinline__ void ocn_any_tile(const OcnAnyDesc& d, const void* a, const void* b, void* c, void* c2, float* ws, const OcnAnyEpilogue& ep,
                                             int tm, int tn, int split, int r0, int r1, unsigned char* smem) {
  constexpr bool F32 = !(ABF && BBF);
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
  // a residue that no tap has (an axis of fewer taps than its step) sums nothing and reads nothing: `b` is then where
  // the tap would be, past the weights as they are stored
  bool none = false;
  if constexpr (WIN) {
    none = r0 >= d.win_taps[0] || r1 >= d.win_taps[1];
    if (none && d.accumulate) return;
  }
  const int ksteps = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;
  const bool ra = ocn_any_regular<A_KC, F32>(d.a, d.dm, d.dk, d.M), rb = ocn_any_regular<B_KC, F32>(d.b, d.dn, d.dk, d.N);
  const bool edge_a = m0 + BM > d.M, edge_b = n0 + BN > d.N;

  SA sa; SB sb;
  sa.init(d.a, d.dm, m0, d.M, tid);
  sb.init(d.b, d.dn, n0, d.N, tid);
  if (!(ra && rb)) sa.shift = sb.shift = 0;      // (gathered at their own rows)
  typename SA::Set qa[PF];
  typename SB::Set qb[PF];
  ocn_f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  auto fetch = [&](typename SA::Set& x, typename SB::Set& y, int k, auto tail, auto single) __attribute__((always_inline)) {
    constexpr bool T = decltype(tail)::value, K1 = decltype(single)::value;
    sa.template fetch<ABF, T, K1>(x, d, d.a, a, k, kend, tid, r0, r1);
    sb.template fetch<BBF, T, K1>(y, d, d.b, b, k, kend, tid, r0, r1);
  };
  auto gather = [&](typename SA::Set& x, typename SB::Set& y, int t) __attribute__((always_inline)) {
    const int k = kbeg + t * BK;
    sa.template gather<ABF>(x, d, d.a, d.dm, a, m0, d.M, k, kend, tid, r0, r1);
    sb.template gather<BBF>(y, d, d.b, d.dn, b, n0, d.N, k, kend, tid, r0, r1);
  };
  using Yes = OcnAnyYes;
  using No = OcnAnyNo;
  const int p16 = lane & 15;
  auto multiply = [&](int cur) __attribute__((always_inline)) {
    const Elem* const ap = as + cur * SA::ELEMS;
    const Elem* const bp = bs + cur * SB::ELEMS;
    // all fragments of the step first: with few waves per SIMD nothing else would hide their latency
    if constexpr (!F32) {
      ocn_bf16x8 af[BK / 16][TM], bf[BK / 16][TN];
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          if constexpr (A_KC) af[kk][i] = *reinterpret_cast<const ocn_bf16x8*>(ap + (wm + i * 32 + (lane & 31)) * SA::STRIDE + kk * 16 + (lane >> 5) * 8);
          else af[kk][i] = ocn_any_tr(ap + ((lane >> 5) * 8 + (p16 >> 2) + kk * 16) * SA::STRIDE + ((lane >> 4) & 1) * 16 + (p16 & 3) * 4 + wm + i * 32, SA::STRIDE);
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          if constexpr (B_KC) bf[kk][j] = *reinterpret_cast<const ocn_bf16x8*>(bp + (wn + j * 32 + (lane & 31)) * SB::STRIDE + kk * 16 + (lane >> 5) * 8);
          else bf[kk][j] = ocn_any_tr(bp + ((lane >> 5) * 8 + (p16 >> 2) + kk * 16) * SB::STRIDE + ((lane >> 4) & 1) * 16 + (p16 & 3) * 4 + wn + j * 32, SB::STRIDE);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kk][i], bf[kk][j], acc[i][j], 0, 0, 0);
    } else {
      // v_mfma_f32_32x32x2_f32: instruction q of four multiplies k = q (lanes 0-31) and k = 4 + q (lanes 32-63)
      ocn_f32x4 af[BK / 8][TM], bf[BK / 8][TN];
#pragma unroll
      for (int kk = 0; kk < BK / 8; ++kk) {
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int row = wm + i * 32 + (lane & 31), k = kk * 8 + (lane >> 5) * 4;
          if constexpr (A_KC) af[kk][i] = *reinterpret_cast<const ocn_f32x4*>(ap + row * SA::STRIDE + k);
          else { const Elem* q = ap + k * SA::STRIDE + row; af[kk][i] = ocn_f32x4{q[0], q[SA::STRIDE], q[2 * SA::STRIDE], q[3 * SA::STRIDE]}; }
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int row = wn + j * 32 + (lane & 31), k = kk * 8 + (lane >> 5) * 4;
          if constexpr (B_KC) bf[kk][j] = *reinterpret_cast<const ocn_f32x4*>(bp + row * SB::STRIDE + k);
          else { const Elem* q = bp + k * SB::STRIDE + row; bf[kk][j] = ocn_f32x4{q[0], q[SB::STRIDE], q[2 * SB::STRIDE], q[3 * SB::STRIDE]}; }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < BK / 8; ++kk)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[kk][i][q], bf[kk][j][q], acc[i][j], 0, 0, 0);
    }
  };
  auto put = [&](const typename SA::Set& x, const typename SB::Set& y, int buf, auto tail, auto fetched) __attribute__((always_inline)) {
    constexpr bool T = decltype(tail)::value, R = decltype(fetched)::value && F32;
    sa.template store<T, R && ABF>(x, as + buf * SA::ELEMS, tid, edge_a);
    sb.template store<T, R && BBF>(y, bs + buf * SB::ELEMS, tid, edge_b);
  };

  // Regular operands.  At step t its tile is in LDS buffer t & 1 and those of the next PF - 1 steps are on their way
  // into the other sets; the partial step at the end, if there is one, has been fetched with the first ones.
  // Every step fetches (the last ones the last tile again), so that the loads in flight can be counted.
  auto pipeline = [&](auto single) __attribute__((always_inline)) {
    const int n = kend > kbeg ? (kend - kbeg) / BK : 0;
    typename SA::Set ta;
    typename SB::Set tb;
    auto at = [&](int t) __attribute__((always_inline)) { return kbeg + (t < n ? t : n - 1) * BK; };
    if (n > 0) {
#pragma unroll
      for (int p = 0; p < PF; ++p) fetch(qa[p], qb[p], at(p), No{}, single);
    }
    if (n < ksteps) fetch(ta, tb, kbeg + n * BK, Yes{}, single);
    __builtin_amdgcn_sched_barrier(0);
    if (n > 0) {
      put(qa[0], qb[0], 0, No{}, Yes{});
      ocn_any_barrier();
      for (int t = 0; t < n; t += PF) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
          if (t + p >= n) break;
          fetch(qa[p], qb[p], at(t + p + PF), No{}, single);
          __builtin_amdgcn_sched_barrier(0);
          multiply((t + p) & 1);
          __builtin_amdgcn_sched_barrier(0);
          if (t + p + 1 < n) put(qa[(p + 1) % PF], qb[(p + 1) % PF], (t + p + 1) & 1, No{}, Yes{});
          ocn_any_barrier();
        }
      }
    }
    if (n < ksteps) {
      put(ta, tb, n & 1, Yes{}, Yes{});
      ocn_any_barrier();
      multiply(n & 1);
    }
  };
  if (none) {
  } else if (ra && rb) {
    if (d.dk.n == 1) pipeline(Yes{}); else pipeline(No{});
  } else {
    if (ksteps > 0) gather(qa[0], qb[0], 0);
    if (ksteps > 0) put(qa[0], qb[0], 0, No{}, No{});
    ocn_any_barrier();
    for (int t = 0; t < ksteps; ++t) {
      if (t + 1 < ksteps) gather(qa[0], qb[0], t + 1);
      multiply(t & 1);
      if (t + 1 < ksteps) put(qa[0], qb[0], (t + 1) & 1, No{}, No{});
      ocn_any_barrier();
    }
  }

  // A lane holds column lane % 32 of a 32 x 32 tile; element e is row 8 * (e / 4) + 4 * (lane / 32) + e % 4.  One
  // form of the store per kind of result, picked once: a launch is short, and code that is run once per
  // launch is fetched once per launch.  `each(j, i, n, cn, e, at)` is called for what exists.
  auto cells = [&](auto single, auto each) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + wn + j * 32 + (lane & 31);
      if (n >= d.N) continue;
      const int cn = ocn_digit_off(ocn_digits(d.dn, n), d.c_n);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int mb = m0 + wm + i * 32 + (lane >> 5) * 4;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int m = mb + (e >> 2) * 8 + (e & 3);
          if (m >= d.M) continue;
          if constexpr (decltype(single)::value) each(j, i, n, e, m, m * d.c_m[2] + cn);
          else {
            const OcnDigitVal md = ocn_digits(d.dm, m);
            if constexpr (WIN) { if (d.win_s[0] * md.d1 + r0 >= d.win_pos[0] || d.win_s[1] * md.d2 + r1 >= d.win_pos[1]) continue; }
            each(j, i, n, e, m, ocn_digit_off(md, d.c_m) + cn);
          }
        }
      }
    }
  };
  auto to_bf16 = [](float v) __attribute__((always_inline)) { return __builtin_bit_cast(unsigned short, (__bf16)v); };
  float* const cf = static_cast<float*>(c);
  unsigned short* const ch = static_cast<unsigned short*>(c);
  auto finish = [&](auto single) __attribute__((always_inline)) {
    if (!d.c_bf16 && !d.accumulate && !c2)
      cells(single, [&](int j, int i, int, int e, int, int at) __attribute__((always_inline)) { cf[at] = acc[i][j][e]; });
    else if (!d.c_bf16) {
      if (d.accumulate) cells(single, [&](int j, int i, int, int e, int, int at) __attribute__((always_inline)) { acc[i][j][e] += cf[at]; });
      cells(single, [&](int j, int i, int, int e, int, int at) __attribute__((always_inline)) {
        cf[at] = acc[i][j][e];
        if (c2) static_cast<unsigned short*>(c2)[at] = to_bf16(acc[i][j][e]);
      });
    } else if (!d.accumulate && !ep.bias && !ep.relu_from_c && !ep.relu_c)
      cells(single, [&](int j, int i, int, int e, int, int at) __attribute__((always_inline)) { ch[at] = to_bf16(acc[i][j][e]); });
    else {
      if (d.accumulate) cells(single, [&](int j, int i, int, int e, int, int at) __attribute__((always_inline)) { acc[i][j][e] += __uint_as_float((unsigned)ch[at] << 16); });
      cells(single, [&](int j, int i, int n, int e, int, int at) __attribute__((always_inline)) {
        unsigned short x = to_bf16(acc[i][j][e]);
        if (ep.bias) x = to_bf16(__uint_as_float((unsigned)x << 16) + __uint_as_float((unsigned)ep.bias[n] << 16));
        const unsigned short y = (x & 0x8000u) || (x & 0x7FFFu) > 0x7F80u ? (unsigned short)0 : x;   // fmaxf(0, x)
        if (ep.relu_from_c) *reinterpret_cast<unsigned short*>(reinterpret_cast<char*>(ch + at) + ep.relu_from_c) = y;
        ch[at] = ep.relu_c ? y : x;
      });
    }
  };
  if constexpr (WIN) {
    // A position that a tap does not reach multiplied that tap's weights by zero, which is no term of its sum: it turned
    // NaN if one of them was infinite or NaN.  What has come out as NaN is summed again, one cell at a time, from its own
    // terms (nothing, where the weights are finite), and is NaN only if that sum is.  64 x 34 x 34 x 32 results of a 3 x 3
    // layer with 64 channels behind it, fp32: 49 us, 0.47 ms with a NaN among the weights (one lane a cell, loads waited for).
    static_assert(16 * TM * TN <= 32, "a bit a cell");
    unsigned again = 0;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) again |= (unsigned)((__float_as_uint(acc[i][j][e]) & 0x7FFFFFFFu) > 0x7F800000u) << ((i * TN + j) * 16 + e);
    if (d.accumulate) cells(No{}, [&](int j, int i, int, int e, int, int at) __attribute__((always_inline)) { acc[i][j][e] += cf[at]; });
    cells(No{}, [&](int j, int i, int, int e, int, int at) __attribute__((always_inline)) { if (!(again >> ((i * TN + j) * 16 + e) & 1u)) cf[at] = acc[i][j][e]; });
    for (; again; again &= again - 1) {
      const int cell = __builtin_ctz(again), e = cell & 15, j = (cell >> 4) % TN, i = (cell >> 4) / TN;
      const int n = n0 + wn + j * 32 + (lane & 31), m = m0 + wm + i * 32 + (lane >> 5) * 4 + (e >> 2) * 8 + (e & 3);
      if (m >= d.M || n >= d.N) continue;
      const OcnDigitVal md = ocn_digits(d.dm, m), nd = ocn_digits(d.dn, n);
      if (d.win_s[0] * md.d1 + r0 >= d.win_pos[0] || d.win_s[1] * md.d2 + r1 >= d.win_pos[1]) continue;
      float v = 0.0f;
#pragma unroll 1
      for (int t0 = 0; d.win_s[0] * t0 + r0 < d.win_taps[0]; ++t0) {
        if ((unsigned)(md.d1 - t0) >= (unsigned)d.win_lim[0]) continue;
#pragma unroll 1
        for (int t1 = 0; d.win_s[1] * t1 + r1 < d.win_taps[1]; ++t1) {
          if ((unsigned)(md.d2 - t1) >= (unsigned)d.win_lim[1]) continue;
          long at_a = (long)ocn_digit_off(md, d.a.row) + ocn_digit_off({t0, t1, 0}, d.a.k), at_b = (long)ocn_digit_off(nd, d.b.row) + ocn_digit_off({t0, t1, 0}, d.b.k);
          for (int k = 0; k < d.dk.e2; ++k, at_a += d.a.k[2], at_b += d.b.k[2]) v = __builtin_fmaf(SA::one(a, ABF, at_a), SB::one(b, BBF, at_b), v);
        }
      }
      const int at = ocn_digit_off(md, d.c_m) + ocn_digit_off(nd, d.c_n);
      cf[at] = d.accumulate ? v + cf[at] : v;
    }
  } else if (d.splits > 1) {
    float* const w = ws + (long)split * d.M * d.N;
    cells(Yes{}, [&](int j, int i, int n, int e, int m, int) __attribute__((always_inline)) { w[m * d.N + n] = acc[i][j][e]; });
  } else if (d.dm.n == 1) finish(Yes{});
  else finish(No{});
}
