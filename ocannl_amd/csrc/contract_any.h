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
// What bounds it: in bf16 what the tiles read out of L2.  64 of K of a 64 x 64 tile take 0.29 us where every compute unit has
// one, 0.56 us with two: 14 TB/s, the rate at which tiles reach LDS in every kernel here; alone on a unit the latency of a
// step (0.27 us).  Start, stores and launch are 4.5 to 6 us.  Rows at odd elements cost 1.2 to 1.5 times as much.  With
// fp32 operands in parts 1.0 us (two: 1.9): LDS, a kilobyte of fragments for every 32 cycles of products of a wavefront's
// 32 x 32 cells, beside the 130 vector instructions that split 16 values; 128 x 128 tiles 0.72 us per 64 x 64 cells.
// 1777 x 771 x 1001, k-contiguous: bf16 15.6 us with a loop that waited for all of its loads in every turn, 14.4 now; fp32
// 40.2 us on the fp32 instructions, 32.3 in parts; both row-contiguous 16.9 -> 15.9 and 49.9 -> 35.7.  4001 x 4003 x 1001 in
// fp32 (128 x 128 tiles) 313 -> 196 us; the convolution below with both gradients 137 -> 117 us.
// Kernel trace, as generated kernels with one thread or lane group per element of C -> as tiles, first version: a dense
// layer of 1777 x 1001 -> 771, forward and both gradients, 4192 -> 16 + 21 + 25 us; attention scores and their product with V
// over 197 positions, 96 heads, 438 + 569 -> 12 + 9 us; a 3 x 3 convolution of 64 x 32 x 32 positions, 32 -> 64 channels in
// fp32, forward 314 -> 36 us, weight gradient 2106 -> 64 us with its summing launch, input gradient (which only the batch
// and channel axes kept apart: 2048 threads) 28 500 -> 50 us.
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

// How an operand lies in LDS: bf16, both operands being bf16 (chunks of 8); else in chunks of 4, as the three bf16 parts
// of its fp32 values, each in a plane of its own, or as its bf16 values beside an operand in parts; or, where parts do
// not do (see ocn_any_tile), as fp32, a bf16 source widened.
constexpr int kOcnBf16 = 0, kOcnWhole = 1, kOcnParts = 2, kOcnPart = 3;

// Operands multiplied in parts are taken kOcnScale times as large, a bf16 one beside them too, and the sums kOcnUnscale times: no
// part of any fp32 value is then a subnormal bf16, next to which the matrix cores keep fewer bits of a product.  The bf16
// operand's share is five instructions for two values, 2 to 7 % of a launch; watching for its subnormal values, to multiply
// their tiles again, takes three, but the register it needs costs the fourth workgroup of a compute unit (4001 x 4003 x 250,
// row-contiguous: 56.9 us without either, 58.2 scaled, 62.8 watched).
constexpr float kOcnScale = 0x1p23f, kOcnUnscale = 0x1p-46f;

// Two values rounded to bf16 (to nearest even), x in the low half.
__device__ __forceinline__ unsigned ocn_bf16_pair(float x, float y) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{x, y}), bf16x2));
}

// Two bf16 values, kOcnScale times as large (exactly).
__device__ __forceinline__ unsigned ocn_bf16_scaled(unsigned w) {
  return ocn_bf16_pair(__uint_as_float(w << 16) * kOcnScale, __uint_as_float(w & 0xFFFF0000u) * kOcnScale);
}

// ROWS x BK tile of one operand: global -> registers -> LDS, 256 threads.  WIN: see OcnAnyDesc (1: this is A, 2: B).
// Planes of parts have no padding: the 16-byte pieces of a line change places so that the lanes of a fragment read meet
// all banks (k-contiguous: by row, so that 16 rows do; else by k-line, so that the four k-lines of a transposing read do).
//
// A regular operand (see ocn_any_regular) is fetched without a branch, so that the loads of several steps stay in
// flight and each is waited for by count: rows past the end are clamped to the last one (their results are
// never stored), a chunk that runs past the end of its row or of K starts early and is shifted into place on the
// way to LDS, k past the end and positions outside a window are zeroed there.  Irregular operands (a run of
// memory that is not whole chunks) are gathered element by element, clamped and zeroed the same way.
template <int ROWS, bool KC, int MODE, int WIN, int BKE>
struct OcnAnyStage {
  static constexpr bool F32 = MODE == kOcnWhole || MODE == kOcnParts;   // registers hold fp32
  static constexpr bool PLANES = MODE == kOcnParts || MODE == kOcnPart;
  static constexpr int V = MODE == kOcnBf16 ? 8 : 4, BK = BKE;
  static constexpr int PER = KC ? BK / V : ROWS / V;             // chunks per contiguous line
  static constexpr int CH = ROWS * BK / V / 256;                 // chunks per thread
  static constexpr int LINES = 256 / PER;                        // lines one pass of the workgroup covers
  static constexpr int PAD = PLANES ? 0 : F32 ? (KC ? 4 : 8) : (KC ? 8 : 32);
  static constexpr int STRIDE = (KC ? BK : ROWS) + PAD;          // LDS elements per line
  static constexpr int PLANE = (KC ? ROWS : BK) * STRIDE, ELEMS = (MODE == kOcnParts ? 3 : 1) * PLANE;
  using Elem = typename ocn_if<MODE == kOcnWhole, float, unsigned short>::type;
  static constexpr int RP = KC ? 128 / BK : 1, PPR = KC ? BK / 8 : 1;   // planes: rows per 256 bytes, pieces per row
  static_assert(!PLANES || LINES % (KC ? RP * PPR : 4) == 0, "one place for all chunks of a thread");
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
    if constexpr (MODE == kOcnBf16) __builtin_memcpy(&c.u, static_cast<const unsigned short*>(p) + i, 16);
    else if (MODE == kOcnPart || bf) { ocn_u32x2 t; __builtin_memcpy(&t, static_cast<const unsigned short*>(p) + i, 8); c.u = ocn_u32x4{t.x, t.y, 0, 0}; }
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

  // where a thread's first chunk goes in a plane
  static __device__ __forceinline__ int place(int tid) {
    const int line = tid / PER, c = tid % PER;
    const int turn = KC ? (line / RP) & (PPR - 1) : ROWS >= 128 ? (line & 3) << 2 : ROWS == 64 ? (line >> 1 & 1) << 2 : 0;
    return line * STRIDE + ((c >> 1) ^ turn) * 8 + (c & 1) * 4;
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
      if constexpr (!PLANES) *reinterpret_cast<ocn_u32x4*>(lds + (tid / PER + j * LINES) * STRIDE + (tid % PER) * V) = c.u;
      else {
        Elem* const to = lds + place(tid) + j * LINES * STRIDE;
        put<0>(c, to);
        if constexpr (MODE == kOcnParts) { put<1>(c, to); put<2>(c, to); }
      }
    }
  }
  // part P of a chunk to its plane; what is left of the values stays in the chunk
  template <int P>
  static __device__ __forceinline__ void put(Chunk& c, Elem* to) {
    if constexpr (MODE == kOcnPart) *reinterpret_cast<ocn_u32x2*>(to) = ocn_u32x2{ocn_bf16_scaled(c.u.x), ocn_bf16_scaled(c.u.y)};
    else {
      ocn_f32x4& r = c.f;
      if constexpr (P == 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) r[q] *= kOcnScale;
      }
      const unsigned x = ocn_bf16_pair(r.x, r.y), y = ocn_bf16_pair(r.z, r.w);
      *reinterpret_cast<ocn_u32x2*>(to + P * PLANE) = ocn_u32x2{x, y};
      if constexpr (P < 2) r = ocn_f32x4{r.x - __uint_as_float(x << 16), r.y - __uint_as_float(x & 0xFFFF0000u), r.z - __uint_as_float(y << 16), r.w - __uint_as_float(y & 0xFFFF0000u)};
    }
  }
  // the store of a whole step in pieces, to go between matrix instructions: ready() first, then units 0 .. UNITS - 1
  static constexpr int UNITS = CH * (MODE == kOcnParts ? 3 : 1);
  __device__ __forceinline__ void ready(Set& s, bool edge) const {
    if constexpr (!KC) {
      if (edge) {
#pragma unroll
        for (int j = 0; j < CH; ++j) s.c[j] = shifted(s.c[j], shift);
      }
    }
  }
  template <int U>
  __device__ __forceinline__ void unit(Set& s, Elem* lds, int tid) const {
    constexpr int J = U / (UNITS / CH), P = U % (UNITS / CH);
    if constexpr (WIN != 0 && P == 0) { if (!(s.mask >> J & 1u)) s.c[J].u = ocn_u32x4{0, 0, 0, 0}; }
    put<P>(s.c[J], lds + place(tid) + J * LINES * STRIDE);
  }
  static __device__ __forceinline__ ocn_bf16x8 part(const Elem* plane, int row, int kk, int lane);
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

// fragment (32 rows from `row`, 16 k from kk * 16) out of a plane
template <int ROWS, bool KC, int MODE, int WIN, int BKE>
__device__ __forceinline__ ocn_bf16x8 OcnAnyStage<ROWS, KC, MODE, WIN, BKE>::part(const Elem* plane, int row, int kk, int lane) {
  if constexpr (KC) return *reinterpret_cast<const ocn_bf16x8*>(plane + (row + (lane & 31)) * STRIDE + ((kk * 2 + (lane >> 5)) ^ (((lane & 31) / RP) & (PPR - 1))) * 8);
  else {
    const int p = lane & 15, turn = ROWS >= 128 ? (p >> 2) * 32 : ROWS == 64 ? (p >> 3) * 32 : 0;
    return ocn_any_tr(plane + (kk * 16 + (lane >> 5) * 8 + (p >> 2)) * STRIDE + ((row + ((lane >> 4) & 1) * 16 + (p & 3) * 4) ^ turn), STRIDE);
  }
}

template <bool ABF, bool BBF, bool PARTS> struct OcnAnyModes {
  static constexpr int A = ABF && BBF ? kOcnBf16 : !PARTS ? kOcnWhole : ABF ? kOcnPart : kOcnParts;
  static constexpr int B = ABF && BBF ? kOcnBf16 : !PARTS ? kOcnWhole : BBF ? kOcnPart : kOcnParts;
};
// k of a step: parts of 128 x 128 tiles take half as much, so that two workgroups share a compute unit's LDS
template <int BM, int BN, bool ABF, bool BBF, bool PARTS>
constexpr int ocn_any_bk() { return ABF && BBF ? 64 : PARTS && BM == 128 && BN == 128 ? 16 : 32; }
template <int BM, int BN, bool A_KC, bool B_KC, bool ABF, bool BBF, bool PARTS>
constexpr int ocn_any_smem() {
  constexpr int BK = ocn_any_bk<BM, BN, ABF, BBF, PARTS>();
  using M = OcnAnyModes<ABF, BBF, PARTS>;
  using SA = OcnAnyStage<BM, A_KC, M::A, 0, BK>;
  using SB = OcnAnyStage<BN, B_KC, M::B, 0, BK>;
  return 2 * (int)sizeof(typename SA::Elem) * (SA::ELEMS + SB::ELEMS);
}

template <int I> struct OcnAnyInt { static constexpr int value = I; };
// f(0), f(1), ..  f(N - 1) with compile-time numbers
template <int N, int I = 0, typename F>
__device__ __forceinline__ void ocn_any_each(F&& f) {
  if constexpr (I < N) { f(OcnAnyInt<I>{}); ocn_any_each<N, I + 1>(f); }
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
//
// PARTS: an fp32 operand is multiplied as the sum of three bf16 values, which it is exactly, on the bf16 matrix cores: six of the
// nine products of two such operands (the others are below 2^-24 of the whole), all three with a bf16 operand.  Tiles
// with results that are not finite (an infinity has no remainder; sums from 2^81 on and values from 2^104 on overflow) are
// multiplied again with fp32 instructions (1777 x 771 x 1001, one in every tile: 86 us, 35 without, 43 on those instructions alone).
template <int BM, int BN, bool A_KC, bool B_KC, bool ABF, bool BBF, bool WIN, int PF, bool PARTS>
__device__ __forceinline__ void ocn_any_tile(const OcnAnyDesc& d, const void* a, const void* b, void* c, void* c2, float* ws, const OcnAnyEpilogue& ep,
                                             int tm, int tn, int split, int r0, int r1, unsigned char* smem) {
  constexpr bool F32 = !(ABF && BBF);
  constexpr int BK = ocn_any_bk<BM, BN, ABF, BBF, PARTS>();
  using SA = OcnAnyStage<BM, A_KC, OcnAnyModes<ABF, BBF, PARTS>::A, WIN ? 1 : 0, BK>;
  using SB = OcnAnyStage<BN, B_KC, OcnAnyModes<ABF, BBF, PARTS>::B, WIN ? 2 : 0, BK>;
  using WA = OcnAnyStage<BM, A_KC, kOcnWhole, WIN ? 1 : 0, 32>;
  using WB = OcnAnyStage<BN, B_KC, kOcnWhole, WIN ? 2 : 0, 32>;
  using Elem = typename SA::Elem;
  constexpr int GN = BN == 32 ? 1 : BM == 32 ? 4 : 2, GM = 4 / GN, WM = BM / GM, WN = BN / GN, TM = WM / 32, TN = WN / 32;
  Elem* const as = reinterpret_cast<Elem*>(smem);
  Elem* const bs = as + SA::ELEMS;
  constexpr int STAGE = SA::ELEMS + SB::ELEMS;
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
  // a step of fp32 operands
  auto whole = [&](const float* fa, const float* fb) __attribute__((always_inline)) {
    // v_mfma_f32_32x32x2_f32: instruction q of four multiplies k = q (lanes 0-31) and k = 4 + q (lanes 32-63)
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      ocn_f32x4 af[TM], bf[TN];
      const int k = kk * 8 + (lane >> 5) * 4;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int row = wm + i * 32 + (lane & 31);
        if constexpr (A_KC) af[i] = *reinterpret_cast<const ocn_f32x4*>(fa + row * WA::STRIDE + k);
        else { const float* q = fa + k * WA::STRIDE + row; af[i] = ocn_f32x4{q[0], q[WA::STRIDE], q[2 * WA::STRIDE], q[3 * WA::STRIDE]}; }
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int row = wn + j * 32 + (lane & 31);
        if constexpr (B_KC) bf[j] = *reinterpret_cast<const ocn_f32x4*>(fb + row * WB::STRIDE + k);
        else { const float* q = fb + k * WB::STRIDE + row; bf[j] = ocn_f32x4{q[0], q[WB::STRIDE], q[2 * WB::STRIDE], q[3 * WB::STRIDE]}; }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i][q], bf[j][q], acc[i][j], 0, 0, 0);
    }
  };
  // The products of a step; `units`: how many pieces of the next step's stores there are, `unit(i)` is piece i.  They go
  // evenly between the products and are pinned there: a wavefront alone on its SIMD hides nothing else.
  auto multiply = [&](int cur, auto units, auto unit) __attribute__((always_inline)) {
    const Elem* const ap = as + cur * STAGE;
    const Elem* const bp = bs + cur * STAGE;
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
    } else if constexpr (!PARTS) whole(ap, bp);
    else {
      constexpr int NA = SA::ELEMS / SA::PLANE, NB = SB::ELEMS / SB::PLANE;
      ocn_bf16x8 af[BK / 16][NA][TM], bf[BK / 16][NB][TN];
#pragma unroll
      for (int kk = 0; kk < BK / 16; ++kk) {
#pragma unroll
        for (int p = 0; p < NA; ++p)
#pragma unroll
          for (int i = 0; i < TM; ++i) af[kk][p][i] = SA::part(ap + p * SA::PLANE, wm + i * 32, kk, lane);
#pragma unroll
        for (int p = 0; p < NB; ++p)
#pragma unroll
          for (int j = 0; j < TN; ++j) bf[kk][p][j] = SB::part(bp + p * SB::PLANE, wn + j * 32, kk, lane);
      }
      __builtin_amdgcn_sched_barrier(0);
      constexpr int NQ = NA * NB == 9 ? 6 : 3, ALL = BK / 16 * NQ * TM * TN, U = decltype(units)::value;
      ocn_any_each<ALL>([&](auto mc) __attribute__((always_inline)) {
        constexpr int m = decltype(mc)::value, kk = m / (NQ * TM * TN), q = m / (TM * TN) % NQ, i = m / TN % TM, j = m % TN;
        // small products first: parts 0 2, 2 0, 1 1, 0 1, 1 0, 0 0, or 2, 1, 0 of the operand that has three
        constexpr int pa = NQ == 6 ? (q == 1 ? 2 : q == 2 || q == 4 ? 1 : 0) : NA == 3 ? 2 - q : 0;
        constexpr int pb = NQ == 6 ? (q == 0 ? 2 : q == 2 || q == 3 ? 1 : 0) : NB == 3 ? 2 - q : 0;
        ocn_any_each<U>([&](auto uc) __attribute__((always_inline)) { if constexpr (decltype(uc)::value * ALL / U == m) unit(uc); });
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[kk][pa][i], bf[kk][pb][j], acc[i][j], 0, 0, 0);
        if constexpr (U > 0) __builtin_amdgcn_sched_barrier(0);
      });
    }
  };
  using None = OcnAnyInt<0>;
  auto nothing = [](auto) __attribute__((always_inline)) {};
  auto put = [&](const typename SA::Set& x, const typename SB::Set& y, int buf, auto tail, auto fetched) __attribute__((always_inline)) {
    constexpr bool T = decltype(tail)::value, R = decltype(fetched)::value && F32 && !PARTS;
    sa.template store<T, R && ABF>(x, as + buf * STAGE, tid, edge_a);
    sb.template store<T, R && BBF>(y, bs + buf * STAGE, tid, edge_b);
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
      // (no branch in a turn of the loop: a path on which a set is not stored would make the next one wait for every load)
      int t = 0;
      for (; t + PF <= n; t += PF) {
#pragma unroll
        for (int p = 0; p < PF; ++p) {
          fetch(qa[p], qb[p], at(t + p + PF), No{}, single);
          typename SA::Set& na = qa[(p + 1) % PF];
          typename SB::Set& nb = qb[(p + 1) % PF];
          const int to = (t + p + 1) & 1;
          if constexpr (F32 && PARTS) {
            sa.ready(na, edge_a);
            sb.ready(nb, edge_b);
            __builtin_amdgcn_sched_barrier(0);
            multiply((t + p) & 1, OcnAnyInt<SA::UNITS + SB::UNITS>{}, [&](auto uc) __attribute__((always_inline)) {
              constexpr int u = decltype(uc)::value;
              if constexpr (u < SA::UNITS) sa.template unit<u>(na, as + to * STAGE, tid);
              else sb.template unit<u - SA::UNITS>(nb, bs + to * STAGE, tid);
            });
          } else {
            __builtin_amdgcn_sched_barrier(0);
            multiply((t + p) & 1, None{}, nothing);
            __builtin_amdgcn_sched_barrier(0);
            put(na, nb, to, No{}, Yes{});
          }
          ocn_any_barrier();
        }
      }
#pragma unroll
      for (int p = 0; p + 1 < PF; ++p) {
        if (t + p >= n) break;
        multiply((t + p) & 1, None{}, nothing);
        if (t + p + 1 < n) put(qa[(p + 1) % PF], qb[(p + 1) % PF], (t + p + 1) & 1, No{}, Yes{});
        ocn_any_barrier();
      }
    }
    if (n < ksteps) {
      put(ta, tb, n & 1, Yes{}, Yes{});
      ocn_any_barrier();
      multiply(n & 1, None{}, nothing);
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
      multiply(t & 1, None{}, nothing);
      if (t + 1 < ksteps) put(qa[0], qb[0], (t + 1) & 1, No{}, No{});
      ocn_any_barrier();
    }
  }

  if constexpr (F32 && PARTS) {
    float nan = 0.0f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) nan = __builtin_fmaf(acc[i][j][e], 0.0f, nan);
    if (!__syncthreads_or(nan != nan)) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] *= kOcnUnscale;
    } else {
      WA wa; WB wb;
      wa.init(d.a, d.dm, m0, d.M, tid);
      wb.init(d.b, d.dn, n0, d.N, tid);
      if (!(ra && rb)) wa.shift = wb.shift = 0;
      float* const fa = reinterpret_cast<float*>(smem);
      float* const fb = fa + WA::ELEMS;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
#pragma unroll 1
      for (int k0 = kbeg; k0 < kend; k0 += 32) {
        typename WA::Set xa;
        typename WB::Set xb;
        if (ra && rb) {
          wa.template fetch<ABF, true, false>(xa, d, d.a, a, k0, kend, tid, r0, r1);
          wb.template fetch<BBF, true, false>(xb, d, d.b, b, k0, kend, tid, r0, r1);
          ocn_any_barrier();
          wa.template store<true, ABF>(xa, fa, tid, edge_a);
          wb.template store<true, BBF>(xb, fb, tid, edge_b);
        } else {
          wa.template gather<ABF>(xa, d, d.a, d.dm, a, m0, d.M, k0, kend, tid, r0, r1);
          wb.template gather<BBF>(xb, d, d.b, d.dn, b, n0, d.N, k0, kend, tid, r0, r1);
          ocn_any_barrier();
          wa.template store<true, false>(xa, fa, tid, edge_a);
          wb.template store<true, false>(xb, fb, tid, edge_b);
        }
        ocn_any_barrier();
        whole(fa, fb);
      }
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
