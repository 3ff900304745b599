// Hand-written CDNA4 (gfx950) MFMA kernels for OCANNL's `+*` contractions:
//     C[batch, m, n] (+)= sum_k A[batch, m, k] * B[batch, n, k]
// i.e. the loop nests `c[..] := fma(a[..], b[..], c[..])` that Assignments.to_low_level emits for
// matmul / einsum and their gradients (arrayjit/lib/assignments.ml:311-488,
// tensor/operation.ml:77-99), which the reference runs as a serial scalar loop.
//
// Layout freedom: each operand is unit-stride either along K or along its row dimension (M for A,
// N for B) with an arbitrary leading stride, plus up to three batch strides -- this covers the
// forward (both K-contiguous), dX (B row-contiguous) and dW (both row-contiguous) forms and the
// attention contractions on [b, s, h, d] tensors without any transposition pass.
//
// Kernel structure (bf16 compute, fp32 accumulate):
//   * 256 threads = 4 wavefronts in a 2x2 grid; block tile BM x BN, K step 64;
//   * global -> registers (16-byte loads) -> LDS, double buffered, one barrier per K step; a
//     K-contiguous operand is held [row][k] (rows padded by 16 bytes: ds_read_b128 of 16 rows hits
//     distinct banks), a row-contiguous operand stays [k][row] as it lies in memory and its MFMA
//     fragments are read with ds_read_b64_tr_b16 -- no transposition anywhere; fp32 sources are
//     rounded to bf16 (RNE) on the way to LDS;
//   * v_mfma_f32_32x32x16_bf16, each wavefront owns a (BM/2) x (BN/2) sub-tile;
//   * workgroup ids are remapped so that each XCD (ids are dealt round-robin over 8 XCDs) works on
//     a compact band of tiles and shares B/A panels through its own L2.
// fp32 operands: gemm_f32.hip.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <type_traits>
#include <utility>

#include "gemm.hpp"
#include "gemm_common.hpp"

namespace ocannl {

// gemm_dtl.hip: the direct-to-LDS instance of that shape (one of those dtl_shape() names).
hipError_t launch_gemm_dtl(int bm, int bn, int bk, int ns, bool akc, bool bkc, const GemmArgs& a, hipStream_t s, hipEvent_t ev);
// gemm_dtl_chain.hip: the same for several operand pairs into one C
hipError_t launch_gemm_dtl_chain(int bm, int bn, int bk, int ns, bool akc, bool bkc, const GemmArgs& a, hipStream_t s, hipEvent_t ev);
// gemm_f32.hip: fp32 operands, 256 x 256 (big) or 128 x 128 tiles.
hipError_t launch_gemm_f32(bool big, bool akc, bool bkc, const GemmArgs& a, hipStream_t s, hipEvent_t ev);

namespace {


// One wavefront per SIMD for the 256x256 tile (the 256 accumulator registers live in AGPRs and the
// whole 512-register budget is available); two for the 128x128 tile.
// PF = 2: global loads run two K stages ahead in two register sets, for launches of at most one
// workgroup per CU, where nothing else hides the HBM latency of a stage; that needs the whole
// register file, so one wavefront per SIMD.
// CHAIN: the launch accumulates several operand pairs into one C (`c =+ a_p * b_p`, p < npairs):
// the K pipeline runs once per pair and the accumulators stay in registers in between.  Only the
// 128x128 tile with two register sets is built that way (the loop around the pipeline costs
// registers that the other variants do not have).
template <int BM, int BN, typename AT, typename BT, bool A_KC, bool B_KC, int PF, bool CHAIN = false>
__global__ void __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu((BM < 256 && sizeof(AT) == 2 && sizeof(BT) == 2 && PF == 1) ? 2 : 1,
                                   (BM >= 256 || PF > 1) ? 1 : 2)))
gemm_bf16_kernel(const GemmArgs g) {
  constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 32, TN = WN / 32;
  constexpr int kAT = lds_tile_elems<BM, A_KC>(), kBT = lds_tile_elems<BN, B_KC>();   // one stage of each operand
  constexpr int kAS = Stager<BM, AT, A_KC>::kLineStride, kBS = Stager<BN, BT, B_KC>::kLineStride;
  extern __shared__ __align__(16) unsigned short smem[];
  unsigned short* const As0 = smem;
  unsigned short* const Bs0 = smem + 2 * kAT;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm0 = (wave >> 1) * WM, wn0 = (wave & 1) * WN;
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
  const AT* A = static_cast<const AT*>(abase) + ao;
  const BT* B = static_cast<const BT*>(bbase) + bo;
  const long lda = A_KC ? g.a_row : g.a_k, ldb = B_KC ? g.b_row : g.b_k;

  // per-lane offsets of the MFMA fragments inside a stage of each operand
  const unsigned a_frag = A_KC ? (unsigned)((wm0 + (lane & 31)) * kAS + (lane >> 5) * 8) : (unsigned)wm0 + tr_lane_offset(lane, kAS);
  const unsigned b_frag = B_KC ? (unsigned)((wn0 + (lane & 31)) * kBS + (lane >> 5) * 8) : (unsigned)wn0 + tr_lane_offset(lane, kBS);
  // fragment of 32-row block `blk`, 16-k sub-step `kk`, from the stage starting at `stage`
  auto a_fragment = [&](const unsigned short* stage, int blk, int kk) OCN_LAMBDA_INLINE -> bf16x8 {
    if constexpr (A_KC) return *reinterpret_cast<const bf16x8*>(stage + a_frag + blk * 32 * kAS + kk * 16);
    else return tr_fragment(stage + a_frag + kk * 16 * kAS + blk * 32, kAS);
  };
  auto b_fragment = [&](const unsigned short* stage, int blk, int kk) OCN_LAMBDA_INLINE -> bf16x8 {
    if constexpr (B_KC) return *reinterpret_cast<const bf16x8*>(stage + b_frag + blk * 32 * kBS + kk * 16);
    else return tr_fragment(stage + b_frag + kk * 16 * kBS + blk * 32, kBS);
  };

  f32x16 acc[TM][TN];
  static_for<TM>([&](auto ic) OCN_LAMBDA_INLINE {
    static_for<TN>([&](auto jc) OCN_LAMBDA_INLINE {
      static_for<16>([&](auto ec) OCN_LAMBDA_INLINE { acc[decltype(ic)::value][decltype(jc)::value][decltype(ec)::value] = 0.0f; });
    });
  });

  // split-K: blockIdx.y owns a contiguous range of K steps
  const long all_steps = (g.K + kBK - 1) / kBK;
  const long per_split = (all_steps + g.splits - 1) / g.splits;
  const long kbeg = (long)blockIdx.y * per_split * kBK;
  const long kend = (kbeg + per_split * kBK) < g.K ? (kbeg + per_split * kBK) : g.K;
  const long ksteps = kend > kbeg ? (kend - kbeg + kBK - 1) / kBK : 0;

  // Software pipeline.  LDS is double buffered; global loads run kPF tiles ahead of the tile being
  // multiplied, held in kPF register sets (one or two).
  constexpr int kPF = PF;
  static_assert(PF == 1 || (PF == 2 && sizeof(AT) == 2 && sizeof(BT) == 2), "two register sets: bf16 sources only");
  Stager<BM, AT, A_KC> sa[kPF];
  Stager<BN, BT, B_KC> sb[kPF];
  static_assert(!CHAIN || (BM == 128 && PF == 2), "chains: 128x128 tiles with two register sets");
  // (the pipeline is a lambda so that the variants without chains hold no loop statement around it:
  // a loop with one trip still cost the 256x256 variants registers)
  auto pipeline = [&]() __attribute__((always_inline)) {
  sa[0].load(A, lda, m0, kbeg, g.M, kend, tid);
  sb[0].load(B, ldb, n0, kbeg, g.N, kend, tid);
  if (kPF > 1) {
    sa[kPF - 1].load(A, lda, m0, kbeg + kBK, g.M, kend, tid);
    sb[kPF - 1].load(B, ldb, n0, kbeg + kBK, g.N, kend, tid);
  }
  sa[0].store(As0, tid);
  sb[0].store(Bs0, tid);
  __syncthreads();

  // one K step; `par` = ks % kPF is a compile-time constant so that the register sets are
  // addressed statically
  auto step = [&](long ks, auto par_c) __attribute__((always_inline)) {
    constexpr int par = decltype(par_c)::value;
    const int cur = ks & 1;
    // register set `par` held tile ks (already in LDS): refill it with tile ks + kPF
    if (ks + kPF < ksteps) {
      sa[par].load(A, lda, m0, kbeg + (ks + kPF) * kBK, g.M, kend, tid);
      sb[par].load(B, ldb, n0, kbeg + (ks + kPF) * kBK, g.N, kend, tid);
    }
    __builtin_amdgcn_sched_barrier(0);   // the loads are issued before the MFMA block, not sunk below it
    const unsigned short* as = As0 + cur * kAT;
    const unsigned short* bs = Bs0 + cur * kBT;
    // fragments are double buffered: the LDS reads of sub-step kk + 1 are issued before the MFMAs
    // of sub-step kk, so that a lone wave per SIMD does not sit out the LDS latency every time
    bf16x8 af[2][TM], bf[2][TN];
    auto read_frags = [&](auto kkc) OCN_LAMBDA_INLINE {
      constexpr int kk = decltype(kkc)::value, fb = kk & 1;
      static_for<TM>([&](auto ic) OCN_LAMBDA_INLINE {
        constexpr int i = decltype(ic)::value;
        af[fb][i] = a_fragment(as, i, kk);
      });
      static_for<TN>([&](auto jc) OCN_LAMBDA_INLINE {
        constexpr int j = decltype(jc)::value;
        bf[fb][j] = b_fragment(bs, j, kk);
      });
    };
    read_frags(std::integral_constant<int, 0>{});
    static_for<kBK / 16>([&](auto kkc) OCN_LAMBDA_INLINE {
      constexpr int kk = decltype(kkc)::value, fb = kk & 1;
      if constexpr (kk + 1 < kBK / 16) {
        read_frags(std::integral_constant<int, kk + 1>{});
        __builtin_amdgcn_sched_barrier(0);
      }
      static_for<TM>([&](auto ic) OCN_LAMBDA_INLINE {
        static_for<TN>([&](auto jc) OCN_LAMBDA_INLINE {
          constexpr int i = decltype(ic)::value, j = decltype(jc)::value;
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[fb][i], bf[fb][j], acc[i][j], 0, 0, 0);
        });
      });
    });
    __builtin_amdgcn_sched_barrier(0);
    // tile ks + 1 sits in the other register set (or, with one set, in the one just refilled)
    if (ks + 1 < ksteps) {
      constexpr int nxt = (par + 1) % kPF;
      sa[nxt].store(As0 + (cur ^ 1) * kAT, tid);
      sb[nxt].store(Bs0 + (cur ^ 1) * kBT, tid);
    }
    __syncthreads();
  };
  // Interleaved K step for full tiles: one basic block in which the other instructions are placed
  // between the MFMAs by hand (and pinned there), so that they issue while the matrix pipe is busy
  // -- with one wave per SIMD nothing else would hide them.  Global loads of tile ks + 1 go with
  // the first half of the MFMAs, its LDS writes with the second half, the LDS reads of the next
  // sub-step's fragments with the current sub-step.
  auto fast_step = [&](long ks, auto loads_c, auto stores_c, auto par_c) __attribute__((always_inline)) {
    constexpr bool kLoads = decltype(loads_c)::value, kStores = decltype(stores_c)::value;
    constexpr int kLoadSet = decltype(par_c)::value, kStoreSet = (kLoadSet + 1) % kPF;   // tile ks + kPF in, tile ks + 1 out
    constexpr int kSub = kBK / 16, kPer = TM * TN, kAll = kSub * kPer, kHalf = kAll / 2;
    constexpr int kA = Stager<BM, AT, A_KC>::kOps, kL = kA + Stager<BN, BT, B_KC>::kOps, kR = TM + TN;
    const int cur = ks & 1;
    const long kn = kbeg + (ks + kPF) * kBK;
    const AT* const a_next = A_KC ? A + m0 * lda + kn : A + kn * lda + m0;
    const BT* const b_next = B_KC ? B + n0 * ldb + kn : B + kn * ldb + n0;
    unsigned short* const an = As0 + (cur ^ 1) * kAT;
    unsigned short* const bn = Bs0 + (cur ^ 1) * kBT;
    const unsigned short* as = As0 + cur * kAT;
    const unsigned short* bs = Bs0 + cur * kBT;
    bf16x8 af[2][TM], bf[2][TN];
    auto read_frag = [&](auto kkc, auto rc) OCN_LAMBDA_INLINE {
      constexpr int kk = decltype(kkc)::value, r = decltype(rc)::value, fb = kk & 1;
      if constexpr (r < TM) af[fb][r] = a_fragment(as, r, kk);
      else bf[fb][r - TM] = b_fragment(bs, r - TM, kk);
    };
    static_for<kR>([&](auto rc) OCN_LAMBDA_INLINE { read_frag(std::integral_constant<int, 0>{}, rc); });
    __builtin_amdgcn_sched_barrier(0);
    static_for<kAll>([&](auto mc) OCN_LAMBDA_INLINE {
      constexpr int m = decltype(mc)::value, kk = m / kPer, idx = m % kPer, i = idx / TN, j = idx % TN, fb = kk & 1;
      if constexpr (kk + 1 < kSub) {
        static_for<(idx + 1) * kR / kPer - idx * kR / kPer>([&](auto rc) OCN_LAMBDA_INLINE {
          read_frag(std::integral_constant<int, kk + 1>{}, std::integral_constant<int, idx * kR / kPer + decltype(rc)::value>{});
        });
      }
      if constexpr (kLoads && m < kHalf) {
        static_for<(m + 1) * kL / kHalf - m * kL / kHalf>([&](auto oc) OCN_LAMBDA_INLINE {
          constexpr int o = m * kL / kHalf + decltype(oc)::value;
          if constexpr (o < kA) sa[kLoadSet].template load_op<o>(a_next, lda);
          else sb[kLoadSet].template load_op<o - kA>(b_next, ldb);
        });
      }
      if constexpr (kStores && m >= kHalf) {
        static_for<(m - kHalf + 1) * kL / kHalf - (m - kHalf) * kL / kHalf>([&](auto oc) OCN_LAMBDA_INLINE {
          constexpr int o = (m - kHalf) * kL / kHalf + decltype(oc)::value;
          if constexpr (o < kA) sa[kStoreSet].template store_op<o>(an);
          else sb[kStoreSet].template store_op<o - kA>(bn);
        });
      }
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[fb][i], bf[fb][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    });
    __syncthreads();
  };

  static_for<kPF>([&](auto p) OCN_LAMBDA_INLINE { sa[decltype(p)::value].init_ops(lda, tid); sb[decltype(p)::value].init_ops(ldb, tid); });
  // (fp32 sources stage twice the registers: with double-buffered fragments on top the loop
  // spills, so they keep the plain loop)
  constexpr bool kInterleave = sizeof(AT) == 2 && sizeof(BT) == 2 && kPF <= 2;
  const bool full_tile = kInterleave && m0 + BM <= g.M && n0 + BN <= g.N && ksteps > 0 && kbeg + ksteps * kBK <= kend;
  if constexpr (kInterleave) {
    if (full_tile) {
      using Y = std::true_type; using N = std::false_type;
      using P0 = std::integral_constant<int, 0>; using P1 = std::integral_constant<int, 1 % kPF>;
      if constexpr (kPF == 1) {
        for (long ks = 0; ks + 1 < ksteps; ++ks) fast_step(ks, Y{}, Y{}, P0{});
        fast_step(ksteps - 1, N{}, N{}, P0{});
      } else {
        // two register sets: steps come in pairs so that the set numbers are compile-time constants
        long ks = 0;
        for (; ks + 3 < ksteps; ks += 2) { fast_step(ks, Y{}, Y{}, P0{}); fast_step(ks + 1, Y{}, Y{}, P1{}); }
        const long rem = ksteps - ks;   // 1, 2 or 3 steps left; ks is even
        if (rem == 3) { fast_step(ks, Y{}, Y{}, P0{}); fast_step(ks + 1, N{}, Y{}, P1{}); fast_step(ks + 2, N{}, N{}, P0{}); }
        else if (rem == 2) { fast_step(ks, N{}, Y{}, P0{}); fast_step(ks + 1, N{}, N{}, P1{}); }
        else fast_step(ks, N{}, N{}, P0{});
      }
    }
  }
  if (!full_tile) {
    long ks = 0;
    for (; ks + kPF <= ksteps; ks += kPF) static_for<kPF>([&](auto p) OCN_LAMBDA_INLINE { step(ks + decltype(p)::value, p); });
    static_for<kPF>([&](auto p) OCN_LAMBDA_INLINE { if (ks + decltype(p)::value < ksteps) step(ks + decltype(p)::value, p); });
  }
  };   // pipeline
  if constexpr (CHAIN) {
    for (int pair = 0; pair < g.npairs; ++pair) {
      if (pair > 0) {
        A = static_cast<const AT*>(pair == 1 ? g.a_more[0] : pair == 2 ? g.a_more[1] : g.a_more[2]) + ao;
        B = static_cast<const BT*>(pair == 1 ? g.b_more[0] : pair == 2 ? g.b_more[1] : g.b_more[2]) + bo;
      }
      pipeline();
    }
  } else {
    pipeline();
  }

  // (every wave has passed the last barrier of the main loop: the operand stages are free)
  epilogue<TM, TN>(g, cbase, c2base, acc, m0 + wm0, n0 + wn0, co, lane,
                   reinterpret_cast<float*>(smem) + wave * ((kAT + kBT) / 4));
}

template <int BM, int BN, bool A_KC, bool B_KC>
constexpr size_t bf16_smem() { return 2ull * (lds_tile_elems<BM, A_KC>() + lds_tile_elems<BN, B_KC>()) * sizeof(unsigned short); }

// Tile grids of one launch along z: batch entries times grouped contractions.
long batch_count(const GemmDesc& d) {
  long nb = 1 + (long)d.group.size();
  for (int i = 0; i < d.nbatch; ++i) nb *= d.batch_ext[i];
  return nb;
}


// Tile size and split-K factor, from a measured sweep on MI355X (bf16 operands).  256x256 tiles
// (one workgroup per CU) win only when the output alone gives >= 256 of them and K runs at least
// 8 stages (below that a launch is all prologue and epilogue); anything else
// runs 128x128 tiles, two workgroups per CU, and when those are fewer than 256 K is split
// towards ~512 workgroups (~256 for bf16 sources), never below 8 K stages per split.  Splits are summed in index order by
// splitk_reduce_kernel (deterministic).
struct TileConfig { bool big; int splits; int prefetch; bool narrow = false; };

TileConfig tile_config(const GemmDesc& d) {
  const long nb = batch_count(d);
  const long t256 = ((d.M + 255) / 256) * ((d.N + 255) / 256) * nb;
  const long t128 = ((d.M + 127) / 128) * ((d.N + 127) / 128) * nb;
  TileConfig c;
  const bool bf16_sources = d.a.prec == Prec::Bfloat16 && d.b.prec == Prec::Bfloat16;
  if (d.more.empty() && t256 >= 256 && d.M > 128 && d.N > 128 && d.K >= 512) { c.big = true; c.splits = 1; }
  else {
    c.big = false;
    long s = 1;
    // bf16 sources: towards one workgroup per CU, which then loads two stages ahead (below);
    // otherwise towards two per CU
    const long target = bf16_sources ? 256 : 512;
    if (t128 < 256 && d.epi_bias < 0 && d.epi_relu < 0) {   // (folded consumers are applied by the contraction's own epilogue)
      while (s * 2 * t128 <= target && s * 2 <= d.K / 512 && s < 64) s *= 2;
    }
    c.splits = (int)s;
  }
  // two stages of global loads in flight when the launch puts at most one workgroup on a CU and
  // each runs at least 8 K stages (measured: 8192x512x2048 bf16 595 -> 738 TFLOP/s)
  c.prefetch = (!c.big && bf16_sources && t128 * c.splits <= 256 && d.K / c.splits >= 512) ? 2 : 1;
  if (!d.more.empty()) c.prefetch = 2;   // the only variant built for chains
  // results of at most 64 columns (the attention products against V, K, Q: N = head size) take a
  // 128 x 64 tile: with 128 columns half of every tile would be masked and the launch would run the
  // checked loop for ragged tiles
  c.narrow = !c.big && bf16_sources && d.more.empty() && d.N <= 64 && d.N > 16;
  return c;
}
bool narrow_tile(const GemmDesc& d) { return tile_config(d).narrow; }

bool big_tile(const GemmDesc& d) { return tile_config(d).big; }
int split_count(const GemmDesc& d) { return tile_config(d).splits; }
int prefetch_depth(const GemmDesc& d) { return tile_config(d).prefetch; }

template <int BM, int BN, typename AT, typename BT, int PF = 1, bool CHAIN = false>
hipError_t launch_bf16_layout(bool akc, bool bkc, const GemmArgs& a, hipStream_t s, hipEvent_t ev) {
  if (akc && bkc) return launch(gemm_bf16_kernel<BM, BN, AT, BT, true, true, PF, CHAIN>, bf16_smem<BM, BN, true, true>(), BM, BN, a, s, ev);
  if (akc && !bkc) return launch(gemm_bf16_kernel<BM, BN, AT, BT, true, false, PF, CHAIN>, bf16_smem<BM, BN, true, false>(), BM, BN, a, s, ev);
  if (!akc && bkc) return launch(gemm_bf16_kernel<BM, BN, AT, BT, false, true, PF, CHAIN>, bf16_smem<BM, BN, false, true>(), BM, BN, a, s, ev);
  return launch(gemm_bf16_kernel<BM, BN, AT, BT, false, false, PF, CHAIN>, bf16_smem<BM, BN, false, false>(), BM, BN, a, s, ev);
}

bool a_kcontig(const GemmDesc& d) { return d.a.s_k == 1 || d.K == 1; }
bool b_kcontig(const GemmDesc& d) { return d.b.s_k == 1 || d.K == 1; }

// ---- the direct-to-LDS kernel (gemm_dtl.hpp) -----------------------------------------------------
// Shape of the instance for a contraction, or bm = 0 when the register-staged kernels take it: bf16
// operands, full tiles, every K split a whole number of at least NS - 1 steps.  256 x 256 tiles run
// four stages of 32 k (128 KB of LDS); 128 x 128 tiles five stages of 64 k when the launch puts at
// most one workgroup on a compute unit -- what such a launch lacks is loads in flight -- and four
// stages of 32 k (64 KB: two workgroups per compute unit) otherwise; 128 x 64 tiles (results of at
// most 64 columns: short-K batched products of attention) four stages of 32 k (48 KB: three
// workgroups per compute unit, measured 2 % of a transformer step against five stages of 64 k).
struct DtlShape { int bm = 0, bn = 0, bk = 0, ns = 0; };

// Chains (one pair's K after the other's) from this many workgroups on, the fewest measured; fewer run on contract_direct.hip
// or the register-staged loop.  Three products, register-staged -> direct to LDS, both k-contiguous (row-contiguous): 1024 x
// 512 x 512 (32 workgroups) 19.1 -> 14.0 (19.8 -> 15.6) us, 4096 x 512 x 512 20.0 -> 14.8 (20.8 -> 16.4), 8192 x 512 x 512 24.1
// -> 18.2 (24.6 -> 19.3), 8192 x 1024 x 1024 73 -> 62 (75 -> 51).
constexpr long kChainWorkgroups = 32;

DtlShape dtl_shape(const GemmDesc& d) {
  DtlShape none, s;
  if (d.a.prec != Prec::Bfloat16 || d.b.prec != Prec::Bfloat16) return none;
  const TileConfig c = tile_config(d);
  const long pairs = 1 + (long)d.more.size();
  if (c.big) s = {256, 256, 32, 4};
  else if (c.narrow) s = {128, 64, 32, 4};
  else {
    const long t128 = ((d.M + 127) / 128) * ((d.N + 127) / 128) * batch_count(d);
    if (pairs > 1 && t128 * c.splits < kChainWorkgroups) return none;
    if (t128 * c.splits <= 256) s = {128, 128, 64, 5};
    else s = {128, 128, 32, 4};
    // K = 64, batched products of attention above all: two steps, three stages (48 KB), for at most 1024 tiles, two rounds of
    // two a unit.  Register-staged -> so, four layouts, fp32 and bf16 results: batches of 256 x 256, 256 of them 21 -> 20.5 and
    // 19.8 -> 19.1 us, but 1024 of them 67 -> 70 and 57 -> 60; 128 x 1024, 256 of them (2048 tiles) 40 -> 42 and 31 -> 33; 2048 x
    // 2048 10.4 -> 10.0 and 8.9 -> 8.6.  Fewer tiles: gemm_prefers_any.
    if (t128 >= 256 && t128 <= 1024 && pairs == 1 && d.K == 64) s = {128, 128, 32, 3};
  }
  if (d.M % s.bm || d.N % s.bn || d.K % s.bk) return none;
  const long steps = d.K / s.bk;
  if (steps % c.splits || steps / c.splits * pairs < s.ns - 1) return none;
  return s;
}

// Operand addresses and strides as the direct loads need them: 16-byte aligned bases and lines, lane
// offsets within 32 bits.
bool dtl_operands_ok(const GemmArgs& a, bool akc, bool bkc) {
  auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  const int64_t lda = akc ? a.a_row : a.a_k, ldb = bkc ? a.b_row : a.b_k;
  if (!aligned(a.a) || !aligned(a.b) || lda % 8 || ldb % 8 || lda <= 0 || ldb <= 0 || lda >= (1 << 24) || ldb >= (1 << 24)) return false;
  if ((akc ? a.a_k : a.a_row) != 1 || (bkc ? a.b_k : a.b_row) != 1) return false;
  for (int i = 0; i < a.nbatch; ++i) if (a.a_batch[i] % 8 || a.b_batch[i] % 8) return false;
  for (int g = 1; g < a.ngroups || g < a.npairs; ++g) if (!aligned(a.a_more[g - 1]) || !aligned(a.b_more[g - 1])) return false;
  return true;
}

}  // namespace

void as_any_shape(GemmDesc& g) {
  auto digits = [](GemmOperand& o) { o.row_stride[2] = o.s_row; o.k_stride[2] = o.s_k; };
  digits(g.a); digits(g.b); digits(g.c);
  for (auto& m : g.group) { digits(m.a); digits(m.b); digits(m.c); }
  for (auto& p : g.more) { digits(p.first); digits(p.second); }
  g.m_ext[2] = g.M; g.n_ext[2] = g.N; g.k_ext[2] = g.K;
  g.any = true;
}

// Fewer 128 x 128 tiles than compute units: the register-staged kernels leave some idle and hide no latency on the
// rest, where 64 x 64 tiles of contract_any.hip put several workgroups on each; but they split K further, and the
// smaller tile reads twice the operands per product.  Compared is what a compute unit goes through, area of C by k, a
// stage of the smaller tile costing more by what was measured for it: 12 and 25 % in fp32 with one and both operands
// row-contiguous (fragments of four reads), 8 % in bf16 with both, and 15 % where no unit holds a second workgroup.  On
// the other side stand the register-staged kernel's longer start and the launch that sums its splits: 2.5 M, 13 us in
// fp32, 4 in bf16.  Measured over 9 shapes of C of 16 to 192 tiles, K of 256 to 16384 and the operand layouts, one
// product, register-staged against small tile: 1000 x 1000, both row-contiguous: K = 1024 fp32 50 against 33 us, bf16
// 18 against 12; 2048 fp32 52 against 59, bf16 21 against 20; 8192 fp32 157 against 225, bf16 44 against 66.  From 256
// tiles on the larger tile wins (8000 x 1000 x 1000 bf16, both gradients too: 122 against 173 us).
// A workspace that would take the routine beyond the static scratch array, where the small tile's does not, is no choice.
// Few enough tiles for contract_direct.hip: that, whatever the layout (512 x 512 x 1024 in fp32 12 us, 30 on 64 x 64 tiles),
// and chains too (three products of 594 x 320 x 320, 15 tiles of 128 x 128: 24.9 -> 11.0 us).
bool gemm_prefers_any(const GemmDesc& d, uint64_t room) {
  if (d.any || d.a.prec != d.b.prec || !contract_any_fits(d)) return false;
  GemmDesc few = d;
  as_any_shape(few);
  if (!d.more.empty()) return contract_any_direct(few);
  const int64_t t128 = (int64_t)((d.M + 127) / 128) * ((d.N + 127) / 128) * batch_count(d);
  if (t128 >= 256) return false;
  const bool f32 = d.a.prec == Prec::Single;
  if (!f32 && dtl_shape(d).bm != 0) return false;
  if (contract_any_direct(few)) return true;   // (its splits: contract_any_settle)
  if (gemm_workspace_bytes(d) > room) {
    contract_any_settle(few, room);
    if (contract_any_workspace_bytes(few) <= room) return true;
  }
  const TileConfig c = tile_config(d);
  const int64_t staged = (t128 * c.splits + 255) / 256 * 128 * (c.narrow ? 64 : 128) / c.splits;
  bool alone;
  const int64_t small = contract_any_area(d, alone);
  const int lines = !a_kcontig(d) + !b_kcontig(d);
  const int extra = (alone ? 15 : 0) + (f32 ? (lines == 2 ? 25 : 12 * lines) : lines == 2 ? 8 : 0);
  return (double)small * (100 + extra) / 100 * d.K <= (double)staged * d.K + 2.5e6;
}

const char* gemm_kernel_name(const GemmDesc& d) {
  if (d.any) return contract_any_name(d);
  // the instantiation as a profiler prints it (without namespaces)
  static thread_local char buf[128];
  const bool af = d.a.prec == Prec::Single, bf = d.b.prec == Prec::Single;
  const int tile = big_tile(d) ? 256 : 128, tile_n = narrow_tile(d) ? 64 : tile;
  const char* tf[2] = {"false", "true"};
  const DtlShape ds = dtl_shape(d);
  if (af && bf)
    snprintf(buf, sizeof buf, "gemm_f32_kernel<%d, %d, 2, 2, %s, %s>", tile, tile, tf[a_kcontig(d)], tf[b_kcontig(d)]);
  else if (ds.bm)   // (operands that turn out misaligned at launch take the register-staged kernel instead)
    snprintf(buf, sizeof buf, "gemm_bf16_dtl_kernel<%d, %d, %d, %d, %s, %s, %s, %s>", ds.bm, ds.bn, ds.bk, ds.ns, tf[a_kcontig(d)], tf[b_kcontig(d)],
             tf[dtl_odd(ds.bk, ds.ns, d.K, split_count(d), 1 + (int)d.more.size())], tf[!d.more.empty()]);
  else
    snprintf(buf, sizeof buf, "gemm_bf16_kernel<%d, %d, %s, %s, %s, %s, %d, %s>", tile, tile_n, af ? "float" : "unsigned short",
             bf ? "float" : "unsigned short", tf[a_kcontig(d)], tf[b_kcontig(d)], prefetch_depth(d), tf[!d.more.empty()]);
  return buf;
}

size_t gemm_workspace_bytes(const GemmDesc& d) {
  if (d.any) return contract_any_workspace_bytes(d);
  const int sp = split_count(d);
  return sp > 1 ? (size_t)sp * (size_t)batch_count(d) * (size_t)d.M * (size_t)d.N * sizeof(float) : 0;
}

hipError_t launch_gemm(const GemmDesc& d, const GemmArgs& a_in, void* workspace, hipStream_t s, hipEvent_t ev) {
  if (d.any) return launch_contract_any(d, a_in, workspace, s, ev);
  GemmArgs a = a_in;
  a.splits = split_count(d);
  a.ws = static_cast<float*>(workspace);
  const bool akc = a_kcontig(d), bkc = b_kcontig(d);
  const bool big = big_tile(d);
  {
    // XCD partition: every A panel is read by each of the xcd_n rectangle columns, every B panel
    // by each of the xcd_m rows
    const long tile = big ? 256 : 128, tile_n = narrow_tile(d) ? 64 : tile;
    const long tiles_m = (d.M + tile - 1) / tile, tiles_n = (d.N + tile_n - 1) / tile_n;
    const double a_bytes = (double)d.M * prec_in_bytes(d.a.prec), b_bytes = (double)d.N * prec_in_bytes(d.b.prec);
    // a grouped launch of 2 or 4 unbatched members without a K split: each member on 4 or 2 XCDs of
    // its own, so that its panels are fetched into that many L2 caches instead of all eight
    const int members = 1 + (int)d.group.size();
    int nx = 8;
    a.member_xcds = 0;
    if ((members == 2 || members == 4) && d.nbatch == 0 && a.splits == 1 && (tiles_m * tiles_n) % (8 / members) == 0) {
      nx = 8 / members;
      a.member_xcds = nx;
    }
    a.xcd_m = 0;
    double best = 0;
    for (int xm = 1; xm <= nx; xm *= 2) {
      const int xn = nx / xm;
      if (tiles_m % xm || tiles_n % xn) continue;
      const double cost = a_bytes * xn + b_bytes * xm;
      if (a.xcd_m == 0 || cost < best) { a.xcd_m = xm; best = cost; }
    }
  }
  const bool af = d.a.prec == Prec::Single, bf = d.b.prec == Prec::Single;
  if (af && bf) return launch_gemm_f32(big, akc, bkc, a, s, ev);
  if (a.npairs > 1 && (af || bf)) return hipErrorInvalidValue;   // chains: bf16 operands only
  if (!af && !bf) {
    const DtlShape ds = dtl_shape(d);
    if (ds.bm && dtl_operands_ok(a, akc, bkc)) {
      return (a.npairs > 1 ? launch_gemm_dtl_chain : launch_gemm_dtl)(ds.bm, ds.bn, ds.bk, ds.ns, akc, bkc, a, s, ev);
    }
    if (a.npairs > 1) return launch_bf16_layout<128, 128, unsigned short, unsigned short, 2, true>(akc, bkc, a, s, ev);
    if (big) return launch_bf16_layout<256, 256, unsigned short, unsigned short>(akc, bkc, a, s, ev);
    if (narrow_tile(d))
      return prefetch_depth(d) == 2 ? launch_bf16_layout<128, 64, unsigned short, unsigned short, 2>(akc, bkc, a, s, ev)
                                    : launch_bf16_layout<128, 64, unsigned short, unsigned short>(akc, bkc, a, s, ev);
    return prefetch_depth(d) == 2 ? launch_bf16_layout<128, 128, unsigned short, unsigned short, 2>(akc, bkc, a, s, ev)
                                  : launch_bf16_layout<128, 128, unsigned short, unsigned short>(akc, bkc, a, s, ev);
  }
  if (af && !bf)
    return big ? launch_bf16_layout<256, 256, float, unsigned short>(akc, bkc, a, s, ev)
               : launch_bf16_layout<128, 128, float, unsigned short>(akc, bkc, a, s, ev);
  return big ? launch_bf16_layout<256, 256, unsigned short, float>(akc, bkc, a, s, ev)
             : launch_bf16_layout<128, 128, unsigned short, float>(akc, bkc, a, s, ev);
}

}  // namespace ocannl
