// Contractions of any extents and strides: instances for bf16 operands, choice of the tile, launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include "contract_any.hpp"

namespace ocannl {
namespace {

// Sums the K splits in index order and applies them to C.
__global__ void __launch_bounds__(256) contract_any_reduce_kernel(const OcnAnyDesc d, const AnyBatch q, const AnyPtrs p) {
  const long cells = (long)d.M * d.N, i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= cells) return;
  const int z = blockIdx.y;
  const void *a, *b;
  void *c, *c2;
  any_operands(d, q, p, z, a, b, c, c2);
  const float* ws = p.ws + (long)z * d.splits * cells + i;
  float v = 0.0f;
#pragma unroll 16
  for (int s = 0; s < d.splits; ++s) v += ws[s * cells];
  const int m = (int)(i / d.N), n = (int)(i - (long)m * d.N);
  const long at = (long)ocn_digit_off(ocn_digits(d.dm, m), d.c_m) + ocn_digit_off(ocn_digits(d.dn, n), d.c_n);
  if (d.c_bf16) {
    unsigned short* const o = static_cast<unsigned short*>(c) + at;
    if (d.accumulate) v += __uint_as_float((unsigned)*o << 16);
    *o = __builtin_bit_cast(unsigned short, (__bf16)v);
  } else {
    float* const o = static_cast<float*>(c) + at;
    if (d.accumulate) v += *o;
    *o = v;
    if (c2) static_cast<unsigned short*>(c2)[at] = __builtin_bit_cast(unsigned short, (__bf16)v);
  }
}

OcnDigits digits_of(const int64_t (&ext)[3], int n) {
  OcnDigits r{};
  r.n = n;
  r.e1 = (int)ext[1]; r.e2 = (int)ext[2];
  digit_magic(ext[1], r.mul1, r.sh1);
  digit_magic(ext[2], r.mul2, r.sh2);
  return r;
}

bool any_is_f32(const GemmDesc& d) { return d.a.prec != Prec::Bfloat16 || d.b.prec != Prec::Bfloat16; }
bool any_mixed(const GemmDesc& d) { return d.a.prec != d.b.prec; }
// k-contiguous (or contiguous along nothing), else row-contiguous
bool any_kc(const GemmOperand& o) { return o.k_stride[2] == 1 || o.row_stride[2] != 1; }

// Whole chunks of memory along k or along the rows, as DirectOperand takes them.
bool any_regular(const GemmDesc& d) {
  auto operand = [&](const GemmOperand& o, int64_t rows, const int64_t (&ext)[3], int digits) {
    if (any_kc(o)) return o.k_stride[2] == 1 && (d.k_digits == 1 || d.k_ext[2] % (o.prec == Prec::Bfloat16 ? 8 : 4) == 0);
    return o.row_stride[2] == 1 && rows >= 2 && (digits == 1 || ext[2] % 2 == 0);
  };
  return operand(d.a, d.M, d.m_ext, d.m_digits) && operand(d.b, d.N, d.n_ext, d.n_digits);
}

long any_entries(const GemmDesc& d) {
  long nb = 1 + (long)d.group.size();
  for (int i = 0; i < d.nbatch; ++i) nb *= d.batch_ext[i];
  return nb;
}

// Do 32 x 32 tiles whose wavefronts share K and read their operands straight from memory (contract_direct.hip) take it, and
// in how many splits?  They read twice the operands per product that 64 x 64 tiles do, so up to one tile a compute unit, and
// long sums only where splits are free for them.  Measured (staged tile -> these, us) over products, batches and groups
// of 16 to 768 tiles, K of 66 to 4096 and all layouts:
//   fp32, up to 256 tiles: K = 128 7.2 -> 6.1 to 6.8, 512 14 -> 9 to 10, 1024 18 -> 13 to 15, 2048 20 -> 19 with a row-contiguous
//     operand, but 19 -> 22 without one (1800: 18 to 21 -> 19), and 3072 24 -> 25 to 29; in splits, 128 tiles, 2 x 1024 19
//     -> 17, 2 x 1500 23 -> 18, but 2 x 1536, where the staged tile has eight, 18 -> 20; 64 tiles, 4 x 1024 20 -> 17.
//   257 to 512 tiles, a row-contiguous operand: K = 512 16 -> 13, 1024 20 -> 18, 1500 25 -> 23, 2048 26 -> 29; with one operand
//     k-contiguous 81 6.6 -> 6.1, 128 7.5 -> 7.9, 131 8.6 -> 8.0, 200 10.3 -> 8.6.
//   bf16, up to 256 tiles, a row-contiguous operand: K = 128 5.5 -> 5.3, 1024 10 -> 7 to 8, 2560 16 -> 13, 3056 18 -> 13, but
//     3072, where the staged tile has four splits, 14 -> 15; in two, 128 tiles, 13.2 -> 13.0 there and 14.5 -> 14.3 at 4096.  k-contiguous operands touch 32 rows with every
//     load: K = 160 5.6 -> 5.1, 320 5.4 -> 5.7; rows 128 bytes apart or a multiple of that collide, K = 128 5.3 -> 5.5, 256 5.7
//     -> 5.5.  Rows at odd elements, which the vector memory path takes apart, lose at once (K = 1001 9.5 -> 12.9).
//   One or two tiles to an entry of a batch, where a staged tile is mostly padding: at any K (200 x 32 x 32 x 4000 fp32 79 ->
//     44, bf16 34 -> 24).
// A grouped launch goes by all of its tiles, so its members may be summed in another order than apart.  Not so up to 128 tiles
// each and 512 of K: k-contiguous fp32 products keep to these tiles then, at 8.7, 11.5 and 15.6 us for K = 128, 256, 512
// against 7.4, 9.6 and 14.2.
int direct_splits(const GemmDesc& d) {
  const long members = 1 + (long)d.group.size(), tiles = ((d.M + 31) / 32) * ((d.N + 31) / 32) * any_entries(d);
  const bool f32 = any_is_f32(d), both_kc = any_kc(d.a) && any_kc(d.b), one_kc = any_kc(d.a) != any_kc(d.b);
  const int64_t all_k = d.K * (int64_t)(1 + d.more.size());
  if (all_k <= 64 || all_k > 4096 || tiles > (f32 ? 512 : 256) || !any_regular(d)) return 0;
  if (tiles > 256 && (both_kc ? tiles / members > 128 || all_k > 512 : all_k > 1536 || (one_kc && !any_mixed(d) && all_k > 96 && all_k <= 128))) return 0;
  if (!f32 && both_kc && (all_k > 256 || (d.more.empty() && all_k < 256 && (d.a.row_stride[2] % 64 == 0 || d.b.row_stride[2] % 64 == 0)))) return 0;
  auto odd = [&](const GemmOperand& o) {
    int64_t all = o.offset;
    for (auto& t : o.static_terms) all |= t.second;
    for (int i = 0; i < d.nbatch; ++i) all |= o.s_batch[i];
    for (int i = 0; i < 3; ++i) all |= o.row_stride[i];
    return o.prec == Prec::Bfloat16 && any_kc(o) && (all & 1);
  };
  if (odd(d.a) || odd(d.b)) return 0;
  if (!d.more.empty()) return f32 || d.c.prec != Prec::Single ? 0 : 1;
  int splits = 1;
  if (!d.unsplit && d.epi_bias < 0 && d.epi_relu < 0) while (splits * 2 * tiles <= 256 && d.K / (splits * 2) >= (f32 ? 768 : 1536)) splits *= 2;
  const bool padding = std::min(d.M, d.N) <= 32 && std::max(d.M, d.N) <= 64;
  const int64_t most = !f32 ? 3071 : splits > 1 ? 1535 : both_kc && !any_mixed(d) ? 1800 : 2048;
  return padding || d.unsplit || d.K / splits <= most ? splits : 0;
}

// 128 x 128 tiles when they fill the chip twice over, else 64 x 64 (128 x 32 or 32 x 128 when one extent is at most
// 32: half of a square tile would be padding).  K is split towards two workgroups per compute unit when the tiles
// are fewer than one each and a split keeps a dozen K steps: fewer do not give back the launch that sums the splits, 4 to
// 5 us (17 such launches in a bf16 transformer block of odd extents at 128 of K a split: 569 us, 551 without them; 64 rows
// through 4096 x 4096, four splits: 13.6 us).
AnyShape staged_shape(const GemmDesc& d) {
  const long nb = any_entries(d);
  AnyShape s{64, 64, 1, false, false};
  if (any_mixed(d)) {}   // (the one tile built for a bf16 and an fp32 operand)
  else if (d.N <= 32) { s.bm = 128; s.bn = 32; }
  else if (d.M <= 32) { s.bm = 32; s.bn = 128; }
  else if (d.M > 64 && d.N > 64 && ((d.M + 127) / 128) * ((d.N + 127) / 128) * nb >= 512) s.bm = s.bn = 128;
  const long tiles = ((d.M + s.bm - 1) / s.bm) * ((d.N + s.bn - 1) / s.bn) * nb;
  s.parts = any_is_f32(d) && d.K >= (tiles > 256 ? kPartsFrom : kPartsFromAlone);
  if (tiles < 192 && d.epi_bias < 0 && d.epi_relu < 0) while ((long)s.splits * 2 * tiles <= 512 && d.K / (s.splits * 2) >= (any_is_f32(d) ? 384 : 768)) s.splits *= 2;
  return s;
}

AnyShape any_shape(const GemmDesc& d) {
  if (const int splits = direct_splits(d)) return {32, 32, splits, false, true};
  return staged_shape(d);
}

}  // namespace

// Offsets by row and by k are computed apart, each in an int, and added in 64 bits; 2^30 leaves room for a tile and a
// K step past the end.  Batch strides are 64 bits wide and may be anything.
bool contract_any_fits(const GemmDesc& d) {
  constexpr int64_t kLimit = (int64_t)1 << 30;
  auto reach = [&](const int64_t (&ext)[3], const int64_t (&stride)[3], int64_t n, int64_t s) {
    if (!d.any) return (n - 1) * std::abs(s);
    int64_t r = 0;
    for (int i = 0; i < 3; ++i) r += (ext[i] - 1) * std::abs(stride[i]);
    return r;
  };
  if (d.M > kLimit || d.N > kLimit || d.K > kLimit) return false;
  return reach(d.m_ext, d.a.row_stride, d.M, d.a.s_row) <= kLimit && reach(d.k_ext, d.a.k_stride, d.K, d.a.s_k) <= kLimit &&
         reach(d.n_ext, d.b.row_stride, d.N, d.b.s_row) <= kLimit && reach(d.k_ext, d.b.k_stride, d.K, d.b.s_k) <= kLimit &&
         reach(d.m_ext, d.c.row_stride, d.M, d.c.s_row) + reach(d.n_ext, d.c.k_stride, d.N, d.c.s_k) <= kLimit;
}

bool contract_any_direct(const GemmDesc& d) { return direct_splits(d) > 0; }

void contract_any_settle(GemmDesc& d, uint64_t room) {
  if (!d.any || contract_any_workspace_bytes(d) <= room) return;
  d.unsplit = true;
  if (contract_any_workspace_bytes(d) > room) d.unsplit = false;
}

int64_t contract_any_area(const GemmDesc& d, bool& alone) {
  const AnyShape s = staged_shape(d);
  const int64_t groups = (int64_t)((d.M + s.bm - 1) / s.bm) * ((d.N + s.bn - 1) / s.bn) * any_entries(d) * s.splits;
  alone = groups <= 256;
  return (groups + 255) / 256 * s.bm * s.bn / s.splits;
}

const char* contract_any_name(const GemmDesc& d) {
  static thread_local char buf[96];
  const AnyShape s = any_shape(d);
  const char* tf[2] = {"false", "true"};
  const char *ak = tf[any_kc(d.a)], *bk = tf[any_kc(d.b)], *ab = tf[d.a.prec == Prec::Bfloat16], *bb = tf[d.b.prec == Prec::Bfloat16];
  if (s.direct) snprintf(buf, sizeof buf, "gemm_%s_kernel_any_direct<%s, %s, %s, %s, %d, %s>", any_is_f32(d) ? "f32" : "bf16", ak, bk, ab, bb,
                         any_is_f32(d) || !d.more.empty() ? 2 : 3, tf[!d.more.empty()]);
  else if (!any_is_f32(d)) snprintf(buf, sizeof buf, "gemm_bf16_kernel_any<%d, %d, %s, %s>", s.bm, s.bn, ak, bk);
  else snprintf(buf, sizeof buf, "gemm_f32_kernel_any<%d, %d, %s, %s, %s, %s, %s>", s.bm, s.bn, ak, bk, ab, bb, tf[s.parts]);
  return buf;
}

size_t contract_any_workspace_bytes(const GemmDesc& d) {
  const AnyShape s = any_shape(d);
  return s.splits > 1 ? (size_t)s.splits * any_entries(d) * d.M * d.N * sizeof(float) : 0;
}

hipError_t launch_contract_any(const GemmDesc& g, const GemmArgs& in, void* workspace, hipStream_t s, hipEvent_t after_main) {
  const AnyShape sh = any_shape(g);
  OcnAnyDesc d{};
  d.M = (int)g.M; d.N = (int)g.N; d.K = (int)g.K;
  d.dm = digits_of(g.m_ext, g.m_digits); d.dn = digits_of(g.n_ext, g.n_digits); d.dk = digits_of(g.k_ext, g.k_digits);
  auto operand = [](const GemmOperand& o) {
    OcnAnyOperand r{};
    for (int i = 0; i < 3; ++i) { r.row[i] = (int)o.row_stride[i]; r.k[i] = (int)o.k_stride[i]; }
    r.bf16 = o.prec == Prec::Bfloat16;
    return r;
  };
  d.a = operand(g.a); d.b = operand(g.b);
  for (int i = 0; i < 3; ++i) { d.c_m[i] = (int)g.c.row_stride[i]; d.c_n[i] = (int)g.c.k_stride[i]; }
  d.c_bf16 = in.c_is_bf16; d.accumulate = in.accumulate;
  d.splits = sh.splits;
  d.tiles_m = (int)((g.M + sh.bm - 1) / sh.bm); d.tiles_n = (int)((g.N + sh.bn - 1) / sh.bn);
  AnyBatch q{};
  q.nbatch = g.nbatch; q.members = in.ngroups; q.batches = 1;
  for (int i = 0; i < g.nbatch; ++i) {
    q.ext[i] = (int)g.batch_ext[i]; q.batches *= q.ext[i];
    q.a[i] = g.a.s_batch[i]; q.b[i] = g.b.s_batch[i]; q.c[i] = g.c.s_batch[i];
  }
  AnyPtrs p{};
  p.a[0] = in.a; p.b[0] = in.b; p.c[0] = in.c; p.c2[0] = in.c2;
  for (int i = 1; i < in.ngroups; ++i) { p.a[i] = in.a_more[i - 1]; p.b[i] = in.b_more[i - 1]; p.c[i] = in.c_more[i - 1]; p.c2[i] = in.c2_more[i - 1]; }
  p.pairs = in.npairs;
  for (int i = 1; i < in.npairs; ++i) { p.a[i] = in.a_more[i - 1]; p.b[i] = in.b_more[i - 1]; }
  p.ws = static_cast<float*>(workspace);
  p.ep = {static_cast<const unsigned short*>(in.bias), in.relu_out ? static_cast<const char*>(in.relu_out) - static_cast<const char*>(in.c) : 0, in.relu_c};
  const long entries = (long)q.batches * q.members, tiles = (long)d.tiles_m * d.tiles_n * entries;
  if (tiles <= 0 || tiles > 0x3FFFFFFFL || entries > 65535 || in.npairs < 1 || in.npairs > 4 || (in.npairs > 1 && (!sh.direct || in.ngroups > 1)) || (sh.splits > 1 && !p.ws)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((tiles + 7) / 8 * 8), (unsigned)sh.splits, 1);
  const bool akc = any_kc(g.a), bkc = any_kc(g.b), f32 = any_is_f32(g);
  hipError_t e = sh.direct ? launch_direct(akc, bkc, grid, d, &q, &p, s)
                 : f32 ? launch_any_f32(sh.bm, sh.bn, sh.parts, d.a.bf16, d.b.bf16, akc, bkc, grid, d, &q, &p, s)
                 : sh.bn == 32 ? launch_layout<128, 32, true, true, false>(akc, bkc, grid, d, q, p, s)
                 : sh.bm == 32 ? launch_layout<32, 128, true, true, false>(akc, bkc, grid, d, q, p, s)
                 : sh.bm == 128 ? launch_layout<128, 128, true, true, false>(akc, bkc, grid, d, q, p, s)
                                : launch_layout<64, 64, true, true, false>(akc, bkc, grid, d, q, p, s);
  if (e == hipSuccess && after_main) e = hipEventRecord(after_main, s);
  if (e != hipSuccess || sh.splits == 1) return e;
  const long cells = (long)d.M * d.N;
  hipLaunchKernelGGL(contract_any_reduce_kernel, dim3((unsigned)((cells + 255) / 256), (unsigned)entries), dim3(256), 0, s, d, q, p);
  return hipGetLastError();
}

}  // namespace ocannl
