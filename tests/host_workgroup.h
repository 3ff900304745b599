// Runs a generated kernel of one 256-thread contraction tile on the host, for tests that need no GPU: the threads of a
// workgroup are fibers that take turns at barriers and matrix instructions, every tensor ends where a page that cannot
// be touched begins.  Include ahead of the kernel's source; the test supplies `host_kernel(void** tensors)`.
//   usage: program BLOCKS FILE BYTES...   (the tensors lie in FILE one after the other and are written back to it;
//   prints how many fp32 matrix instructions the threads went through)
#include <sys/mman.h>
#include <ucontext.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#define __device__
#define __global__
#define __forceinline__ inline
#define __shared__ static
#define __launch_bounds__(n)
#define __bf16 unsigned short   // (carried as bits: results are fp32)

struct HostIndex { unsigned x, y; };
static HostIndex threadIdx, blockIdx;
static ucontext_t host_scheduler, host_fiber[256];
static bool host_done[256];
static int host_turn;
static void host_yield() { const int t = host_turn; swapcontext(&host_fiber[t], &host_scheduler); }

static inline unsigned __umulhi(unsigned a, unsigned b) { return (unsigned)((unsigned long long)a * b >> 32); }
static inline float __uint_as_float(unsigned x) { float f; memcpy(&f, &x, 4); return f; }
static inline unsigned __float_as_uint(float x) { unsigned u; memcpy(&u, &x, 4); return u; }
static inline unsigned __funnelshift_r(unsigned lo, unsigned hi, int n) { return (unsigned)(((unsigned long long)hi << 32 | lo) >> (n & 31)); }

// v_mfma_f32_32x32x16_bf16 and v_mfma_f32_32x32x2_f32: lane l holds row l % 32 of its operand and the K / 2 values of k from
// (l / 32) * K / 2 on; of the result, column l % 32 and rows 8 * (e / 4) + 4 * (l / 32) + e % 4
static float host_a[2][256][8], host_b[2][256][8];
static int host_step[256];
template <typename C> static C host_mfma(const float* a, const float* b, int per_lane, C c) {
  const int t = host_turn, s = host_step[t]++ & 1, wave = t & ~63;
  memcpy(host_a[s][t], a, per_lane * sizeof(float));
  memcpy(host_b[s][t], b, per_lane * sizeof(float));
  host_yield();
  for (int e = 0; e < 16; ++e) {
    const int row = 8 * (e / 4) + 4 * ((t & 63) / 32) + e % 4;
    for (int k = 0; k < 2 * per_lane; ++k) {
      const int half = k / per_lane * 32;
      c[e] = fmaf(host_a[s][wave + half + row][k % per_lane], host_b[s][wave + half + (t & 31)][k % per_lane], c[e]);
    }
  }
  return c;
}
template <typename V, typename C> static C host_mfma_bf16(V a, V b, C c) {
  unsigned short x[8], y[8];
  float fa[8], fb[8];
  memcpy(x, &a, 16); memcpy(y, &b, 16);
  for (int i = 0; i < 8; ++i) { fa[i] = __uint_as_float((unsigned)x[i] << 16); fb[i] = __uint_as_float((unsigned)y[i] << 16); }
  return host_mfma(fa, fb, 8, c);
}
// ds_read_b64_tr_b16: of 16 lanes, lane 4 j + q points at (k = j, rows 4 q ..); lane p receives row p at k = 0 .. 3
static const unsigned short* host_at[2][256];
template <typename V> static V host_transposed(const void* at) {
  const int t = host_turn, s = host_step[t]++ & 1;
  host_at[s][t] = (const unsigned short*)at;
  host_yield();
  V v;
  for (int j = 0; j < 4; ++j) v[j] = (short)host_at[s][(t & ~15) + 4 * j + (t & 15) / 4][t & 3];
  return v;
}
#define __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, x, y, z) host_mfma_bf16(a, b, c)
static long host_f32_products;
template <typename C> static C host_mfma_f32(float a, float b, C c) { ++host_f32_products; return host_mfma(&a, &b, 1, c); }
#define __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, x, y, z) host_mfma_f32(a, b, c)
#define __builtin_amdgcn_ds_read_tr16_b64_v4i16(p) host_transposed<s16x4>((const void*)(p))
// fp32 -> bf16 bits, to nearest even
static inline unsigned short host_bf16(float x) {
  const unsigned u = __float_as_uint(x);
  return (unsigned short)(x != x ? u >> 16 | 0x40 : (u + 0x7FFF + (u >> 16 & 1)) >> 16);
}
template <typename T, typename V> static T host_bf16_pair(V v) { T t; t[0] = host_bf16(v[0]); t[1] = host_bf16(v[1]); return t; }
#define __builtin_convertvector(v, T) host_bf16_pair<T>(v)
static int host_votes[2][256];
static int __syncthreads_or(int x) {
  const int t = host_turn, s = host_step[t]++ & 1;
  host_votes[s][t] = x;
  host_yield();
  int any = 0;
  for (int i = 0; i < 256; ++i) any |= host_votes[s][i];
  return any;
}
#define __builtin_amdgcn_readfirstlane(x) (x)
#define __builtin_amdgcn_fence(...) ((void)0)
#define __builtin_amdgcn_sched_barrier(x) ((void)0)
#define __builtin_amdgcn_s_barrier() host_yield()

void host_kernel(void** tensors);
static void** host_tensors;
static void host_entry() {
  host_kernel(host_tensors);
  host_done[host_turn] = true;
  host_yield();
}

int main(int argc, char** argv) {
  const size_t page = 4096, guard = (size_t)1 << 30;
  const int n = argc - 3;
  void** p = (void**)calloc(n, sizeof(void*));
  FILE* f = fopen(argv[2], "r+b");
  if (!f || n < 1) return 2;
  for (int i = 0; i < n; ++i) {
    const size_t bytes = strtoull(argv[3 + i], nullptr, 10), room = (bytes + page - 1) / page * page;
    char* base = (char*)mmap(nullptr, room + 2 * guard, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (base == MAP_FAILED || mprotect(base + guard, room, PROT_READ | PROT_WRITE)) return 2;
    memset(base + guard, 0xFF, room);   // (NaN ahead of the tensor)
    p[i] = base + guard + room - bytes;
    if (fread(p[i], 1, bytes, f) != bytes) return 2;
  }
  host_tensors = p;
  const size_t stack = 256 * 1024;
  char* stacks = (char*)malloc(256 * stack);
  for (blockIdx.x = 0; blockIdx.x < (unsigned)atoi(argv[1]); ++blockIdx.x) {
    for (int t = 0; t < 256; ++t) {
      getcontext(&host_fiber[t]);
      host_fiber[t].uc_stack.ss_sp = stacks + t * stack;
      host_fiber[t].uc_stack.ss_size = stack;
      host_done[t] = false;
      makecontext(&host_fiber[t], host_entry, 0);
    }
    for (bool busy = true; busy;) {
      busy = false;
      for (int t = 0; t < 256; ++t) {
        if (host_done[t]) continue;
        busy = true;
        host_turn = t;
        threadIdx.x = t;
        swapcontext(&host_scheduler, &host_fiber[t]);
      }
    }
  }
  rewind(f);
  for (int i = 0; i < n; ++i) fwrite(p[i], 1, strtoull(argv[3 + i], nullptr, 10), f);
  fclose(f);
  printf("%ld\n", host_f32_products);
  return 0;
}
