// The tile loops of gemm_rs and their entry point, compiled for the host: every request that a workgroup's threads make is looked at
// instead of made.  loops.inc and entry.inc are cut from the kernels' sources by tile_loops.py, which builds and runs this.  Threads
// run one after the other, so what they read from the LDS means nothing; the addresses they ask for do not depend on it.
//
// Standard input: a launch a line,
//   form M N Kl W groups pitch cols a_at b_at a_gap b_gap     (gaps in 16-byte vectors, at: the operands' own, modulo a line)
// or a call of gemm_rs_forward (bytes of workspace, which begins `ws_at` bytes behind a 16-byte boundary; 0 bytes: none),
//   call what option M N Kl W a_at b_at a_gap b_gap bytes ws_at     (what: 0, 1 to walk its launches, 2 to print their whole numbers)
// Standard output: of a launch, and of a call's whose launches are to be walked, the requests inside the buffers, those of them outside
// the operands' rows, and the 16-byte vectors of the operands' rows that nothing asked for; of a call before that the status and
// the kernels, and of any call the bytes that gemm_rs_workspace_used and _bytes answer at the end.
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "gemm_rs.h"
#include "moe_a2a.h"

#define __device__
#define __host__
#define __global__
#define __forceinline__ inline
#define __shared__ static
#define __launch_bounds__(...)
#define __align__(N) __attribute__((aligned(N)))
#define __syncthreads()
struct dim3 {
  unsigned x, y;
  dim3(unsigned x = 1, unsigned y = 1) : x(x), y(y) {}
};
typedef dim3 Dim;
typedef void* hipStream_t;
static Dim threadIdx, blockIdx, blockDim, gridDim;
struct uint2 { uint32_t x, y; };
struct uint4 { uint32_t x, y, z, w; };
struct float4 { float x, y, z, w; };
static uint2 make_uint2(uint32_t a, uint32_t b) { return {a, b}; }
static uint4 make_uint4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) { return {a, b, c, d}; }
template <class T> T min(T a, T b) { return a < b ? a : b; }
template <class T> T max(T a, T b) { return a > b ? a : b; }
static int __float_as_int(float f) { return __builtin_bit_cast(int, f); }
static float __int_as_float(int i) { return __builtin_bit_cast(float, i); }

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
struct Bf16 {
  static float lo(uint32_t) { return 0; }
  static float hi(uint32_t) { return 0; }
  static uint32_t pack(float, float) { return 0; }
};
struct F16 : Bf16 {};
template <class E> f32x4_t mfma_16x16x32(const u32x4_t&, const u32x4_t&, const f32x4_t& c) { return c; }
template <class E> f32x16_t mfma_32x32x16(const uint4&, const uint4&, const f32x16_t& c) { return c; }
template <class E> void store4(uint16_t*, const f32x4_t&) {}
constexpr int kWave = 64, kXcds = 8, kXcdCus = 32, kGemmM = 128, kGemmN = 128, kGemmK = 64, kGemmLd = kGemmK + 8, kGemmThreads = 256;

struct Buffer {
  uint64_t at;
  uint32_t bytes;
};
static void request(const Buffer& b, uint32_t offset, uint32_t scalar);
#define __amdgpu_buffer_rsrc_t Buffer
#define __builtin_amdgcn_make_buffer_rsrc(P, STRIDE, BYTES, FLAGS) Buffer{(uint64_t)(P), (uint32_t)(BYTES)}
#define __builtin_amdgcn_raw_ptr_buffer_load_lds(B, LDS, SIZE, OFFSET, SCALAR, ...) request(B, OFFSET, SCALAR)
#define __builtin_amdgcn_raw_buffer_load_b128(B, OFFSET, SCALAR, AUX) (request(B, OFFSET, SCALAR), u32x4_t{0, 0, 0, 0})
#define __builtin_amdgcn_readfirstlane(X) (X)
#define __builtin_amdgcn_sched_barrier(...)
#define __builtin_amdgcn_sched_group_barrier(...)
#define __builtin_amdgcn_s_waitcnt(...)
#define __builtin_amdgcn_s_barrier()
#define __builtin_amdgcn_s_setprio(...)
#define __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4 mfma_scaled
template <class A, class... R> static f32x4_t mfma_scaled(A, A, f32x4_t c, R...) { return c; }

#include "loops.inc"

// The launch that is walked, and what its workgroups have asked for so far: a flag for each vector of either operand's shards.
struct Operand {
  uint64_t at;      // address
  long long shard;  // vectors from one shard to the next
  int rows, kvec, shards;
  std::vector<uint8_t> asked;
  bool ask(uint64_t address) {
    const long long v = ((long long)address - (long long)at) / 16;
    if (address < at || (address - at) % 16 != 0) return false;
    const long long s = std::min(v / shard, (long long)shards - 1), in = v - s * shard;
    if (in >= (long long)rows * kvec) return false;
    asked[s * rows * kvec + in] = 1;
    return true;
  }
};
static Operand op_a, op_b;
static long long requests, outside;
static void request(const Buffer& b, uint32_t offset, uint32_t scalar) {
  if (offset >= b.bytes) return;  // (the scalar offset is not part of the hardware's check)
  ++requests;
  const uint64_t address = b.at + offset + scalar;
  if (!op_a.ask(address) && !op_b.ask(address)) ++outside;
}

template <class F>
static void walk(F kernel, Dim grid, int threads) {
  gridDim = grid;
  for (blockIdx.y = 0; blockIdx.y < grid.y; ++blockIdx.y)
    for (blockIdx.x = 0; blockIdx.x < grid.x; ++blockIdx.x)
      for (threadIdx.x = 0; threadIdx.x < (unsigned)threads; ++threadIdx.x) kernel();
}

static void place(int M, int N, int Kl, int W, int a_at, int b_at, long long a_gap, long long b_gap, bool walked) {
  const int kvec = Kl / 8;
  op_a = {(1ull << 44) + 16 * a_at, (long long)M * kvec + a_gap, M, kvec, W, std::vector<uint8_t>(walked ? (size_t)W * M * kvec : 0)};
  op_b = {(1ull << 45) + 16 * b_at, (long long)N * kvec + b_gap, N, kvec, W, std::vector<uint8_t>(walked ? (size_t)W * N * kvec : 0)};
  requests = outside = 0;
}
static void report() {
  long long missed = 0;
  for (const Operand* o : {&op_a, &op_b}) missed += std::count(o->asked.begin(), o->asked.end(), 0);
  printf("%lld %lld %lld", requests, outside, missed);
}

// What the entry point is made of besides.
enum { KID_GEMM_RS_WIDE, KID_GEMM_RS_TILE, KID_GEMM_RS_REDUCE, KID_GEMM_RS_NARROW, KID_GEMM_RS_SPLIT };
static const char* const kNames[] = {"wide", "tile", "reduce", "narrow", "split"};
static int forced;
static int option(int) { return forced; }
static bool aligned16(const void* p) { return (uintptr_t)p % 16 == 0; }
static int ceil_div(int a, int b) { return (a + b - 1) / b; }
static std::string launched;
static bool walked, numbers;
template <class T>
static void show(const T& v) {
  if constexpr (std::is_integral_v<T>) launched += "," + std::to_string(v);
}
template <class T> struct same_type { typedef T type; };
template <class... A>
static int launch(int kid, void (*kernel)(A...), Dim grid, Dim block, size_t, hipStream_t, typename same_type<A>::type... args) {
  launched += std::string(" ") + kNames[kid];
  if (numbers) (show(args), ...);
  if (walked && kid != KID_GEMM_RS_REDUCE && kernel != (void (*)(A...))nullptr) walk([&] { kernel(args...); }, grid, (int)block.x);
  return 0;
}
#include "entry.inc"

static void call() {
  int what, M, N, Kl, W, a_at, b_at, ws_at;
  long long a_gap, b_gap, bytes;
  if (scanf("%d %d %d %d %d %d %d %d %lld %lld %lld %d", &what, &forced, &M, &N, &Kl, &W, &a_at, &b_at, &a_gap, &b_gap, &bytes, &ws_at) != 12) return;
  walked = what == 1, numbers = what == 2;
  place(M, N, Kl, W, a_at, b_at, a_gap, b_gap, walked);
  launched.clear();
  std::vector<uint4> out(walked ? (size_t)M * N / 8 + 1 : 1), room(walked ? bytes / 16 + 2 : 2);
  const int rc = gemm_rs_forward((const void*)op_a.at, (const void*)op_b.at, nullptr, out.data(), M, N, Kl * W, W, op_a.shard * 8, op_b.shard * 8,
                                 MOE_A2A_BF16, bytes ? (char*)room.data() + ws_at : nullptr, (size_t)bytes, nullptr);
  printf("%d%s ", rc, launched.c_str());
  if (walked) report();
  printf(" %zu %zu\n", gemm_rs_workspace_used(M, N, Kl * W, W), gemm_rs_workspace_bytes(M, N, Kl * W, W));
}

int main() {
  char form[16];
  while (scanf("%15s", form) == 1) {
    if (form[0] == 'c') {
      call();
      continue;
    }
    int M, N, Kl, W, groups, pitch, cols, a_at, b_at;
    long long a_gap, b_gap;
    if (scanf("%d %d %d %d %d %d %d %d %d %lld %lld", &M, &N, &Kl, &W, &groups, &pitch, &cols, &a_at, &b_at, &a_gap, &b_gap) != 11) return 1;
    place(M, N, Kl, W, a_at, b_at, a_gap, b_gap, true);
    GemmRsArgs g{(const uint4*)op_a.at, (const uint4*)op_b.at, nullptr, M, N, Kl, W, op_a.shard, op_b.shard, (float)W, W / groups};
    std::vector<uint16_t> out((size_t)M * N);
    std::vector<float> partial((size_t)groups * M * N);
    const int tm = (M + pitch - 1) / pitch, tn = (N + cols - 1) / cols;
    const unsigned eighths = (unsigned)(8 * ((tm * tn + 7) / 8)), y = (unsigned)groups;
    const bool whole = Kl % 64 == 0;
    switch (form[0] == 'w' ? 0 : form[0] == 's' ? 1 : form[0] == 'n' ? 2 : 3) {
      case 0:
#define WIDE(ALONG) walk([&] { gemm_rs_wide_kernel<Bf16, ALONG>(g, out.data(), tm, tn, pitch, -1); }, Dim{eighths, 1}, kG8Threads)
        if (whole) WIDE(kG8Whole);
        else if (form[1] == 'l') WIDE(kG8Lines);
        else WIDE(kG8Ragged);
        break;
      case 1: {
        const Dim grid{(unsigned)(8 * ((tm * tn * groups + 7) / 8)), 1};
#define SPLIT(ALONG) walk([&] { gemm_rs_split_kernel<Bf16, ALONG>(g, partial.data(), tm, tn, groups, pitch, cols); }, grid, kG8Threads)
        if (whole) SPLIT(kG8Whole);
        else if (form[1] == 'l') SPLIT(kG8Lines);
        else SPLIT(kG8Ragged);
        break;
      }
      case 2:
#define NARROW(P, ALONG, SP) walk([&] { gemm_rs_narrow_kernel<Bf16, ALONG, SP, P>(g, out.data(), partial.data(), tm, tn, groups, 1); }, Dim{eighths, y}, kG8Threads)
#define NARROW_A(P, SP) (whole ? NARROW(P, kG8Whole, SP) : form[1] == 'l' ? NARROW(P, kG8Lines, SP) : NARROW(P, kG8Ragged, SP))
#define NARROW_OF(P) (groups > 1 ? NARROW_A(P, true) : NARROW_A(P, false))
        if (groups == 1) gridDim.y = 1;
        if (pitch == 256) NARROW_OF(256);
        else if (pitch == 192) NARROW_OF(192);
        else NARROW_OF(128);
        break;
      default:
#define ROWS(TN, RK, SP) walk([&] { gemm_rs_rows_kernel<Bf16, TN, RK, SP, false>(g, out.data(), partial.data()); }, Dim{(unsigned)tn, y}, kGemmThreads)
#define ROWS_K(TN, SP) (whole ? ROWS(TN, kRowsWhole, SP) : form[1] == 'l' ? ROWS(TN, kRowsLines, SP) : ROWS(TN, kRowsRagged, SP))
        if (cols == 128) groups > 1 ? ROWS_K(128, true) : ROWS_K(128, false);
        else groups > 1 ? ROWS_K(64, true) : ROWS_K(64, false);
    }
    report();
    printf("\n");
  }
  return 0;
}
