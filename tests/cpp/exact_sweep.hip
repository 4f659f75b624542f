// The short quotients and roots of gbr_exact.h on the GPU against the same
// value computed in double precision and rounded to float: for a quotient or a
// root of floats whose result is normal, rounding twice gives the correctly
// rounded float (53 >= 2 * 24 + 2).  Each sweep counts the operands that differ
// and keeps one of them (tests/test_gpu_exact.py).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gbr_exact.h"

namespace {

struct Result {
  unsigned long long checked, bad;
  uint32_t a, b;  // bits of operands that differ
};

__device__ Result g_result;

constexpr int kBlocks = 2048, kThreads = 256;

__device__ bool same(float x, float y) { return __float_as_uint(x) == __float_as_uint(y); }

// a thread's counts, added to the result when it has taken all its operands
struct Tally {
  uint32_t checked = 0, bad = 0;
  __device__ void count(bool in, bool ok, float a, float b) {
    checked += in;
    if (!in || ok) return;
    ++bad;
    g_result.a = __float_as_uint(a);
    g_result.b = __float_as_uint(b);
  }
  __device__ ~Tally() {
    atomicAdd(&g_result.checked, (unsigned long long)checked);
    if (bad) atomicAdd(&g_result.bad, (unsigned long long)bad);
  }
};

__device__ bool within(float x, int lo, int hi) {  // 2^lo <= |x| <= 2^hi
  const double v = fabs((double)x);
  return v >= ldexp(1.0, lo) && v <= ldexp(1.0, hi);
}

// n floats from bit pattern `first` on
__global__ __launch_bounds__(kThreads) void k_rcp(uint32_t first, uint64_t n) {
  Tally t;
  for (uint64_t i = blockIdx.x * (uint64_t)kThreads + threadIdx.x; i < n; i += (uint64_t)kBlocks * kThreads) {
    const float x = __uint_as_float(first + (uint32_t)i);
    const bool in = within(x, -126, 126);
    t.count(in, same(gbr::rcp_exact(x), (float)(1.0 / (double)x)), 1.0f, x);
  }
}

__global__ __launch_bounds__(kThreads) void k_sqrt(uint32_t first, uint64_t n) {
  Tally t;
  for (uint64_t i = blockIdx.x * (uint64_t)kThreads + threadIdx.x; i < n; i += (uint64_t)kBlocks * kThreads) {
    const float x = __uint_as_float(first + (uint32_t)i);
    const bool in = x > 0.0f && within(x, -80, 80);
    t.count(in, same(gbr::sqrt_exact(x), (float)sqrt((double)x)), x, 0.0f);
  }
}

__device__ void check_div(Tally& t, bool in, float a, float b) {
  const float q = (float)((double)a / (double)b);
  // (the sign of a zero is not kept)
  const float short_q = gbr::div_exact(a, b, gbr::rcp_exact(b));
  t.count(in, a == 0.0f ? short_q == 0.0f : same(short_q, q), a, b);
}

__device__ uint64_t mix(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

// a float of random sign and mantissa (one in eight within 16 units of a power
// of two, where the rounding is tightest) and an exponent of [lo, hi]
__device__ float draw(uint64_t bits, int lo, int hi) {
  uint32_t m = (uint32_t)bits & 0x7fffffu;
  if ((bits >> 23 & 7u) == 0) m = (bits >> 26 & 1u) ? 0x7fffffu - (m & 15u) : m & 15u;
  const int e = lo + (int)((uint32_t)(bits >> 32) % (uint32_t)(hi - lo + 1));
  return __uint_as_float((uint32_t)(bits >> 27 & 1u) << 31 | (uint32_t)(e + 127) << 23 | m);
}

__global__ __launch_bounds__(kThreads) void k_div(uint64_t seed, uint64_t n, int alo, int ahi, int blo, int bhi, int qlo,
                                                  int qhi) {
  Tally t;
  for (uint64_t i = blockIdx.x * (uint64_t)kThreads + threadIdx.x; i < n; i += (uint64_t)kBlocks * kThreads) {
    const float a = draw(mix(seed + 2 * i), alo, ahi), b = draw(mix(seed + 2 * i + 1), blo, bhi);
    const double q = fabs((double)a / (double)b);
    check_div(t, q >= ldexp(1.0, qlo) && q <= ldexp(1.0, qhi), a, b);
  }
}

// num / k for k = 1 .. n
__global__ __launch_bounds__(kThreads) void k_div_integers(float num, uint64_t n) {
  Tally t;
  for (uint64_t i = blockIdx.x * (uint64_t)kThreads + threadIdx.x; i < n; i += (uint64_t)kBlocks * kThreads)
    check_div(t, true, num, (float)(i + 1));
}

// (m - 1) / (m + 1) for every m of [1, 2)
__global__ __launch_bounds__(kThreads) void k_div_log2() {
  Tally t;
  for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < (1u << 23); i += kBlocks * kThreads) {
    const float m = __uint_as_float(0x3f800000u | i);
    check_div(t, true, m - 1.0f, m + 1.0f);
  }
}

int finish(Result* out) {
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpyFromSymbol(out, HIP_SYMBOL(g_result), sizeof *out);
  return (int)e;
}

int begin() {
  const Result zero{};
  return (int)hipMemcpyToSymbol(HIP_SYMBOL(g_result), &zero, sizeof zero);
}

}  // namespace

extern "C" {

int exact_rcp(Result* out) {
  if (int e = begin()) return e;
  k_rcp<<<kBlocks, kThreads>>>(0u, 1ull << 32);
  return finish(out);
}

int exact_sqrt(Result* out) {
  if (int e = begin()) return e;
  k_sqrt<<<kBlocks, kThreads>>>(0u, 1ull << 31);
  return finish(out);
}

int exact_div(uint64_t seed, uint64_t n, const int* range, Result* out) {
  if (int e = begin()) return e;
  k_div<<<kBlocks, kThreads>>>(seed, n, range[0], range[1], range[2], range[3], range[4], range[5]);
  return finish(out);
}

int exact_div_integers(float num, uint64_t n, Result* out) {
  if (int e = begin()) return e;
  k_div_integers<<<kBlocks, kThreads>>>(num, n);
  return finish(out);
}

int exact_div_log2(Result* out) {
  if (int e = begin()) return e;
  k_div_log2<<<kBlocks, kThreads>>>();
  return finish(out);
}

}  // extern "C"
