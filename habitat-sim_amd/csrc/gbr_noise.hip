// Redwood depth noise model on the GPU (src/esp/sensor/RedwoodNoiseModel.cu,
// RedwoodNoiseModel.h; Python face redwood_depth_noise_model.py): pixel
// shuffle by N(0, 0.25 m) in x and y, 2x2 downsample, the 80x80x5
// undistortion table of the 640x480 Redwood sensor, disparity quantisation
// to 1/8 with N(0, 0.027778 m) noise, 0 beyond 10 m.
//
// One thread per output pixel of a batch of images.  The three standard
// normal deviates of a pixel come either from the caller or from a
// counter-based generator: one Philox4x32-10 block (Salmon et al., "Parallel
// random numbers: as easy as 1, 2, 3", SC'11) per (call, pixel) with the
// model's seed as key, turned into normals by the Box-Muller transform.  A
// counter generator needs no per-thread state in memory (the reference keeps
// a curand state per thread) and makes every call reproducible from (seed,
// call index).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <new>
#include <string>

#include "gbr.h"
#include "gbr_exact.h"
#include "gbr_host.h"

#pragma STDC FP_CONTRACT OFF

namespace gbr {
namespace {

constexpr int kRwCols = 80, kRwDims = 5;
constexpr int kNoiseBlock = 256;

__device__ __forceinline__ void philox4x32(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                           uint32_t k0, uint32_t k1, uint32_t* out) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    // one 64-bit product (v_mad_u64_u32) instead of its two halves, and both
    // exclusive ors in one operation
    const uint64_t p0 = (uint64_t)c0 * 0xD2511F53u, p1 = (uint64_t)c2 * 0xCD9E8D57u;
    c0 = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c1, k0, 0x96);
    c1 = (uint32_t)p1;
    c2 = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c3, k1, 0x96);
    c3 = (uint32_t)p0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  out[0] = c0;
  out[1] = c1;
  out[2] = c2;
  out[3] = c3;
}

// uniform in (0, 1): the top 24 bits plus a half, by 2^-24
__device__ __forceinline__ float unit_open(uint32_t x) {
  return __builtin_fmaf((float)(x >> 8), 0x1p-24f, 0x1p-25f);
}

// three N(0, 1) deviates of pixel `g` in call `call`
__device__ __forceinline__ void pixel_normals(uint64_t seed, uint64_t call, uint64_t g,
                                              float* n) {
  uint32_t r[4];
  philox4x32((uint32_t)g, (uint32_t)(g >> 32), (uint32_t)call, (uint32_t)(call >> 32),
             (uint32_t)seed, (uint32_t)(seed >> 32), r);
  // Box-Muller with the hardware transcendental instructions (~1 ulp;
  // deviates need a distribution, not correctly rounded values):
  // -2 ln u = -2 ln2 log2 u; v_sin/v_cos take the angle in revolutions
  const float m2ln2 = -1.38629436111989061883f;
  const float ra = __builtin_amdgcn_sqrtf(m2ln2 * __builtin_amdgcn_logf(unit_open(r[0])));
  const float rb = __builtin_amdgcn_sqrtf(m2ln2 * __builtin_amdgcn_logf(unit_open(r[2])));
  const float ta = unit_open(r[1]), tb = unit_open(r[3]);
  n[0] = ra * __builtin_amdgcn_cosf(ta);
  n[1] = ra * __builtin_amdgcn_sinf(ta);
  n[2] = rb * __builtin_amdgcn_cosf(tb);
}

// n / d for n < 2^31 by a multiplication: d > 1 is fixed for a launch
// (Granlund & Montgomery 1994: with 2^(shift-1) < d <= 2^shift and
// mul = ceil(2^(31 + shift) / d) the error stays below 1 / d)
struct Divider {
  uint32_t mul, shift;  // n / d = (n * mul >> 32) >> shift
};

Divider make_divider(uint32_t d) {
  uint32_t s = 1;
  while ((1ull << s) < d) ++s;
  return {(uint32_t)(((1ull << (31 + s)) + d - 1) / d), s - 1};
}

// the largest float that is a row or column number of a side of n pixels:
// n - 1 itself up to 2^24, beyond which (float)(n - 1) may round up to n and
// a pixel clamped to it lies outside the image
float last_index(int n) {
  const float f = (float)(n - 1);
  return (double)f > (double)(n - 1) ? std::nextafter(f, 0.0f) : f;
}

__device__ __forceinline__ uint32_t divide(uint32_t n, Divider d) { return __umulhi(n, d.mul) >> d.shift; }

// the disparity step in the general arithmetic
__device__ __forceinline__ float disparity(float u, float nz) {
  double t = (double)35.130f / (double)u;
  t = t + (double)nz;
  t = t * 8.0;
  const double q = round(t);
  return q > 1e-5 ? (float)((double)(35.130f * 8.0f) / q) : 0.0f;
}

struct RedwoodArgs {
  const float* depth;    // images x rows x cols, consecutive
  const float* model;
  const float* normals;  // 3 per pixel, or null (generator)
  float* out;
  uint32_t total;        // pixels, < 2^31
  uint32_t npx, W;
  Divider by_npx, by_w;
  float xmax, ymax;      // last_index() of W and H
  double rx, ry;         // 1 / (W - 1), 1 / (H - 1), the sides rounded to floats
  float mult, mult4;     // the noise multiplier, and a quarter of it
  uint64_t seed, call, first;  // first: the generator's number of pixel 0
};

// One thread per pixel.  8 bytes a pixel move, but what bounds the kernel is
// the arithmetic: ten Philox rounds, two Box-Muller transforms, five quotients
// and four integer divisions (one of 64 bits), 340 vector operations a pixel in
// the general forms and 165 here: 512 images of 128x128 take 35 us, and took 56
// (the copy of their bytes takes 13).  Every quotient is the cheapest form that
// rounds the same:
//  * pixel -> image, row, column: multiplications (`Divider`);
//  * x / (W - 1): (float)((double)x * rx).  The product errs by less than 2^-52,
//    and a quotient of two 24-bit numbers lies at least 2^-49 from the middle
//    between two floats;
//  * z / f and 281.04 / q: div_exact();
//  * 35.13 / u in double: one Newton step from the single reciprocal (2^-45)
//    and a correction by the exact remainder (2^-90); the quotient of two
//    24-bit numbers lies at least 2^-78 from the middle between two doubles;
//  * the last quotient in single precision: for two floats a double quotient
//    rounded to float is the float quotient (53 >= 2 * 24 + 2).
// Operands outside their ranges (depths under a millimetre, factors f over 8,
// quotients q of 2^23 and more, infinities and NaN in the table) take the
// general arithmetic.
__global__ __launch_bounds__(kNoiseBlock) void k_redwood(RedwoodArgs a) {
  const uint32_t g = blockIdx.x * kNoiseBlock + threadIdx.x;
  if (g >= a.total) return;
  const uint32_t img = divide(g, a.by_npx), idx = g - img * a.npx;
  float n[3];
  if (a.normals) {
    const float* nn = a.normals + 3 * (size_t)g;
    n[0] = nn[0];
    n[1] = nn[1];
    n[2] = nn[2];
  } else {
    pixel_normals(a.seed, a.call, a.first + g, n);
  }
  const uint32_t j = divide(idx, a.by_w), i = idx - j * a.W;
  const float fy = n[0] * a.mult4 + (float)(int)j;
  const float fx = n[1] * a.mult4 + (float)(int)i;
  // nearest row and column, clamped (the median; 0 for NaN)
  const int y = (int)__builtin_amdgcn_fmed3f(fy + 0.5f, 0.0f, a.ymax);
  const int x = (int)__builtin_amdgcn_fmed3f(fx + 0.5f, 0.0f, a.xmax);
  const float d = a.depth[(size_t)(g - idx + (uint32_t)(y & ~1) * a.W + (uint32_t)(x & ~1))];
  float res = 0.0f;
  // beyond 10 m the sensor returns 0; zero, negative and NaN depths give 0 too
  if (d > 0.0f && d < 10.0f) {
    float ux = (float)((double)(float)x * a.rx);
    ux = ux * 639.0f;
    ux = ux + 0.5f;
    float uy = (float)((double)(float)y * a.ry);
    uy = uy * 479.0f;
    uy = uy + 0.5f;
    // the undistortion factor of (column / 8, row / 6) at this depth (the
    // product is row / 6 for rows up to 1000)
    const uint32_t cell = (__umul24((uint32_t)(int)uy, 10923u) >> 16) * kRwCols + ((uint32_t)(int)ux >> 3);
    const int i2 = (int)((d + 1.0f) * 0.5f);
    const float w = (d - __builtin_fmaf((float)i2, 2.0f, -1.0f)) * 0.5f;
    const uint32_t at = cell * kRwDims;
    const float wa = 1.0f - w;
    const float p = wa * a.model[at + (uint32_t)max(i2 - 1, 0)];
    const float q = w * a.model[at + (uint32_t)min(i2, 4)];
    const float f = p + q;
    if (!(f < 1e-5f)) {
      float nz = n[2] * 0.027778f;
      nz = nz * a.mult;
      const float u = div_exact(d, f, rcp_exact(f));
      const double du = (double)u, r0 = (double)__builtin_amdgcn_rcpf(u);
      const double r1 = __builtin_fma(__builtin_fma(-du, r0, 1.0), r0, r0);
      const double q0 = (double)35.130f * r1;
      double t = __builtin_fma(__builtin_fma(-du, q0, (double)35.130f), r1, q0);
      t = t + (double)nz;
      if (d >= 0x1p-10f && f <= 8.0f && fabs(t) < 0x1p20) {
        // 8 t rounded half away from zero: half to even, and one more where
        // that went down from a half (a negative one ends as 0 either way)
        const double shifted = __builtin_fma(t, 8.0, 0x1.8p52);
        int k = (int)(uint32_t)__builtin_bit_cast(uint64_t, shifted);
        k += __builtin_fma(t, 8.0, 0x1.8p52 - shifted) == 0.5 ? 1 : 0;
        const float kf = (float)k;
        if (k > 0) res = div_exact(35.130f * 8.0f, kf, rcp_exact(kf));
      } else {
        const float v = d / f;
        if (v != 0.0f) res = disparity(v, nz);
      }
    }
  }
  a.out[g] = res;
}

__global__ __launch_bounds__(kNoiseBlock) void k_philox_bits(uint64_t seed, uint64_t call,
                                                             uint64_t first, uint64_t n,
                                                             uint32_t* __restrict__ out) {
  const uint64_t k = (uint64_t)blockIdx.x * kNoiseBlock + threadIdx.x;
  if (k >= n) return;
  const uint64_t g = first + k;
  uint32_t r[4];
  philox4x32((uint32_t)g, (uint32_t)(g >> 32), (uint32_t)call, (uint32_t)(call >> 32),
             (uint32_t)seed, (uint32_t)(seed >> 32), r);
  uint4 v;
  v.x = r[0];
  v.y = r[1];
  v.z = r[2];
  v.w = r[3];
  reinterpret_cast<uint4*>(out)[k] = v;
}

}  // namespace

// Staging of gbr_redwood_simulate_host_noalloc(): the input depth image in
// the first kRwScratchPixels floats, the output image in the second.  Every
// GPU the library runs on holds its own copy (8 MiB) until the process ends.
// Host code never names the array in a launch or copy: it uses the per-device
// address from hipGetSymbolAddress (scratch_address below).
constexpr long long kRwScratchPixels = GBR_REDWOOD_NOALLOC_MAX_PIXELS;
static __device__ __align__(256) float scratch[2 * kRwScratchPixels];

namespace {

constexpr int kScratchDevices = 64;
std::mutex g_scratch_mutex;
float* g_scratch[kScratchDevices] = {};

// the device address of `scratch` on device `dev`, which must be current;
// looked up once per device
gbr_status scratch_address(int dev, float** out) {
  if (dev < 0 || dev >= kScratchDevices)
    return fail(GBR_ERR_UNSUPPORTED, "redwood_create: device ordinal beyond the scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(GBR_ERR_DEVICE, std::string("redwood_create: hipGetSymbolAddress(scratch): ") +
                                      hipGetErrorString(e));
    g_scratch[dev] = static_cast<float*>(p);
  }
  *out = g_scratch[dev];
  return GBR_OK;
}

}  // namespace
}  // namespace gbr

struct gbr_redwood {
  int device = 0;
  float mult = 1.0f;
  uint64_t seed = 0;
  uint64_t calls = 0;  // generator calls so far (the counter's high word)
  gbr::DevBuf<float> d_model;
  gbr::DevBuf<float> d_in, d_out;  // staging of the host entry point
  float* scratch = nullptr;        // this device's `scratch` (no-allocation entry point)
};

using gbr::fail;

namespace {

gbr_status check_dims(int32_t images, int32_t rows, int32_t cols, const char* fn) {
  if (images < 0 || rows < 2 || cols < 2)
    return fail(GBR_ERR_ARGUMENT, std::string(fn) + ": need images >= 0 and images of at least 2x2 pixels");
  if ((long long)rows * cols >= (1ll << 31))
    return fail(GBR_ERR_SIZE, std::string(fn) + ": image of 2^31 pixels or more");
  return GBR_OK;
}

gbr_status launch(gbr_redwood* m, const float* depth, int32_t images, int32_t rows, int32_t cols,
                  const float* normals, float* out, hipStream_t s) {
  const long long npx = (long long)rows * cols, total = images * npx;
  if (total == 0) return GBR_OK;
  if ((total + gbr::kNoiseBlock - 1) / gbr::kNoiseBlock > 0x7fffffffll)
    return fail(GBR_ERR_SIZE, "redwood: batch too large");
  gbr::RedwoodArgs a{};
  a.model = m->d_model.ptr;
  a.npx = (uint32_t)npx;
  a.W = (uint32_t)cols;
  a.by_npx = gbr::make_divider(a.npx);
  a.by_w = gbr::make_divider(a.W);
  a.xmax = gbr::last_index(cols);
  a.ymax = gbr::last_index(rows);
  a.rx = 1.0 / (double)(float)(cols - 1);
  a.ry = 1.0 / (double)(float)(rows - 1);
  a.mult = m->mult;
  a.mult4 = m->mult * 0.25f;
  a.seed = m->seed;
  a.call = m->calls;
  // launches of as many whole images as keep the pixel number under 2^31
  const long long run = 0x7fffffffll / npx * npx;
  for (long long first = 0; first < total; first += run) {
    a.depth = depth + first;
    a.normals = normals ? normals + 3 * first : nullptr;
    a.out = out + first;
    a.first = (uint64_t)first;
    a.total = (uint32_t)std::min(run, total - first);
    hipLaunchKernelGGL(gbr::k_redwood, dim3((a.total + gbr::kNoiseBlock - 1) / gbr::kNoiseBlock),
                       dim3(gbr::kNoiseBlock), 0, s, a);
    HIP_TRY(hipGetLastError());
  }
  if (!normals) ++m->calls;
  return GBR_OK;
}

}  // namespace

extern "C" {

gbr_status gbr_redwood_create(const float* model, int32_t device, float noise_multiplier,
                              uint64_t seed, gbr_redwood** out) {
  if (!model || !out) return fail(GBR_ERR_ARGUMENT, "redwood_create: null argument");
  *out = nullptr;
  if (!std::isfinite(noise_multiplier))
    return fail(GBR_ERR_ARGUMENT, "redwood_create: noise multiplier is not finite");
  int ndev = 0;
  HIP_TRY(hipGetDeviceCount(&ndev));
  int dev = device;
  if (dev < 0) HIP_TRY(hipGetDevice(&dev));
  if (dev >= ndev) return fail(GBR_ERR_ARGUMENT, "redwood_create: device ordinal out of range");
  HIP_TRY(hipSetDevice(dev));
  gbr_redwood* m = new (std::nothrow) gbr_redwood();
  if (!m) return fail(GBR_ERR_OOM, "redwood_create: out of host memory");
  m->device = dev;
  m->mult = noise_multiplier;
  m->seed = seed;
  const size_t n = (size_t)GBR_REDWOOD_MODEL_FLOATS;
  gbr_status st = gbr::scratch_address(dev, &m->scratch);
  if (st == GBR_OK) st = m->d_model.reserve(n);
  if (st == GBR_OK) {
    const hipError_t e = hipMemcpy(m->d_model.ptr, model, n * sizeof(float), hipMemcpyHostToDevice);
    if (e != hipSuccess) st = fail(GBR_ERR_DEVICE, std::string("redwood_create: ") + hipGetErrorString(e));
  }
  if (st != GBR_OK) {
    delete m;
    return st;
  }
  *out = m;
  return GBR_OK;
}

gbr_status gbr_redwood_destroy(gbr_redwood* m) {
  if (!m) return GBR_OK;
  (void)hipSetDevice(m->device);
  delete m;
  return GBR_OK;
}

gbr_status gbr_redwood_simulate(gbr_redwood* m, const float* depth, int32_t images, int32_t rows,
                                int32_t cols, float* out, void* stream) {
  if (!m || !depth || !out) return fail(GBR_ERR_ARGUMENT, "redwood_simulate: null argument");
  TRY(check_dims(images, rows, cols, "redwood_simulate"));
  HIP_TRY(hipSetDevice(m->device));
  return launch(m, depth, images, rows, cols, nullptr, out, static_cast<hipStream_t>(stream));
}

gbr_status gbr_redwood_simulate_normals(gbr_redwood* m, const float* depth, int32_t images,
                                        int32_t rows, int32_t cols, const float* normals,
                                        float* out, void* stream) {
  if (!m || !depth || !normals || !out)
    return fail(GBR_ERR_ARGUMENT, "redwood_simulate_normals: null argument");
  TRY(check_dims(images, rows, cols, "redwood_simulate_normals"));
  HIP_TRY(hipSetDevice(m->device));
  return launch(m, depth, images, rows, cols, normals, out, static_cast<hipStream_t>(stream));
}

gbr_status gbr_redwood_simulate_host(gbr_redwood* m, const float* depth, int32_t rows, int32_t cols,
                                     float* out) {
  if (!m || !depth || !out) return fail(GBR_ERR_ARGUMENT, "redwood_simulate_host: null argument");
  TRY(check_dims(1, rows, cols, "redwood_simulate_host"));
  HIP_TRY(hipSetDevice(m->device));
  const size_t n = (size_t)rows * cols;
  TRY(m->d_in.reserve(n));
  TRY(m->d_out.reserve(n));
  HIP_TRY(hipMemcpy(m->d_in.ptr, depth, n * sizeof(float), hipMemcpyHostToDevice));
  TRY(launch(m, m->d_in.ptr, 1, rows, cols, nullptr, m->d_out.ptr, nullptr));
  HIP_TRY(hipMemcpy(out, m->d_out.ptr, n * sizeof(float), hipMemcpyDeviceToHost));
  return GBR_OK;
}

gbr_status gbr_redwood_simulate_host_noalloc(gbr_redwood* m, const float* depth, int32_t rows,
                                             int32_t cols, float* out) {
  if (!m || !depth || !out)
    return fail(GBR_ERR_ARGUMENT, "redwood_simulate_host_noalloc: null argument");
  TRY(check_dims(1, rows, cols, "redwood_simulate_host_noalloc"));
  const long long n = (long long)rows * cols;
  if (n > gbr::kRwScratchPixels)
    return fail(GBR_ERR_SIZE, "redwood_simulate_host_noalloc: rows x cols = " + std::to_string(n) +
                                  " exceeds GBR_REDWOOD_NOALLOC_MAX_PIXELS (" +
                                  std::to_string(gbr::kRwScratchPixels) + ")");
  if (!m->scratch) return fail(GBR_ERR_STATE, "redwood_simulate_host_noalloc: no scratch address");
  HIP_TRY(hipSetDevice(m->device));
  // the input region is written whole before the kernel reads it, and the
  // kernel writes every output pixel: nothing in the scratch needs clearing
  float* in = m->scratch;
  float* res = m->scratch + gbr::kRwScratchPixels;
  HIP_TRY(hipMemcpy(in, depth, (size_t)n * sizeof(float), hipMemcpyHostToDevice));
  TRY(launch(m, in, 1, rows, cols, nullptr, res, nullptr));
  HIP_TRY(hipMemcpy(out, res, (size_t)n * sizeof(float), hipMemcpyDeviceToHost));
  return GBR_OK;
}

gbr_status gbr_redwood_calls(const gbr_redwood* m, uint64_t* out) {
  if (!m || !out) return fail(GBR_ERR_ARGUMENT, "redwood_calls: null argument");
  *out = m->calls;
  return GBR_OK;
}

gbr_status gbr_redwood_random_bits(gbr_redwood* m, uint64_t call, uint64_t first, uint64_t n,
                                   uint32_t* out, void* stream) {
  if (!m || (!out && n)) return fail(GBR_ERR_ARGUMENT, "redwood_random_bits: null argument");
  if (n == 0) return GBR_OK;
  const uint64_t blocks = (n + gbr::kNoiseBlock - 1) / gbr::kNoiseBlock;
  if (blocks > 0x7fffffffull) return fail(GBR_ERR_SIZE, "redwood_random_bits: too many blocks");
  HIP_TRY(hipSetDevice(m->device));
  hipLaunchKernelGGL(gbr::k_philox_bits, dim3((uint32_t)blocks), dim3(gbr::kNoiseBlock), 0,
                     static_cast<hipStream_t>(stream), m->seed, call, first, n, out);
  HIP_TRY(hipGetLastError());
  return GBR_OK;
}

}  // extern "C"
