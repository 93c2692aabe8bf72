// fa_quant.hip - per-tensor e4m3 quantisation for the fp8 forward (fa_quantize_fp8, fa_quantize_fp8_amax).
//
// Two passes over the tensor, the least there can be when the scale is the tensor's own maximum: one
// reads it for max |x|, one reads it again and writes the e4m3 codes.  Both are bound by memory.  As
// chained elementwise PyTorch operations (to float32, abs, max, divide, clamp, convert) the same work
// moved about eight times the bytes.  Quantising q, k and v and the fp8 forward of a full causal layer
// (L = 8192, Hq = 64, Hkv = 8, D = 64, bfloat16 in): 882 -> 599 us, of which the forward is 515.  The
// host waits for the maximum only, behind which the codes are already being written, so three
// tensors in a row keep the GPU busy but for the launches.
//
// The codes are those of (x / descale).clamp(-448, 448).to(float8_e4m3fn) on float32 values, where
// PyTorch divides a GPU tensor by a host number (a double) as a product with that number's reciprocal rounded
// to float32; NaNs stay NaNs of their sign (this file is compiled with NaNs honoured).
#include <hip/hip_runtime.h>

#include <cstring>

#include "../../include/fa_gfx950.h"
#include "fa_common.h"

namespace fa {
namespace {

constexpr float kE4m3Max = 448.f;
constexpr int kThreads = 256;

// element types of a 16-byte load
struct LoadBF16 {
  static constexpr int N = 8;
  static __device__ void get(u32x4 v, float (&x)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = __builtin_bit_cast(float, v[i] << 16);
      x[2 * i + 1] = __builtin_bit_cast(float, v[i] & 0xffff0000u);
    }
  }
};
struct LoadF16 {
  static constexpr int N = 8;
  static __device__ void get(u32x4 v, float (&x)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w = v[i];  // (a bit cast of v[i] itself would take element 0)
      const f16x2 h = __builtin_bit_cast(f16x2, w);
      x[2 * i] = float(h[0]);
      x[2 * i + 1] = float(h[1]);
    }
  }
};
struct LoadF32 {
  static constexpr int N = 4;
  static __device__ void get(u32x4 v, float (&x)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w = v[i];
      x[i] = __builtin_bit_cast(float, w);
    }
  }
};

// The last, partial 16 bytes of the tensor (zeros past its end).
template <typename T>
__device__ u32x4 load_tail(const void* x, int64_t n, int64_t first) {
  constexpr int EB = 16 / T::N;
  uint32_t w[4] = {0, 0, 0, 0};
  for (int i = 0; first + i < n; ++i) {
    if (EB == 2) w[i / 2] |= uint32_t(static_cast<const uint16_t*>(x)[first + i]) << (16 * (i & 1));
    else w[i] = static_cast<const uint32_t*>(x)[first + i];
  }
  return u32x4{w[0], w[1], w[2], w[3]};
}

// The largest |x| as float bits, whose order as unsigned numbers is that of the values, NaNs above all.
__device__ uint32_t block_max(uint32_t m) {
  __shared__ uint32_t wave_m[kThreads / 64];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = max(m, uint32_t(__shfl_xor(int(m), o)));
  if ((threadIdx.x & 63) == 0) wave_m[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kThreads / 64; ++w) m = max(m, wave_m[w]);
  return m;
}

// Workgroup i's largest |x| to parts[i] (all FA_AMAX_PARTS of them) and, for the host, host_parts[i].
template <typename T>
__global__ __launch_bounds__(kThreads) void amax_kernel(const void* x, int64_t n, float* parts, float* host_parts) {
  const int64_t whole = n / T::N;  // 16-byte pieces
  const u32x4* p = static_cast<const u32x4*>(x);
  const int64_t step = int64_t(gridDim.x) * kThreads;
  uint32_t m = 0;
  auto take = [&](u32x4 v) {
    float f[T::N];
    T::get(v, f);
#pragma unroll
    for (int j = 0; j < T::N; ++j) m = max(m, __builtin_bit_cast(uint32_t, f[j]) & 0x7fffffffu);
  };
  int64_t i = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  for (; i + 3 * step < whole; i += 4 * step) {  // four loads in flight
    const u32x4 a = p[i], b = p[i + step], c = p[i + 2 * step], d = p[i + 3 * step];
    take(a);
    take(b);
    take(c);
    take(d);
  }
  for (; i < whole; i += step) take(p[i]);
  if (whole * T::N < n && blockIdx.x == 0 && threadIdx.x == 0) take(load_tail<T>(x, n, whole * T::N));
  m = block_max(m);
  if (threadIdx.x == 0) {
    parts[blockIdx.x] = __builtin_bit_cast(float, m);
    host_parts[blockIdx.x] = __builtin_bit_cast(float, m);
  }
}

// out[i] = e4m3(clamp(x[i] * inv)); with `parts`, inv is the reciprocal of max(parts) / 448 (1 when
// the maximum is 0 or NaN), rounded to float32 as PyTorch rounds it.
template <typename T>
__global__ __launch_bounds__(kThreads) void quantize_kernel(const void* x, int64_t n, uint8_t* out, float inv,
                                                            const float* parts) {
  if (parts) {
    uint32_t m = 0;
    for (int i = threadIdx.x; i < FA_AMAX_PARTS; i += kThreads) m = max(m, __builtin_bit_cast(uint32_t, parts[i]));
    m = block_max(m);
    const float amax = __builtin_bit_cast(float, m);
    inv = amax > 0.f ? float(1.0 / (double(amax) / 448.0)) : 1.f;
  }
  auto clamp = [](float a) { return a < -kE4m3Max ? -kE4m3Max : a > kE4m3Max ? kE4m3Max : a; };
  auto code2 = [&](float a, float b, int old, bool hi) {
    a = clamp(a);
    b = clamp(b);
    return hi ? __builtin_amdgcn_cvt_pk_fp8_f32(a, b, old, true) : __builtin_amdgcn_cvt_pk_fp8_f32(a, b, old, false);
  };
  // a unit is 16 codes
  constexpr int PIECES = 16 / T::N;
  const u32x4* p = static_cast<const u32x4*>(x);
  const int64_t units = n / 16, step = int64_t(gridDim.x) * kThreads;
  auto encode = [&](const u32x4 (&v)[PIECES]) {
    float f[16];
    bool nan = false;
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
      float g[T::N];
      T::get(v[j], g);
#pragma unroll
      for (int e = 0; e < T::N; ++e) {
        f[T::N * j + e] = g[e] * inv;
        nan |= f[T::N * j + e] != f[T::N * j + e];
      }
    }
    u32x4 o;
#pragma unroll
    for (int w = 0; w < 4; ++w) o[w] = uint32_t(code2(f[4 * w + 2], f[4 * w + 3], code2(f[4 * w], f[4 * w + 1], 0, false), true));
    if (nan) {  // the conversion gives every NaN the code 0xff; a NaN keeps its sign (of two, the scale's counts)
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (f[i] != f[i]) o[i / 4] ^= (~__builtin_bit_cast(uint32_t, inv != inv ? inv : f[i]) >> 31) << (8 * (i % 4) + 7);
    }
    return o;
  };
  for (int64_t u = int64_t(blockIdx.x) * kThreads + threadIdx.x; u < units; u += step) {
    u32x4 v[PIECES];
#pragma unroll
    for (int j = 0; j < PIECES; ++j) v[j] = p[u * PIECES + j];
    *reinterpret_cast<u32x4*>(out + 16 * u) = encode(v);
  }
  if (16 * units < n && blockIdx.x == 0 && threadIdx.x == 0) {  // the last, partial unit
    u32x4 v[PIECES];
#pragma unroll
    for (int j = 0; j < PIECES; ++j) v[j] = load_tail<T>(x, min(n, 16 * units + T::N * (j + 1)), 16 * units + T::N * j);
    const u32x4 o = encode(v);
    for (int i = 0; 16 * units + i < n; ++i) out[16 * units + i] = uint8_t(o[i / 4] >> (8 * (i % 4)));
  }
}

int status(const void* x, const void* out, int32_t dtype, int64_t n) {
  if (!x || !out) return FA_ERR_NULL;
  if (n < 1 || n >= (int64_t(1) << 40)) return FA_ERR_SHAPE;
  if (dtype != FA_DTYPE_BF16 && dtype != FA_DTYPE_F16 && dtype != FA_DTYPE_F32) return FA_ERR_DTYPE;
  if ((reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(out) & 15)) return FA_ERR_ALIGN;
  return FA_OK;
}

}  // namespace
}  // namespace fa

namespace fa {
namespace {

void launch_quantize(const void* x, int32_t dtype, int64_t n, void* out, float inv, const float* parts, hipStream_t s) {
  const int64_t wgs = ((n + 15) / 16 + kThreads - 1) / kThreads;
  const dim3 grid(unsigned(wgs < 2048 ? wgs : 2048)), block(kThreads);
  uint8_t* o = static_cast<uint8_t*>(out);
  if (dtype == FA_DTYPE_BF16) hipLaunchKernelGGL(quantize_kernel<LoadBF16>, grid, block, 0, s, x, n, o, inv, parts);
  else if (dtype == FA_DTYPE_F16) hipLaunchKernelGGL(quantize_kernel<LoadF16>, grid, block, 0, s, x, n, o, inv, parts);
  else hipLaunchKernelGGL(quantize_kernel<LoadF32>, grid, block, 0, s, x, n, o, inv, parts);
}

}  // namespace
}  // namespace fa

extern "C" int fa_quantize_fp8(const void* x, int32_t dtype, int64_t n, void* out, double descale, void* stream) {
  const int rc = fa::status(x, out, dtype, n);
  if (rc != FA_OK) return rc;
  fa::launch_quantize(x, dtype, n, out, float(1.0 / descale), nullptr, static_cast<hipStream_t>(stream));
  return hipGetLastError() == hipSuccess ? FA_OK : FA_ERR_LAUNCH;
}

extern "C" int fa_quantize_fp8_amax(const void* x, int32_t dtype, int64_t n, void* out, float* parts, float* host_parts,
                                    float* amax, void* stream) {
  const int rc = fa::status(x, out, dtype, n);
  if (rc != FA_OK) return rc;
  if (!parts || !host_parts || !amax) return FA_ERR_NULL;
  const dim3 grid(FA_AMAX_PARTS), block(fa::kThreads);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  hipStreamCaptureStatus capture;  // (the host cannot wait for a captured kernel, which would write `host_parts` at replays)
  if (hipStreamIsCapturing(s, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) return FA_ERR_LAUNCH;
  if (dtype == FA_DTYPE_BF16) hipLaunchKernelGGL(fa::amax_kernel<fa::LoadBF16>, grid, block, 0, s, x, n, parts, host_parts);
  else if (dtype == FA_DTYPE_F16) hipLaunchKernelGGL(fa::amax_kernel<fa::LoadF16>, grid, block, 0, s, x, n, parts, host_parts);
  else hipLaunchKernelGGL(fa::amax_kernel<fa::LoadF32>, grid, block, 0, s, x, n, parts, host_parts);
  if (hipGetLastError() != hipSuccess) return FA_ERR_LAUNCH;
  // the host waits for the first kernel only, while the second runs
  hipEvent_t known = nullptr;
  bool good = hipEventCreateWithFlags(&known, hipEventDisableTiming) == hipSuccess && hipEventRecord(known, s) == hipSuccess;
  if (good) {
    fa::launch_quantize(x, dtype, n, out, 0.f, parts, s);
    good = hipGetLastError() == hipSuccess && hipEventSynchronize(known) == hipSuccess;
  }
  if (known) (void)hipEventDestroy(known);
  if (!good) {
    (void)hipStreamSynchronize(s);  // the caller takes `host_parts` back
    return FA_ERR_LAUNCH;
  }
  uint32_t m = 0;
  for (int i = 0; i < FA_AMAX_PARTS; ++i) {
    uint32_t v;
    std::memcpy(&v, host_parts + i, sizeof(v));
    m = v > m ? v : m;
  }
  std::memcpy(amax, &m, sizeof(m));
  return FA_OK;
}
