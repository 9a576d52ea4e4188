// Shared definitions of the servelab_amd kernels (gfx950, 64-wide wavefronts).
//
// Every source is compiled twice: with -DSL_F32 the activation type is float
// (the true 32-bit path: nothing is rounded to fewer bits; products of many rows
// multiply their operands as exact sums of bfloat16 terms, gemm_f32_split.h),
// without it the activation type is bfloat16.  Accumulation, softmax, norms
// and rotation are float in both.
//
// Every extern "C" entry point returns nullptr on success or a static message
// that says which size it refuses; nothing here allocates device memory.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#if defined(SL_F32)
typedef float act_t;
#define SL_ACT_NAME "float32"
#else
typedef __bf16 act_t;
#define SL_ACT_NAME "bfloat16"
#endif

#define SL_WAVE 64

__device__ __forceinline__ float to_f(float x) { return x; }
__device__ __forceinline__ float to_f(__bf16 x) { return (float)x; }
template <typename T> __device__ __forceinline__ T from_f(float x);
template <> __device__ __forceinline__ float from_f<float>(float x) { return x; }
template <> __device__ __forceinline__ __bf16 from_f<__bf16>(float x) { return (__bf16)x; }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = SL_WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, SL_WAVE);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = SL_WAVE / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, SL_WAVE));
  return v;
}

// Sum over a block of up to 1024 threads; `scratch` holds 16 floats of LDS.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  v = wave_sum(v);
  const int wave = threadIdx.x / SL_WAVE, lane = threadIdx.x % SL_WAVE;
  const int nwaves = (blockDim.x + SL_WAVE - 1) / SL_WAVE;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nwaves; ++i) t += scratch[i];
  return t;
}

// Activations by number, as the calls of the kernel table pass them: 1 silu, 2 relu, 3 relu squared,
// 4 the tanh form of gelu; 5 only as a gate (sl_gated): clamped operands, a sigmoid of 1.702 g, up + 1.
enum { SL_ACT_SILU = 1, SL_ACT_RELU = 2, SL_ACT_RELU2 = 3, SL_ACT_GELU_TANH = 4, SL_ACT_CLAMPED_SWISH = 5 };
__device__ __forceinline__ float sl_act(float z, int act) {
  // (expf and a division, whose worst error over all floats is 2.7 units in the last place.  v_exp_f32 and v_rcp_f32 on a z that
  // is kept from infinity take 0.45 of the time, a wavefront's value 20 ns instead of 42, and are 3.7 off; with the quotient's
  // remainder put back as well it is 0.7 of the time and still a little further off on average.)
  if (act == SL_ACT_SILU) return z / (1.f + expf(-z));
  if (act == SL_ACT_GELU_TANH) return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
  const float r = fmaxf(z, 0.f);
  return act == SL_ACT_RELU2 ? r * r : r;
}
// A gate times its up product: act(g) * u; for the clamped form, with g' = min(g, limit) and
// u' = clamp(u, -limit, limit): g' sigmoid(1.702 g') (u' + 1).
__device__ __forceinline__ float sl_gated(float g, float u, int act, float limit) {
  if (act == SL_ACT_CLAMPED_SWISH) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g / (1.f + expf(-1.702f * g)) * (u + 1.f);
  }
  return sl_act(g, act) * u;
}

#define SL_CHECK(cond, msg) \
  do { if (!(cond)) return msg; } while (0)

static inline const char* sl_launch_status() {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? nullptr : hipGetErrorString(e);
}

// CUs of the current device (asked once per device).
static inline int device_cus() {
  static int cus[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cus[dev] == 0 &&
      hipDeviceGetAttribute(&cus[dev], hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
  return cus[dev];
}
