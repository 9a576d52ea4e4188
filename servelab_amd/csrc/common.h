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

// The value of lane ^ O, O = 1, 2, 4 or 8, by moves between the lanes of a row of 16 (register to register: 8 cycles, where an
// exchange through the LDS's crossbar takes about 130).  The source lanes have to be active.
template <int CTRL, int BANKS = 0xf> __device__ __forceinline__ int row_move(int old, int v) {
  return __builtin_amdgcn_update_dpp(old, v, CTRL, 0xf, BANKS, false);
}
template <int O> __device__ __forceinline__ float lane_xor(float v) {
  static_assert(O == 1 || O == 2 || O == 4 || O == 8, "within a row of 16 lanes");
  const int x = __float_as_int(v);
  if (O == 1) return __int_as_float(row_move<0xB1>(0, x));                 // quad_perm [1, 0, 3, 2]
  if (O == 2) return __int_as_float(row_move<0x4E>(0, x));                 // quad_perm [2, 3, 0, 1]
  if (O == 8) return __int_as_float(row_move<0x128>(0, x));                // rotated by 8
  return __int_as_float(row_move<0x114, 0xa>(row_move<0x104, 0x5>(0, x), x));   // quads 0, 2 from the next, 1, 3 from the one before
}
// op(v of this lane, v of lane ^ O) in both lanes, O = 16 or 32; op does not mind the order.  (After a swap of a register with
// itself one result holds the lower partner in every lane and the other the upper one.)
template <int O, class Op> __device__ __forceinline__ float rows_meet(float v, Op op) {
  static_assert(O == 16 || O == 32, "rows of 16 lanes, halves of the wavefront");
  const unsigned x = __float_as_uint(v);
  if (O == 32) {
    auto a = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return op(__uint_as_float(a[0]), __uint_as_float(a[1]));
  }
  auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  return op(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
// The value of lane + 32 in lanes 0 .. 31.
__device__ __forceinline__ float lane_and_32_on(float v) {
  const unsigned x = __float_as_uint(v);
  return __uint_as_float(__builtin_amdgcn_permlane32_swap(x, x, false, false)[1]);
}
__device__ __forceinline__ float add_f(float a, float b) { return a + b; }
__device__ __forceinline__ float max_f(float a, float b) { return fmaxf(a, b); }

// Over a wavefront whose lanes are all active, pairs 32, 16, 8, 4, 2, 1 apart in turn; every lane gets the result.  Six exchanges
// through the LDS's crossbar stood here, in a row: most of the time of a kernel of a few rows is such chains.
template <class Op> __device__ __forceinline__ float wave_meet(float v, Op op) {
  v = rows_meet<32>(v, op);
  v = rows_meet<16>(v, op);
  v = op(v, lane_xor<8>(v));
  v = op(v, lane_xor<4>(v));
  v = op(v, lane_xor<2>(v));
  return op(v, lane_xor<1>(v));
}
// Over the 16 lanes of a row (pairs 8, 4, 2, 1 apart), and over the four lanes l, l + 16, l + 32, l + 48 (16, then 32 apart).
template <class Op> __device__ __forceinline__ float row_meet(float v, Op op) {
  v = op(v, lane_xor<8>(v));
  v = op(v, lane_xor<4>(v));
  v = op(v, lane_xor<2>(v));
  return op(v, lane_xor<1>(v));
}
template <class Op> __device__ __forceinline__ float column_meet(float v, Op op) { return rows_meet<32>(rows_meet<16>(v, op), op); }
__device__ __forceinline__ float wave_sum(float v) { return wave_meet(v, add_f); }
__device__ __forceinline__ float wave_max(float v) { return wave_meet(v, max_f); }

// The sum over this lane and the ones before it, all lanes active: within rows of 16 by shifts of 1, 2, 4 and 8, then the last
// lanes of rows 0 and 2 to the rows behind them and lane 31 to the upper half.
__device__ __forceinline__ int sum_up_to(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
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
  const float part = scratch[lane & 15];               // (a lane a wavefront's sum: added up in a row they wait for one another)
  return row_meet((lane & 15) < nwaves ? part : 0.f, add_f);
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
