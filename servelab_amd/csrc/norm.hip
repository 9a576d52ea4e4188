// RMSNorm fused with the residual add that precedes it.
//   resid (float, in place) += delta;  out = resid * rsqrt(mean(resid^2) + eps) * w
// delta is a tensor in the activation dtype, or the float partial sums of a
// product whose K was split over workgroups (parts [nparts][T][H], optionally a
// bias [H]): the partial sums are then added here instead of by a kernel of
// their own.
// Formula and float32 math: servelab/attention/triton/paged_attention.py:76-91,
// tests/test_triton_kernels.py:57-59; the adds it absorbs are
// servelab/parallel/tp_model.py:131,133.  One block per row.
#include "common.h"

// rows == nullptr: row r of the stream, which is updated in place.
// rows != nullptr: row rows[r] of the stream (and of delta) is read, nothing
// but out[r] is written.
struct SplitDelta {
  const float* parts;            // [nparts][stride], or nullptr
  int nparts;
  size_t stride;                 // T * H
  const float* bias;             // [H] or nullptr
};

__global__ void add_rmsnorm_kernel(float* __restrict__ resid, const act_t* __restrict__ delta,
                                   const SplitDelta sd, const int* __restrict__ rows,
                                   const float* __restrict__ w, act_t* __restrict__ out, int H,
                                   float eps) {
  __shared__ float scratch[16];
  const int r = blockIdx.x;
  const size_t src = rows != nullptr ? (size_t)rows[r] : (size_t)r;
  float* x = resid + src * H;
  const act_t* d = delta != nullptr ? delta + src * H : nullptr;
  const float* p = sd.parts != nullptr ? sd.parts + src * H : nullptr;
  const bool adds = d != nullptr || p != nullptr;
  auto delta_at = [&](int i) {
    float v = d != nullptr ? to_f(d[i]) : 0.f;
    if (p != nullptr) {
      for (int j = 0; j < sd.nparts; ++j) v += p[j * sd.stride + i];
      if (sd.bias != nullptr) v += sd.bias[i];
    }
    return v;
  };
  float ss = 0.f;
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    float v = x[i];
    if (adds) {
      v += delta_at(i);
      if (rows == nullptr) x[i] = v;
    }
    ss += v * v;
  }
  ss = block_sum(ss, scratch);
  const float inv = rsqrtf(ss / (float)H + eps);
  act_t* o = out + (size_t)r * H;
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    float v = x[i];
    if (adds && rows != nullptr) v += delta_at(i);
    o[i] = from_f<act_t>(v * inv * w[i]);
  }
}

// The same for rows of up to 4 * 8 * blockDim values that are a multiple of 4
// wide: every value is read once with 16-byte loads and kept in registers
// between the sum of squares and the scaling.
struct __attribute__((aligned(16))) f4 { float v[4]; };
#if defined(SL_F32)
struct __attribute__((aligned(16))) a4 { act_t v[4]; };
#else
struct __attribute__((aligned(8))) a4 { act_t v[4]; };
#endif

// The most threads of a workgroup whose threads have ITERS groups of four values each (``row_threads``).  Eight groups, more than 256 rows of more
// than 8,192 values: no more than 512 threads share the register file, and the gains are asked for behind the sums, so that two workgroups fit a CU
// (2,048 rows of 10,240 values, us: two partial sums 94 with room for 1,024 threads and gains in registers, which spilled, now 65; layer norm 50, now 41; of
// 16,384 values, layer norm 111, now 69; float32 181, now 93).
constexpr int row_most(int iters) { return iters > 4 ? 512 : 1024; }

// A step of few rows is one trip to memory and one sum, so all that a row needs is asked for at once, PARTS partial sums a trip (0: a
// delta instead, -1: neither), and no load stands behind a condition, which would be waited for where the ways meet; the stream's new row is written behind the sum.  64 rows of 3,584 values
// with eight partial sums: 5.2 us with the loads in turn, 4.9 here, 2,048 with two: 23.0, now 22.5.
template <int ITERS, int PARTS>
__global__ __launch_bounds__(row_most(ITERS), 4) void add_rmsnorm_vec_kernel(float* __restrict__ resid, const act_t* __restrict__ delta,
                                       const SplitDelta sd, const int* __restrict__ rows,
                                       const float* __restrict__ w, act_t* __restrict__ out, int H,
                                       float eps) {
  __shared__ float scratch[16];
  const int r = blockIdx.x;
  const size_t src = rows != nullptr ? (size_t)rows[r] : (size_t)r;
  float* x = resid + src * H;
  const bool plain = delta != nullptr;
  const act_t* d = delta + src * H;
  const float* p = sd.parts + src * H;
  const int H4 = H / 4;
  f4 v[ITERS], wv[ITERS], pv[PARTS > 0 ? PARTS : 1][ITERS];
  a4 dv[ITERS];
  auto group = [&](int it) { return min((int)(threadIdx.x + it * blockDim.x), H4 - 1); };
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    v[it] = ((const f4*)x)[group(it)];
    if (PARTS == 0) dv[it] = ((const a4*)d)[group(it)];
    if (ITERS <= 4) wv[it] = ((const f4*)w)[group(it)];
  }
  auto ask = [&](int q0) {
#pragma unroll
    for (int q = 0; q < PARTS; ++q)
#pragma unroll
      for (int it = 0; it < ITERS; ++it) pv[q][it] = ((const f4*)(p + min(q0 + q, sd.nparts - 1) * sd.stride))[group(it)];
  };
  auto add = [&](int q0) {
#pragma unroll
    for (int q = 0; q < PARTS; ++q)
#pragma unroll
      for (int it = 0; it < ITERS; ++it)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[it].v[j] += q0 + q < sd.nparts ? pv[q][it].v[j] : 0.f;
  };
  ask(0);
  if (PARTS > 0 && plain)                              // (rare beside partial sums, as a bias is)
#pragma unroll
    for (int it = 0; it < ITERS; ++it) dv[it] = ((const a4*)d)[group(it)];
#pragma unroll
  for (int it = 0; it < ITERS; ++it)
#pragma unroll
    for (int j = 0; j < 4; ++j) v[it].v[j] += PARTS == 0 || (PARTS > 0 && plain) ? to_f(dv[it].v[j]) : 0.f;
  add(0);
  if (PARTS > 0) {
    for (int q0 = PARTS; q0 < sd.nparts; q0 += PARTS) {
      ask(q0);
      add(q0);
    }
    if (sd.bias != nullptr)
#pragma unroll
      for (int it = 0; it < ITERS; ++it) {
        const f4 bv = ((const f4*)sd.bias)[group(it)];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[it].v[j] += bv.v[j];
      }
  }
  float ss = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it)
#pragma unroll
    for (int j = 0; j < 4; ++j) ss += threadIdx.x + it * blockDim.x < H4 ? v[it].v[j] * v[it].v[j] : 0.f;
  ss = block_sum(ss, scratch);
  const float inv = rsqrtf(ss / (float)H + eps);
  act_t* o = out + (size_t)r * H;
  const bool store = PARTS >= 0 && rows == nullptr;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int i = threadIdx.x + it * blockDim.x;
    if (i < H4) {
      a4 ov;
      if (ITERS > 4) wv[it] = ((const f4*)w)[i];
#pragma unroll
      for (int j = 0; j < 4; ++j) ov.v[j] = from_f<act_t>(v[it].v[j] * inv * wv[it].v[j]);
      if (store) ((f4*)x)[i] = v[it];
      ((a4*)o)[i] = ov;
    }
  }
}

// Rows of n groups of four values (n up to 8 * 512): a workgroup's threads.  A group a thread is the shortest chain, and what a few rows
// want (8 rows of 3,584 values with their output's norm: 896 threads 2.85 us, 512 with two groups each 3.4 before); with more rows than
// CUs the waits of one cover another's, and workgroups stay at 512 as they were.
static int row_threads(int R, int n) {
  const int most = R <= 256 ? 1024 : 512, turns = (n + most - 1) / most;
  return ((n + turns - 1) / turns + 63) / 64 * 64;
}
// Calls f with the number of groups a thread has in a kernel for it (a group that no thread of a workgroup has is read all the same: 700 rows of
// 5,120 values, three groups, 8.1 us in the kernel for four, 7.3 in one for three; 257 rows with eight partial sums 12.5 and 11.9).
template <int N> struct Groups { static constexpr int n = N; };
template <class F> static void with_groups(int n, F f) {
  if (n <= 1) f(Groups<1>{});
  else if (n == 2) f(Groups<2>{});
  else if (n == 3) f(Groups<3>{});
  else if (n == 4) f(Groups<4>{});
  else if (n <= 6) f(Groups<6>{});
  else f(Groups<8>{});
}

// parts != nullptr: nparts float partial sums [nparts][T][H] (T rows in each)
// and an optional bias [H] are the delta (or are added to it).
extern "C" const char* sl_add_rmsnorm(float* resid, const void* delta, const float* parts,
                                      int nparts, int T, const float* bias, const int* rows,
                                      const float* w, void* out, int R, int H, float eps,
                                      hipStream_t stream) {
  SL_CHECK(R >= 0 && H > 0, "add_rmsnorm: sizes must be positive");
  SL_CHECK(parts == nullptr || (nparts >= 1 && T >= 1), "add_rmsnorm: partial sums need their counts");
  SL_CHECK(parts != nullptr || bias == nullptr, "add_rmsnorm: a bias comes with partial sums only");
  if (R == 0) return nullptr;
  const SplitDelta sd{parts, nparts, (size_t)T * H, bias};
  const bool aligned = ((uintptr_t)resid % 16) == 0 && ((uintptr_t)out % sizeof(a4)) == 0 &&
                       ((uintptr_t)delta % sizeof(a4)) == 0 && ((uintptr_t)parts % 16) == 0 &&
                       ((uintptr_t)bias % 16) == 0 && ((uintptr_t)w % 16) == 0;
  if (H % 4 == 0 && H <= 4 * 8 * 512 && aligned) {
    const int H4 = H / 4, threads = row_threads(R, H4), iters = (H4 + threads - 1) / threads;
    const act_t* dl = (const act_t*)delta;
    act_t* o = (act_t*)out;
    auto run = [&](auto kernel) { kernel<<<R, threads, 0, stream>>>(resid, dl, sd, rows, w, o, H, eps); };
    // (as many partial sums a trip as there are: reading one again in place of one that is not there costs many rows what it saves few)
    with_groups(iters, [&](auto groups) {
      constexpr int N = decltype(groups)::n;
      if (parts == nullptr && delta == nullptr) run(add_rmsnorm_vec_kernel<N, -1>);
      else if (parts == nullptr) run(add_rmsnorm_vec_kernel<N, 0>);
      else if constexpr (N > 4) run(add_rmsnorm_vec_kernel<N, 1>);
      else if (N > 2 || nparts <= 2) run(add_rmsnorm_vec_kernel<N, 2>);
      else if constexpr (N <= 2) {
        if (nparts == 3) run(add_rmsnorm_vec_kernel<N, 3>);
        else if (N == 2 || nparts == 4) run(add_rmsnorm_vec_kernel<N, 4>);
        else run(add_rmsnorm_vec_kernel<N, 8>);
      }
    });
    return sl_launch_status();
  }
  const int threads = H >= 2048 ? 512 : 256;
  add_rmsnorm_kernel<<<R, threads, 0, stream>>>(resid, (const act_t*)delta, sd, rows, w,
                                                (act_t*)out, H, eps);
  return sl_launch_status();
}

// Layer norm with a gain and (bias given) a bias, fused with the residual add that precedes it:
//   resid (float, in place) += d1 + d2;  out = (resid - mean) / sqrt(var + eps) * w + bias
// where var is the mean of the squared deviations.  Either delta may be absent.
// rows as above: with rows the stream is only read.  One block per row; the
// row is read three times (sum, squared deviations, output), from cache after
// the first.
__global__ void add_layernorm_kernel(float* __restrict__ resid, const act_t* __restrict__ d1,
                                     const act_t* __restrict__ d2, const int* __restrict__ rows,
                                     const float* __restrict__ w, const float* __restrict__ bias,
                                     act_t* __restrict__ out, int H, float eps) {
  __shared__ float scratch[16];
  const int r = blockIdx.x;
  const size_t src = rows != nullptr ? (size_t)rows[r] : (size_t)r;
  float* x = resid + src * H;
  const act_t* a = d1 != nullptr ? d1 + src * H : nullptr;
  const act_t* b = d2 != nullptr ? d2 + src * H : nullptr;
  const bool adds = a != nullptr || b != nullptr;
  const bool again = adds && rows != nullptr;        // the sum is not stored: form it on every pass
  auto value = [&](int i) {
    float d = 0.f;
    if (a != nullptr) d = to_f(a[i]);
    if (b != nullptr) d += to_f(b[i]);
    return x[i] + d;
  };
  float sum = 0.f;
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    float v = x[i];
    if (adds) {
      v = value(i);
      if (rows == nullptr) x[i] = v;
    }
    sum += v;
  }
  const float mean = block_sum(sum, scratch) / (float)H;
  float sq = 0.f;
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    const float dv = (again ? value(i) : x[i]) - mean;
    sq += dv * dv;
  }
  const float inv = 1.f / sqrtf(block_sum(sq, scratch) / (float)H + eps);
  act_t* o = out + (size_t)r * H;
  for (int i = threadIdx.x; i < H; i += blockDim.x)
    o[i] = from_f<act_t>(((again ? value(i) : x[i]) - mean) * inv * w[i] + (bias != nullptr ? bias[i] : 0.f));
}

// The same for rows of up to 4 * 8 * blockDim values that are a multiple of 4 wide: every value
// is read once with 16-byte loads and stays in registers for the mean, the squared deviations
// and the output.
// All of it is asked for at once, as above, and the stream's new row is written behind the sums (4 rows of 2,048 values: 2.8 us before, 2.5 here).
// A kernel for each number of deltas: one that is not there is no row read in its place (us, loads in turn / the stream's row in that place / here: without
// a delta 300 rows of 8,192 values 5.4 / 6.2 / 5.1, 1,000 of 4,096 5.7 / 6.8 / 5.8; with one 7.7 / 8.4 / 6.9 and 8.1 / 8.9 / 8.1).
template <int ITERS, int DELTAS>
__global__ __launch_bounds__(row_most(ITERS)) void add_layernorm_vec_kernel(float* __restrict__ resid, const act_t* __restrict__ d1,
                                         const act_t* __restrict__ d2, const int* __restrict__ rows,
                                         const float* __restrict__ w, const float* __restrict__ bias,
                                         act_t* __restrict__ out, int H, float eps) {
  __shared__ float scratch[16];
  const int r = blockIdx.x;
  const size_t src = rows != nullptr ? (size_t)rows[r] : (size_t)r;
  float* x = resid + src * H;
  const act_t *a = d1 + src * H, *b = d2 + src * H;
  const float* add = bias != nullptr ? bias : w;
  const int H4 = H / 4;
  f4 v[ITERS], wv[ITERS], bv[ITERS];
  a4 av[ITERS], cv[ITERS];
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int i = min((int)(threadIdx.x + it * blockDim.x), H4 - 1);
    v[it] = ((const f4*)x)[i];
    if (DELTAS > 0) av[it] = ((const a4*)a)[i];
    if (DELTAS > 1) cv[it] = ((const a4*)b)[i];
    if (ITERS <= 4) {
      wv[it] = ((const f4*)w)[i];
      bv[it] = ((const f4*)add)[i];
    }
  }
  float sum = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const bool in = threadIdx.x + it * blockDim.x < H4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (DELTAS > 0) v[it].v[j] += DELTAS > 1 ? to_f(av[it].v[j]) + to_f(cv[it].v[j]) : to_f(av[it].v[j]);
      sum += in ? v[it].v[j] : 0.f;
    }
  }
  const float mean = block_sum(sum, scratch) / (float)H;
  float sq = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const bool in = threadIdx.x + it * blockDim.x < H4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float dv = v[it].v[j] - mean;
      sq += in ? dv * dv : 0.f;
    }
  }
  const float inv = 1.f / sqrtf(block_sum(sq, scratch) / (float)H + eps);
  act_t* o = out + (size_t)r * H;
  const bool store = DELTAS > 0 && rows == nullptr;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int i = threadIdx.x + it * blockDim.x;
    if (i < H4) {
      a4 ov;
      if (ITERS > 4) {
        wv[it] = ((const f4*)w)[i];
        bv[it] = ((const f4*)add)[i];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        ov.v[j] = from_f<act_t>((v[it].v[j] - mean) * inv * wv[it].v[j] + (bias != nullptr ? bv[it].v[j] : 0.f));
      if (store) ((f4*)x)[i] = v[it];
      ((a4*)o)[i] = ov;
    }
  }
}

extern "C" const char* sl_add_layernorm(float* resid, const void* d1, const void* d2, const int* rows,
                                        const float* w, const float* bias, void* out, int R, int H, float eps,
                                        hipStream_t stream) {
  SL_CHECK(R >= 0 && H > 0, "add_layernorm: sizes must be positive");
  if (R == 0) return nullptr;
  const bool aligned = ((uintptr_t)resid % 16) == 0 && ((uintptr_t)out % sizeof(a4)) == 0 &&
                       ((uintptr_t)d1 % sizeof(a4)) == 0 && ((uintptr_t)d2 % sizeof(a4)) == 0 &&
                       ((uintptr_t)w % 16) == 0 && ((uintptr_t)bias % 16) == 0;
  if (H % 4 == 0 && H <= 4 * 8 * 512 && aligned) {
    const int H4 = H / 4, nthreads = row_threads(R, H4), iters = (H4 + nthreads - 1) / nthreads;
    const act_t* a = (const act_t*)(d1 != nullptr ? d1 : d2);
    const act_t* b = (const act_t*)d2;
    act_t* o = (act_t*)out;
    with_groups(iters, [&](auto groups) {
      constexpr int N = decltype(groups)::n;
      auto run = [&](auto kernel) { kernel<<<R, nthreads, 0, stream>>>(resid, a, b, rows, w, bias, o, H, eps); };
      if (a == nullptr) run(add_layernorm_vec_kernel<N, 0>);
      else if (d1 == nullptr || d2 == nullptr) run(add_layernorm_vec_kernel<N, 1>);
      else run(add_layernorm_vec_kernel<N, 2>);
    });
    return sl_launch_status();
  }
  const int threads = H >= 2048 ? 512 : 256;
  add_layernorm_kernel<<<R, threads, 0, stream>>>(resid, (const act_t*)d1, (const act_t*)d2, rows, w, bias,
                                                  (act_t*)out, H, eps);
  return sl_launch_status();
}

// The norm before a sublayer over a stream kept in copies x_1 .. x_S (float, [T][S][H]), after the output of
// the sublayer before has been written to them:
//   y = y1 + y2 (each first divided by its root mean square and multiplied by its gain, where it has one)
//   x_t <- sum_s mix[s][t] x_s + out[t] y, all copies at once from the old ones, in place
//   u = sum_s read[s] x_s (read == nullptr: the plain sum)
//   o = (u - mean) / sqrt(var + eps) * w + bias (not center: u / sqrt(mean(u^2) + eps) * w + bias)
// y1 == nullptr: nothing is written.  rows given: only the listed rows are computed and the copies stay as
// they are.  One block per row; a thread's channels are its own in every copy, so the copies are read
// and rewritten without a barrier; u stays in registers until the norm's sums are known.
struct StreamsNorm {
  float* x;
  int S;
  const act_t *y1, *y2;
  const float *g1, *g2;
  float e1, e2;
  const float *mix, *out, *read;
  const int* rows;
  const float *w, *bias;
  float eps;
  int center;
  act_t* o;
  int H;
};

__device__ __forceinline__ float inv_rms(const act_t* __restrict__ y, int H, float eps, float* scratch) {
  float ss = 0.f;
  for (int i = threadIdx.x; i < H; i += blockDim.x) {
    const float v = to_f(y[i]);
    ss += v * v;
  }
  return 1.f / sqrtf(block_sum(ss, scratch) / (float)H + eps);
}

// MAXS: the copies, exactly (EXACT) or at most.  VEC channels at a time; up to ITERS such groups a thread
// keep their u in registers (ITERS 0: any width, u waits in LDS).
template <int MAXS, bool EXACT, int VEC, int ITERS>
__global__ void streams_norm_kernel(const StreamsNorm a) {
  __shared__ float scratch[16];
  extern __shared__ float u_lds[];
  struct __attribute__((aligned(4 * VEC))) fv { float v[VEC]; };
  struct __attribute__((aligned(sizeof(act_t) * VEC))) av { act_t v[VEC]; };
  const int S = EXACT ? MAXS : a.S, H = a.H, HV = H / VEC;
  const size_t r = a.rows != nullptr ? (size_t)a.rows[blockIdx.x] : (size_t)blockIdx.x;
  float* x = a.x + r * S * H;
  const act_t* y1 = a.y1 != nullptr ? a.y1 + r * H : nullptr;
  const act_t* y2 = a.y2 != nullptr ? a.y2 + r * H : nullptr;
  const float i1 = a.g1 != nullptr ? inv_rms(y1, H, a.e1, scratch) : 1.f;
  const float i2 = a.g2 != nullptr ? inv_rms(y2, H, a.e2, scratch) : 1.f;
  const bool writes = y1 != nullptr, store = a.rows == nullptr;
  // (the copies' weights stand in registers where their number is known: behind a store to the stream they would be
  // read again: one row of four copies of 2,048 values 3.8 us, now 3.0, with two normed outputs 6.1, now 4.9)
  float rd[MAXS], ot[MAXS], mx[EXACT ? MAXS : 1][EXACT ? MAXS : 1];
  if constexpr (EXACT) {
#pragma unroll
    for (int t = 0; t < MAXS; ++t) {
      rd[t] = a.read != nullptr ? a.read[t] : 1.f;
      ot[t] = writes ? a.out[t] : 0.f;
#pragma unroll
      for (int s = 0; s < MAXS; ++s) mx[s][t] = writes ? a.mix[s * MAXS + t] : 0.f;
    }
  }
  auto reads = [&](int t) { return EXACT ? rd[t] : a.read != nullptr ? a.read[t] : 1.f; };
  auto group = [&](int at) -> fv {
    const int i = min(at, HV - 1);
    const bool keeps = store && at < HV;
    fv xs[MAXS], u;
#pragma unroll
    for (int s = 0; s < MAXS; ++s)
      if (EXACT || s < S) xs[s] = *(const fv*)(x + (size_t)s * H + (size_t)i * VEC);
#pragma unroll
    for (int c = 0; c < VEC; ++c) u.v[c] = 0.f;
    if (!writes) {
#pragma unroll
      for (int s = 0; s < MAXS; ++s)
        if (EXACT || s < S) {
          const float f = reads(s);
#pragma unroll
          for (int c = 0; c < VEC; ++c) u.v[c] += f * xs[s].v[c];
        }
      return u;
    }
    fv y;
    {
      const av p = *(const av*)(y1 + (size_t)i * VEC);
      fv g;
      if (a.g1 != nullptr) g = *(const fv*)(a.g1 + (size_t)i * VEC);
#pragma unroll
      for (int c = 0; c < VEC; ++c) y.v[c] = a.g1 != nullptr ? to_f(p.v[c]) * i1 * g.v[c] : to_f(p.v[c]);
    }
    if (y2 != nullptr) {
      const av p = *(const av*)(y2 + (size_t)i * VEC);
      fv g;
      if (a.g2 != nullptr) g = *(const fv*)(a.g2 + (size_t)i * VEC);
#pragma unroll
      for (int c = 0; c < VEC; ++c) y.v[c] += a.g2 != nullptr ? to_f(p.v[c]) * i2 * g.v[c] : to_f(p.v[c]);
    }
#pragma unroll
    for (int t = 0; t < MAXS; ++t)
      if (EXACT || t < S) {
        const float f = reads(t), o1 = EXACT ? ot[t] : a.out[t];
        fv n;
#pragma unroll
        for (int c = 0; c < VEC; ++c) n.v[c] = o1 * y.v[c];
#pragma unroll
        for (int s = 0; s < MAXS; ++s)
          if (EXACT || s < S) {
            const float m = EXACT ? mx[EXACT ? s : 0][EXACT ? t : 0] : a.mix[s * S + t];
#pragma unroll
            for (int c = 0; c < VEC; ++c) n.v[c] += m * xs[s].v[c];
          }
        if (keeps) *(fv*)(x + (size_t)t * H + (size_t)i * VEC) = n;
#pragma unroll
        for (int c = 0; c < VEC; ++c) u.v[c] += f * n.v[c];
      }
    return u;
  };
  constexpr int KEEP = ITERS > 0 ? ITERS : 1;
  fv keep[KEEP];
  float sum = 0.f;
  if constexpr (ITERS > 0) {
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int i = threadIdx.x + it * blockDim.x;
      keep[it] = group(i);
#pragma unroll
      for (int c = 0; c < VEC; ++c) sum += i < HV ? keep[it].v[c] : 0.f;
    }
  } else {
    for (int i = threadIdx.x; i < HV; i += blockDim.x) {      // (VEC 1)
      u_lds[i] = group(i).v[0];
      sum += u_lds[i];
    }
  }
  const float mean = a.center ? block_sum(sum, scratch) / (float)H : 0.f;
  float sq = 0.f;
  if constexpr (ITERS > 0) {
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int i = threadIdx.x + it * blockDim.x;
      if (i < HV) {
#pragma unroll
        for (int c = 0; c < VEC; ++c) {
          keep[it].v[c] -= mean;
          sq += keep[it].v[c] * keep[it].v[c];
        }
      }
    }
  } else {
    for (int i = threadIdx.x; i < HV; i += blockDim.x) {
      const float d = u_lds[i] - mean;
      sq += d * d;
    }
  }
  const float inv = 1.f / sqrtf(block_sum(sq, scratch) / (float)H + a.eps);
  act_t* o = a.o + (size_t)blockIdx.x * H;
  if constexpr (ITERS > 0) {
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
      const int i = threadIdx.x + it * blockDim.x;
      if (i < HV) {
        const fv wv = *(const fv*)(a.w + (size_t)i * VEC);
        fv bv;
#pragma unroll
        for (int c = 0; c < VEC; ++c) bv.v[c] = 0.f;
        if (a.bias != nullptr) bv = *(const fv*)(a.bias + (size_t)i * VEC);
        av ov;
#pragma unroll
        for (int c = 0; c < VEC; ++c) ov.v[c] = from_f<act_t>(keep[it].v[c] * inv * wv.v[c] + bv.v[c]);
        *(av*)(o + (size_t)i * VEC) = ov;
      }
    }
  } else {
    for (int i = threadIdx.x; i < HV; i += blockDim.x)
      o[i] = from_f<act_t>((u_lds[i] - mean) * inv * a.w[i] + (a.bias != nullptr ? a.bias[i] : 0.f));
  }
}

template <int MAXS, bool EXACT>
static const char* launch_streams_norm(const StreamsNorm& a, int R, hipStream_t stream) {
  const uintptr_t f32s = (uintptr_t)a.x | (uintptr_t)a.g1 | (uintptr_t)a.g2 | (uintptr_t)a.w | (uintptr_t)a.bias;
  const uintptr_t acts = (uintptr_t)a.y1 | (uintptr_t)a.y2 | (uintptr_t)a.o;
  if (a.H % 4 == 0 && a.H <= 4 * 8 * 512 && f32s % 16 == 0 && acts % (4 * sizeof(act_t)) == 0) {
    const int H4 = a.H / 4, threads = row_threads(R, H4), iters = (H4 + threads - 1) / threads;
    with_groups(iters, [&](auto groups) { streams_norm_kernel<MAXS, EXACT, 4, decltype(groups)::n><<<R, threads, 0, stream>>>(a); });
    return sl_launch_status();
  }
  SL_CHECK(a.H <= 12288, "streams_norm: rows of odd width hold at most 12,288 values");
  streams_norm_kernel<MAXS, EXACT, 1, 0><<<R, a.H >= 2048 ? 512 : 256, a.H * sizeof(float), stream>>>(a);
  return sl_launch_status();
}

extern "C" const char* sl_streams_norm(float* x, int S, const void* y1, const float* g1, float e1, const void* y2,
                                       const float* g2, float e2, const float* mix, const float* out,
                                       const float* read, const int* rows, const float* w, const float* bias,
                                       float eps, int center, void* o, int R, int H, hipStream_t stream) {
  SL_CHECK(R >= 0 && H > 0 && S >= 1 && S <= 16, "streams_norm: sizes must be positive, at most 16 copies");
  SL_CHECK(x != nullptr && w != nullptr && o != nullptr, "streams_norm: the stream, the gain and the result are required");
  SL_CHECK(y1 == nullptr || (mix != nullptr && out != nullptr), "streams_norm: an output needs mix and out");
  SL_CHECK((y1 != nullptr || (y2 == nullptr && g1 == nullptr)) && (y2 != nullptr || g2 == nullptr),
           "streams_norm: a gain comes with its output, the second output with the first");
  if (R == 0) return nullptr;
  const StreamsNorm a{x, S, (const act_t*)y1, (const act_t*)y2, g1, g2, e1, e2, mix, out, read, rows, w, bias, eps,
                      center, (act_t*)o, H};
  if (S == 1) return launch_streams_norm<1, true>(a, R, stream);
  if (S == 2) return launch_streams_norm<2, true>(a, R, stream);
  if (S == 3) return launch_streams_norm<3, true>(a, R, stream);
  if (S == 4) return launch_streams_norm<4, true>(a, R, stream);
  if (S <= 8) return launch_streams_norm<8, false>(a, R, stream);
  return launch_streams_norm<16, false>(a, R, stream);
}

// resid (float, in place) += delta: for a delta that a norm cannot take with its own add.
__global__ void add_into_kernel(float* __restrict__ resid, const act_t* __restrict__ delta, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) resid[i] += to_f(delta[i]);
}

extern "C" const char* sl_add_into(float* resid, const void* delta, long long n, hipStream_t stream) {
  SL_CHECK(n >= 0, "add_into: the count must not be negative");
  if (n == 0) return nullptr;
  add_into_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(resid, (const act_t*)delta, (size_t)n);
  return sl_launch_status();
}

// RMS norm on a sublayer's output: resid (float, in place) += mult * y * rsqrt(mean(y^2) + eps) * w,
// and the stream's new rows in the activation type for the sublayer that reads them next (out == nullptr:
// they are not wanted).  y == nullptr: only those rows.  One block per row; sums and the stream in float.
// A row is a few trips to memory in turn, so up to KEEP (1, 2, 4 or 8: what a row needs) values a thread of all that is read are
// asked for at once, before the sum, and no load stands behind a condition, which would be waited for where the ways meet (8
// rows of 3,584 values: 6.4 us with a loop after the sum, 4.7 here; 2,048 rows of 64: 3.4 us, 4.6 with eight loads, 3.3 here).
template <int KEEP>
__global__ void add_postnorm_kernel(float* __restrict__ resid, const act_t* __restrict__ y,
                                    const float* __restrict__ w, act_t* __restrict__ out, int H, float eps,
                                    float mult) {
  __shared__ float scratch[16];
  const size_t r = blockIdx.x;
  float* x = resid + r * H;
  act_t* o = out != nullptr ? out + r * H : nullptr;
  if (y == nullptr) {
    for (int i = threadIdx.x; i < H; i += blockDim.x) o[i] = from_f<act_t>(x[i]);
    return;
  }
  const act_t* yr = y + r * H;
  act_t yk[KEEP];
  float xk[KEEP], wk[KEEP];
#pragma unroll
  for (int u = 0; u < KEEP; ++u) {
    const int i = min((int)(threadIdx.x + u * blockDim.x), H - 1);
    yk[u] = yr[i];
    xk[u] = x[i];
    wk[u] = w[i];
  }
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < KEEP; ++u) {
    const float v = threadIdx.x + u * blockDim.x < H ? to_f(yk[u]) : 0.f;
    ss += v * v;
  }
  for (int i = threadIdx.x + KEEP * blockDim.x; i < H; i += blockDim.x) {
    const float v = to_f(yr[i]);
    ss += v * v;
  }
  ss = block_sum(ss, scratch);
  const float inv = 1.f / sqrtf(ss / (float)H + eps);
#pragma unroll
  for (int u = 0; u < KEEP; ++u) {
    const int i = threadIdx.x + u * blockDim.x;
    if (i >= H) break;
    const float v = xk[u] + mult * (to_f(yk[u]) * inv * wk[u]);
    x[i] = v;
    if (o != nullptr) o[i] = from_f<act_t>(v);
  }
  for (int i = threadIdx.x + KEEP * blockDim.x; i < H; i += blockDim.x) {
    const float v = x[i] + mult * (to_f(yr[i]) * inv * w[i]);
    x[i] = v;
    if (o != nullptr) o[i] = from_f<act_t>(v);
  }
}

// The same for rows of up to 4 * 8 * 512 values that are a multiple of 4 wide, 16-byte loads (8 rows of 3,584 values: 2.5 us with single
// ones, 2.1 here; one of 2,048 2.1, now 1.7).
template <int ITERS>
__global__ __launch_bounds__(row_most(ITERS)) void add_postnorm_vec_kernel(float* __restrict__ resid, const act_t* __restrict__ y,
                                                                const float* __restrict__ w, act_t* __restrict__ out, int H, float eps,
                                                                float mult) {
  __shared__ float scratch[16];
  const size_t r = blockIdx.x;
  float* x = resid + r * H;
  const int H4 = H / 4;
  f4 v[ITERS], wv[ITERS];
  a4 yv[ITERS];
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int i = min((int)(threadIdx.x + it * blockDim.x), H4 - 1);
    yv[it] = ((const a4*)(y + r * H))[i];
    v[it] = ((const f4*)x)[i];
    wv[it] = ((const f4*)w)[i];
  }
  float ss = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float n = threadIdx.x + it * blockDim.x < H4 ? to_f(yv[it].v[j]) : 0.f;
      ss += n * n;
    }
  const float inv = 1.f / sqrtf(block_sum(ss, scratch) / (float)H + eps);
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int i = threadIdx.x + it * blockDim.x;
    if (i < H4) {
      a4 ov;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[it].v[j] += mult * (to_f(yv[it].v[j]) * inv * wv[it].v[j]);
        ov.v[j] = from_f<act_t>(v[it].v[j]);
      }
      ((f4*)x)[i] = v[it];
      if (out != nullptr) ((a4*)(out + r * H))[i] = ov;
    }
  }
}

extern "C" const char* sl_add_postnorm(float* resid, const void* y, const float* w, void* out, int T, int H,
                                       float eps, float mult, hipStream_t stream) {
  SL_CHECK(T >= 0 && H > 0, "add_postnorm: sizes must be positive");
  SL_CHECK(y != nullptr || out != nullptr, "add_postnorm: nothing to do");
  if (T == 0) return nullptr;
  if (y != nullptr && H % 4 == 0 && H <= 4 * 8 * 512 && ((uintptr_t)resid | (uintptr_t)w) % 16 == 0 &&
      ((uintptr_t)y | (uintptr_t)out) % sizeof(a4) == 0) {
    const int H4 = H / 4, n = row_threads(T, H4), iters = (H4 + n - 1) / n;
    auto run = [&](auto kernel) { kernel<<<T, n, 0, stream>>>(resid, (const act_t*)y, w, (act_t*)out, H, eps, mult); };
    with_groups(iters, [&](auto groups) { run(add_postnorm_vec_kernel<decltype(groups)::n>); });
    return sl_launch_status();
  }
  const int threads = H >= 2048 ? 512 : 256, need = (H + threads - 1) / threads;
  auto run = [&](auto kernel) { kernel<<<T, threads, 0, stream>>>(resid, (const act_t*)y, w, (act_t*)out, H, eps, mult); };
  if (need <= 1) run(add_postnorm_kernel<1>);
  else if (need <= 2) run(add_postnorm_kernel<2>);
  else if (need <= 4) run(add_postnorm_kernel<4>);
  else run(add_postnorm_kernel<8>);
  return sl_launch_status();
}

// A sublayer's output joins the stream through a norm of its own, and the next sublayer's input norm
// follows at once: v = resid + y * rsqrt(mean(y^2) + eps_y) * wy, out = v * rsqrt(mean(v^2) + eps) * w.
// rows == nullptr: every row, and v goes back to the stream; else only the listed rows are computed
// and the stream stays as it is (the head reads few rows of the last layer's result).  One block per
// row, up to KEEP values a thread asked for at once, as above, and kept in registers between the passes; all
// sums in float (2 rows of 2,048 values: 6.0 us with loads after each sum, 4.4 here).
template <int KEEP>
__global__ void add_normed_rmsnorm_kernel(float* __restrict__ resid, const act_t* __restrict__ y,
                                          const float* __restrict__ wy, float eps_y,
                                          const int* __restrict__ rows, const float* __restrict__ w, float eps,
                                          act_t* __restrict__ out, int H) {
  __shared__ float scratch[16];
  const size_t r = rows != nullptr ? (size_t)rows[blockIdx.x] : (size_t)blockIdx.x;
  float* x = resid + r * H;
  const act_t* yr = y + r * H;
  act_t* o = out + (size_t)blockIdx.x * H;
  act_t yk[KEEP];
  float keep[KEEP], xk[KEEP], wyk[KEEP], wk[KEEP];
#pragma unroll
  for (int u = 0; u < KEEP; ++u) {
    const int i = min((int)(threadIdx.x + u * blockDim.x), H - 1);
    yk[u] = yr[i];
    xk[u] = x[i];
    wyk[u] = wy[i];
    wk[u] = w[i];
  }
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < KEEP; ++u) {
    keep[u] = threadIdx.x + u * blockDim.x < H ? to_f(yk[u]) : 0.f;
    ss += keep[u] * keep[u];
  }
  for (int i = threadIdx.x + KEEP * blockDim.x; i < H; i += blockDim.x) {
    const float v = to_f(yr[i]);
    ss += v * v;
  }
  ss = block_sum(ss, scratch);
  const float inv_y = 1.f / sqrtf(ss / (float)H + eps_y);
  float s2 = 0.f;
#pragma unroll
  for (int u = 0; u < KEEP; ++u) {
    const int i = threadIdx.x + u * blockDim.x;
    if (i < H) {
      keep[u] = xk[u] + keep[u] * inv_y * wyk[u];
      if (rows == nullptr) x[i] = keep[u];
      s2 += keep[u] * keep[u];
    }
  }
  for (int i = threadIdx.x + KEEP * blockDim.x; i < H; i += blockDim.x) {
    const float v = x[i] + to_f(yr[i]) * inv_y * wy[i];
    if (rows == nullptr) x[i] = v;
    s2 += v * v;
  }
  s2 = block_sum(s2, scratch);
  const float inv = 1.f / sqrtf(s2 / (float)H + eps);
#pragma unroll
  for (int u = 0; u < KEEP; ++u) {
    const int i = threadIdx.x + u * blockDim.x;
    if (i < H) o[i] = from_f<act_t>(keep[u] * inv * wk[u]);
  }
  for (int i = threadIdx.x + KEEP * blockDim.x; i < H; i += blockDim.x) {
    const float v = rows == nullptr ? x[i] : x[i] + to_f(yr[i]) * inv_y * wy[i];
    o[i] = from_f<act_t>(v * inv * w[i]);
  }
}

// The same with 16-byte loads, as above; the stream's new row is written behind both sums (2 rows of 2,048 values: 3.0 us, now 2.1).
template <int ITERS>
__global__ __launch_bounds__(row_most(ITERS)) void add_normed_rmsnorm_vec_kernel(float* __restrict__ resid, const act_t* __restrict__ y,
                                                                      const float* __restrict__ wy, float eps_y,
                                                                      const int* __restrict__ rows, const float* __restrict__ w, float eps,
                                                                      act_t* __restrict__ out, int H) {
  __shared__ float scratch[16];
  const size_t r = rows != nullptr ? (size_t)rows[blockIdx.x] : (size_t)blockIdx.x;
  float* x = resid + r * H;
  const int H4 = H / 4;
  f4 v[ITERS], wv[ITERS], wyv[ITERS];
  a4 yv[ITERS];
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int i = min((int)(threadIdx.x + it * blockDim.x), H4 - 1);
    yv[it] = ((const a4*)(y + r * H))[i];
    v[it] = ((const f4*)x)[i];
    wyv[it] = ((const f4*)wy)[i];
    wv[it] = ((const f4*)w)[i];
  }
  float ss = 0.f, s2 = 0.f;
#pragma unroll
  for (int it = 0; it < ITERS; ++it)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float n = threadIdx.x + it * blockDim.x < H4 ? to_f(yv[it].v[j]) : 0.f;
      ss += n * n;
    }
  const float inv_y = 1.f / sqrtf(block_sum(ss, scratch) / (float)H + eps_y);
#pragma unroll
  for (int it = 0; it < ITERS; ++it)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[it].v[j] += to_f(yv[it].v[j]) * inv_y * wyv[it].v[j];
      s2 += threadIdx.x + it * blockDim.x < H4 ? v[it].v[j] * v[it].v[j] : 0.f;
    }
  const float inv = 1.f / sqrtf(block_sum(s2, scratch) / (float)H + eps);
  act_t* o = out + (size_t)blockIdx.x * H;
#pragma unroll
  for (int it = 0; it < ITERS; ++it) {
    const int i = threadIdx.x + it * blockDim.x;
    if (i < H4) {
      a4 ov;
#pragma unroll
      for (int j = 0; j < 4; ++j) ov.v[j] = from_f<act_t>(v[it].v[j] * inv * wv[it].v[j]);
      if (rows == nullptr) ((f4*)x)[i] = v[it];
      ((a4*)o)[i] = ov;
    }
  }
}

extern "C" const char* sl_add_normed_rmsnorm(float* resid, const void* y, const float* wy, float eps_y,
                                             const int* rows, const float* w, float eps, void* out, int R,
                                             int H, hipStream_t stream) {
  SL_CHECK(R >= 0 && H > 0, "add_normed_rmsnorm: sizes must be positive");
  SL_CHECK(y != nullptr && wy != nullptr && w != nullptr, "add_normed_rmsnorm: the output and both gains are required");
  if (R == 0) return nullptr;
  if (H % 4 == 0 && H <= 4 * 8 * 512 && ((uintptr_t)resid | (uintptr_t)w | (uintptr_t)wy) % 16 == 0 &&
      ((uintptr_t)y | (uintptr_t)out) % sizeof(a4) == 0) {
    const int H4 = H / 4, n = row_threads(R, H4), iters = (H4 + n - 1) / n;
    auto run = [&](auto kernel) { kernel<<<R, n, 0, stream>>>(resid, (const act_t*)y, wy, eps_y, rows, w, eps, (act_t*)out, H); };
    with_groups(iters, [&](auto groups) { run(add_normed_rmsnorm_vec_kernel<decltype(groups)::n>); });
    return sl_launch_status();
  }
  const int threads = H >= 2048 ? 512 : 256, need = (H + threads - 1) / threads;
  auto run = [&](auto kernel) {
    kernel<<<R, threads, 0, stream>>>(resid, (const act_t*)y, wy, eps_y, rows, w, eps, (act_t*)out, H);
  };
  if (need <= 1) run(add_normed_rmsnorm_kernel<1>);
  else if (need <= 2) run(add_normed_rmsnorm_kernel<2>);
  else if (need <= 4) run(add_normed_rmsnorm_kernel<4>);
  else run(add_normed_rmsnorm_kernel<8>);
  return sl_launch_status();
}

// out = sa * a + sb * b, float sums: the outputs of two mixers that ran side by side.
__global__ void scaled_sum_kernel(const act_t* __restrict__ a, float sa, const act_t* __restrict__ b, float sb,
                                  act_t* __restrict__ out, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = from_f<act_t>(sa * to_f(a[i]) + sb * to_f(b[i]));
}

extern "C" const char* sl_scaled_sum(const void* a, float sa, const void* b, float sb, void* out, long long n,
                                     hipStream_t stream) {
  SL_CHECK(n >= 0, "scaled_sum: the count must not be negative");
  if (n == 0) return nullptr;
  scaled_sum_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>((const act_t*)a, sa, (const act_t*)b, sb,
                                                                    (act_t*)out, (size_t)n);
  return sl_launch_status();
}

// x = cap * tanh(x / cap) in place on float values (logits).
__global__ void softcap_kernel(float* __restrict__ x, float cap, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = cap * tanhf(x[i] / cap);
}

extern "C" const char* sl_softcap(float* x, float cap, long long n, hipStream_t stream) {
  SL_CHECK(n >= 0 && cap > 0.f, "softcap: the count must not be negative, the cap positive");
  if (n == 0) return nullptr;
  softcap_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(x, cap, (size_t)n);
  return sl_launch_status();
}

// x *= factor in place on float values (logits).
__global__ void scale_kernel(float* __restrict__ x, float factor, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] *= factor;
}

extern "C" const char* sl_scale(float* x, float factor, long long n, hipStream_t stream) {
  SL_CHECK(n >= 0, "scale: the count must not be negative");
  if (n == 0) return nullptr;
  scale_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(x, factor, (size_t)n);
  return sl_launch_status();
}
