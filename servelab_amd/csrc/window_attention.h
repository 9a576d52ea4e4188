// What the two window attention sources share (the float kernel for every size and both
// activation types, and the matrix-core kernel for bfloat16): the parameters of a call, and
// the kernel that merges the shares of the keys.
#pragma once
#include "common.h"

struct WindowAttention {
  const act_t* q;            // head h of token t at q + t * q_stride + h * Dk
  int q_stride;
  const act_t* kc;           // [pages][nkv][page][Dk]
  const act_t* vc;           // [pages][nkv][Dv][page], or nullptr: values are key channels [0, Dv)
  const int* tables;         // [sequences][max_pages]
  int max_pages;
  const int* cu_q;           // [sequences + 1]
  const int* positions;      // [tokens]
  int nh, nkv, Dk, Dv, page;
  float scale;
  float softcap;             // c > 0: the scaled score becomes c tanh(score / c); 0: left as it is
  int window;                // 0: every earlier key
  int chunk;                 // > 0: keys of the query's own chunk of so many positions; 0: no chunks
  int keep_first;
  const float* slopes;       // [nh] or nullptr
  const float* sinks;        // [nh] or nullptr
  const act_t* gate;         // gate of (t, h) at gate[t * gate_stride + h], or nullptr
  int gate_stride;
  const float* channel_gate; // gate of (t, h, d) at channel_gate[t * channel_stride + h * Dv + d], or nullptr
  int channel_stride;
  act_t* out;                // [tokens][nh][Dv]
  int nsplit;
  float* part_o;             // [tokens][nh][nsplit][Dv]
  float* part_ml;            // [tokens][nh][nsplit][2]
};

// The first key that a query at position pos sees by window and chunk (kept first keys aside).
__device__ __forceinline__ int first_key(const WindowAttention& a, int pos) {
  int lo = a.window > 0 && pos - a.window + 1 > 0 ? pos - a.window + 1 : 0;
  if (a.chunk > 0) {
    const int c = pos - pos % a.chunk;
    lo = c > lo ? c : lo;
  }
  return lo;
}

__device__ __forceinline__ float sigmoidf_(float x) { return 1.f / (1.f + expf(-x)); }

// Merges the shares of a (token, head): out = sum_j w_j o_j / (sum_j w_j l_j + sink's term),
// w_j = exp(m_j - top); a share without keys has m = -inf and drops out.  One
// wavefront per (token, head, 64 channels); shares are added in their order.
// Everything a wavefront needs is asked for before anything is used (SHARES shares: for a share that is not there the last one is
// read, and not used), so that a call is one trip to memory: behind the weights, eight shares a trip, 32 shares took four.
template <int SHARES>
__global__ __launch_bounds__(64) void window_attention_combine_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml, int nsplit, int nh, int Dv,
    const float* __restrict__ sinks, const act_t* __restrict__ gate, int gate_stride,
    const float* __restrict__ channel_gate, int channel_stride, act_t* __restrict__ out) {
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, d = blockIdx.z * 64 + lane, dc = d < Dv ? d : Dv - 1;
  const size_t base = ((size_t)t * nh + h) * nsplit;
  float v[SHARES];
#pragma unroll
  for (int j = 0; j < SHARES; ++j) v[j] = part_o[(base + (j < nsplit ? j : nsplit - 1)) * Dv + dc];
  // lane j holds share j (at most 64 shares)
  const size_t mine = (base + (lane < nsplit ? lane : nsplit - 1)) * 2;
  const float m_at = part_ml[mine], l_at = part_ml[mine + 1];
  const float sink = sinks != nullptr ? sinks[h] : -INFINITY;
  const float open = gate != nullptr ? to_f(gate[(size_t)t * gate_stride + h]) : 0.f;
  const float open_here = channel_gate != nullptr ? channel_gate[(size_t)t * channel_stride + h * Dv + dc] : 0.f;
  const float mj = lane < nsplit ? m_at : -INFINITY, lj = lane < nsplit ? l_at : 0.f;
  const float top = fmaxf(wave_max(mj), sink);
  const float wj = mj == -INFINITY ? 0.f : expf(mj - top);
  const float denom = wave_sum(wj * lj) + (sinks != nullptr ? expf(sink - top) : 0.f);
  float f = 1.f / denom;
  if (gate != nullptr) f *= sigmoidf_(open);
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < SHARES; ++j) s += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wj), j)) * (j < nsplit ? v[j] : 0.f);
  if (channel_gate != nullptr) s *= sigmoidf_(open_here);
  if (d < Dv) out[((size_t)t * nh + h) * Dv + d] = from_f<act_t>(s * f);
}

static inline void launch_combine(const WindowAttention& a, int num_tokens, hipStream_t stream) {
  auto run = [&](auto kernel) {
    kernel<<<dim3(num_tokens, a.nh, (a.Dv + 63) / 64), 64, 0, stream>>>(a.part_o, a.part_ml, a.nsplit, a.nh, a.Dv, a.sinks, a.gate, a.gate_stride,
                                                                     a.channel_gate, a.channel_stride, a.out);
  };
  if (a.nsplit <= 8) run(window_attention_combine_kernel<8>);
  else if (a.nsplit <= 16) run(window_attention_combine_kernel<16>);
  else if (a.nsplit <= 32) run(window_attention_combine_kernel<32>);
  else run(window_attention_combine_kernel<64>);
}
