// The recurrences of recurrent.hip in chunks of 32 tokens: what a chunk does to the state and what its tokens read
// are products of matrices, which run on the float32 matrix instructions, so the only chain over time is one
// step a chunk instead of one a token.
//
// With a_t the decay of token t (a vector over the key channels, or one number), g(s, t) the product of the decays
// of tokens s + 1 .. t, w_t what a token adds (1, or a number), S0 the state at the chunk's start and o_t = S_t^T q_t:
//   u_t = v_t;  delta rule:  u_t = beta_t (v_t - (g(-1, t) k_t)^T S0 - sum over s < t of M[t][s] u_s),
//                            M[t][s] = sum_d k_t k_s g(s, t), which is U = V~ - W S0, V~ = R V, W = R (g(-1, .) k),
//                            R = (I + tril(beta M, -1))^-1 diag(beta)
//   o_t = (g(-1, t) q_t)^T S0 + sum over s <= t of A[t][s] u_s,  A[t][s] = w_s sum_d q_t k_s g(s, t)
//   S'  = g(-1, 31) S0 + sum over s of (w_s g(s, 31) k_s) u_s^T
// scan_prepare_*_kernel make, for every chunk and head by itself, the factors that do not depend on S0;
// scan_walk_kernel walks a head's chunks.  Decays are never divided by: a product g is the exponential of a sum of
// logarithms of one sign (running sums inside blocks of 8 tokens, sums of whole blocks between them), so no
// difference of large sums is taken, nothing overflows however strong a decay is, and everything is float32.
// The error against float64 is that of the walk token by token (2,048 tokens: read-outs 1.1e-7 to 1.6e-7 against 1.0e-7
// to 1.4e-7, matrix LSTM 1.0e-6 against 1.1e-6, states 1e-7 either way).
//
// One prompt of 2,048 tokens, us, token by token -> in chunks (prepare + walk): decay, 8 heads of 128 x 256: 486 -> 100
// (26 + 77); forget 450 -> 104; matrix LSTM 680 -> 117 (21 + 92); delta, 16 heads of 128 x 128: 700 -> 161 (64 + 100);
// delta with a decay a head 605 -> 133 (32 + 106); state-space, 64 heads of 128 x 64 in 8 groups: 535 -> 116 (34 + 86).
// The walk is bound by its chain: 1.2 to 1.6 us a chunk, of which the products are 0.6 to 0.8.
#pragma once
#include <type_traits>

typedef float scan_v4 __attribute__((ext_vector_type(4)));
constexpr int SCAN_CHUNK = 32;
constexpr int SCAN_MAX_TILES = 4;                       // key channels: at most 64 of these

// What scan_prepare_*_kernel leave, by chunk.  Operands of the matrix instruction lie as the walk's lanes hold them:
// a 16 x 16 block is 64 lanes of 4 values, row r and column c at lane r + 16 (c / 4), place c % 4.
struct ScanChunks {
  float* q;        // [chunk][head | group][Dp / 16][2][256]   rows of q, times their decay where it is per channel
  float* kt;       // [chunk][head | group][Dp / 16][2][256]   k turned (rows are channels), times its decay to the end
  float* a;        // [chunk][head][2][2][256]
  float* w;        // [chunk][head][Dp / 16][2][256]           delta rule: W
  float* vt;       // [chunk][head][ceil(Dv / 16)][2][256]     delta rule: V~ (lane r / 4 * 16 + c, place r % 4)
  float* keep;     // [chunk][head][Dp] decays of the whole chunk per channel | [chunk][head][96 + 4]: per token the
                   // factors of q and of k, 32 floors e^-m, the chunk's decay, the running maximum at its end
  float* gates;    // matrix LSTM: [chunk][head][64 + 2]: i, f of the tokens; sum of f, maximum they reach from -inf
  int Dp;
};

template <int MODE> struct ScanForm {
  static constexpr bool SCALAR = MODE == SCAN_LSTM || MODE == SCAN_SSD || MODE == SCAN_DELTA_HEAD;
  static constexpr bool DELTA = MODE == SCAN_DELTA || MODE == SCAN_DELTA_HEAD;
};
// chunk ids of a step: sequence s owns cu_q[s] / 32 + s and the ones behind it (there is room for the rounding up)
__device__ __forceinline__ int scan_chunk_id(int first, int s, int ci) { return first / SCAN_CHUNK + s + ci; }

// The matrix LSTM's gates after cap and squashing, and what a chunk does to the running maximum: m -> max(m + F, M).
__global__ __launch_bounds__(256) void scan_gates_kernel(const MatrixScan a, const ScanChunks w) {
  const int s = blockIdx.y, first = a.cu_q[s], len = a.cu_q[s + 1] - first, t0 = blockIdx.x * SCAN_CHUNK;
  if (t0 >= len || len < a.line) return;
  const int nt = min(SCAN_CHUNK, len - t0);
  for (int h = threadIdx.x / SCAN_CHUNK; h < a.H; h += 256 / SCAN_CHUNK) {
    const int tt = threadIdx.x % SCAN_CHUNK;
    float ig = -INFINITY, fg = 0.f;
    if (tt < nt) {
      const float* gr = a.gates + (size_t)(first + t0 + tt) * a.gate_stride;
      ig = a.cap * tanhf(gr[a.i_col + h] / a.cap);
      fg = logsigmoidf_(a.cap * tanhf(gr[a.f_col + h] / a.cap));
    }
    float* out = w.gates + ((size_t)scan_chunk_id(first, s, blockIdx.x) * a.H + h) * (2 * SCAN_CHUNK + 2);
    out[tt] = ig;
    out[SCAN_CHUNK + tt] = fg;
    float F = fg, M = ig;
#pragma unroll
    for (int o = 1; o < SCAN_CHUNK; o <<= 1) {           // (earlier tokens in the lower lane)
      const float F2 = __shfl_down(F, o, SCAN_CHUNK), M2 = __shfl_down(M, o, SCAN_CHUNK);
      M = fmaxf(M + F2, M2);
      F += F2;
    }
    if (tt == 0) {
      out[2 * SCAN_CHUNK] = F;
      out[2 * SCAN_CHUNK + 1] = M;
    }
  }
}

// ---- What the two forms of scan_prepare share.  LDS rows of a chunk: [32][Dp + 4] floats; small squares [32][36].
constexpr int SCAN_AR = SCAN_CHUNK + 4;

// f(place, token, channel) for this thread's places of the chunk's rows, eight at a time, so that eight loads are in flight.
template <typename Load, typename Keep>
__device__ __forceinline__ void scan_rows(int Dp, int tid, Load load, Keep keep) {
  for (int i0 = tid; i0 < SCAN_CHUNK * Dp; i0 += 8 * 256) {
    float x[8][3];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int idx = i0 + e * 256, tt = idx / Dp;
      load(tt, idx - tt * Dp, x[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int idx = i0 + e * 256, tt = idx / Dp;
      keep(tt, idx - tt * Dp, x[e]);
    }
  }
}

// Products of a triangle: t reads s <= t, and the zeros above the diagonal are in the matrix instruction all the same, where an
// infinity or NaN of a later token turns them into NaN.  Whoever finds a result that is not finite (scan_odd gathers that
// without a branch) therefore takes the products again with these sums, which leave the zeros out.  An operand's block is 16 x 16,
// its row at lane row + 16 (column / 4), place column % 4; TRIANGLE_FIRST: `x` is the triangle, else `y` is, turned.
__device__ __forceinline__ float scan_odd(float odd, const scan_v4& result) {
  return fmaf((result[0] + result[1]) + (result[2] + result[3]), 0.f, odd);   // (0, or NaN from the first such result on)
}
template <bool TRIANGLE_FIRST>
__device__ __forceinline__ scan_v4 scan_lower_only(const scan_v4& x, const scan_v4& y, int lane) {
  const int n = lane & 15, r0 = 4 * (lane >> 4);
  scan_v4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int from = 0; from < 64; from += 16)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int s = from / 4 + c;
      const float ys = __shfl(y[c], from + n, SL_WAVE);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float xs = __shfl(x[c], from + r0 + i, SL_WAVE);
        if (s <= (TRIANGLE_FIRST ? r0 + i : n)) sum[i] = fmaf(xs, ys, sum[i]);
      }
    }
  return sum;
}

// A 32 x 32 square of LDS as the walk's first operand.
__device__ __forceinline__ void scan_square_out(const float* As, float* out, int tid) {
  const int l = tid & 63, r = tid >> 7, j = (tid >> 6) & 1;
  *(scan_v4*)(out + tid * 4) = *(const scan_v4*)(As + (16 * r + (l & 15)) * SCAN_AR + 16 * j + 4 * (l >> 4));
}

// The delta rule's R from L = tril(beta M, -1) in Ms (a whole workgroup; As takes R, Ms is used up), then W = R K and
// V~ = R V of one head.  Blocks of 16: their inverses by forward substitution, a column a lane, and the block below
// them as two products.
__device__ __forceinline__ void scan_delta_rows(const MatrixScan& a, const ScanChunks& c, float* As, float* Ms,
                                                const float* ks, const float* beta, int chunk, int h, int first, int nt,
                                                int tid) {
  constexpr int C = SCAN_CHUNK, AR = SCAN_AR;
  const int wave = tid >> 6, lane = tid & 63, n = lane & 15, gq = lane >> 4;
  const int Dp = c.Dp, row = Dp + 4, blocks = Dp / 16;
  if (tid < C) {
    const int b = 16 * (tid >> 4), col = tid & 15;
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float v = t == col ? 1.f : 0.f;
#pragma unroll
      for (int u = 0; u < t; ++u) v -= Ms[(b + t) * AR + b + u] * x[u];
      x[t] = v;
    }
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      As[(b + t) * AR + b + col] = x[t];
      if (b == 0) As[t * AR + 16 + col] = 0.f;
    }
  }
  __syncthreads();
  if (wave == 0) {
    scan_v4 acc = {0.f, 0.f, 0.f, 0.f};
    const scan_v4 lv = *(const scan_v4*)(Ms + (16 + n) * AR + 4 * gq);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(lv[i], As[(4 * gq + i) * AR + n], acc, 0, 0, 0);
    scan_v4 below = {0.f, 0.f, 0.f, 0.f};
    const scan_v4 rv = *(const scan_v4*)(As + (16 + n) * AR + 16 + 4 * gq);
    // (the first product's results lie as the second one's operand)
#pragma unroll
    for (int i = 0; i < 4; ++i) below = __builtin_amdgcn_mfma_f32_16x16x4f32(rv[i], acc[i], below, 0, 0, 0);
    if (__ballot(scan_odd(0.f, below) != 0.f)) below = scan_lower_only<true>(rv, acc, lane);
#pragma unroll
    for (int i = 0; i < 4; ++i) As[(16 + 4 * gq + i) * AR + n] = -below[i];
  }
  __syncthreads();
  scan_v4 rv[2][2];                                     // rows 16 r + n of R, columns 16 j + 4 gq ..
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int j = 0; j < 2; ++j)
      rv[r][j] = *(const scan_v4*)(As + (16 * r + n) * AR + 16 * j + 4 * gq) * *(const scan_v4*)(beta + 16 * j + 4 * gq);
  const int vblocks = (a.Dv + 15) / 16;
  float* vout = c.vt + ((size_t)chunk * a.H + h) * vblocks * 512;
  float* wout = c.w + ((size_t)chunk * a.H + h) * blocks * 512;
  float odd = 0.f;
  auto rows = [&](auto careful) {
    for (int blk = wave; blk < vblocks; blk += 4) {
      const int col = 16 * blk + n;
      scan_v4 v[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int t = 16 * j + 4 * gq + i;
          v[j][i] = t < nt && col < a.Dv ? a.src[(size_t)(first + t) * a.src_stride + a.v_col + h * a.Dv + col] : 0.f;
        }
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        scan_v4 acc[2] = {};
#pragma unroll
        for (int j = 0; j <= r; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(rv[r][j][i], v[j][i], acc[j], 0, 0, 0);
        if (careful) acc[r] = scan_lower_only<true>(rv[r][r], v[r], lane);
        else odd = scan_odd(odd, acc[r]);
        *(scan_v4*)(vout + ((size_t)blk * 2 + r) * 256 + lane * 4) = acc[0] + acc[1];
      }
    }
    for (int blk = wave; blk < blocks; blk += 4)        // W turned: rows are channels, columns tokens
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        scan_v4 acc[2] = {}, kv;
#pragma unroll
        for (int j = 0; j <= r; ++j) {
#pragma unroll
          for (int i = 0; i < 4; ++i) kv[i] = ks[(16 * j + 4 * gq + i) * row + 16 * blk + n];
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[i], rv[r][j][i], acc[j], 0, 0, 0);
        }
        if (careful) acc[r] = scan_lower_only<false>(kv, rv[r][r], lane);
        else odd = scan_odd(odd, acc[r]);
        *(scan_v4*)(wout + ((size_t)blk * 2 + r) * 256 + lane * 4) = acc[0] + acc[1];
      }
  };
  rows(std::false_type{});
  if (__ballot(odd != 0.f)) rows(std::true_type{});
}

// One decay a head: a workgroup per (chunk, group of heads, sequence), since the products of q and k are the group's; a
// head's decays and what a token adds come in afterwards.
template <int MODE>
__global__ __launch_bounds__(256) void scan_prepare_scalar_kernel(const MatrixScan a, const ScanChunks c) {
  constexpr bool DELTA = ScanForm<MODE>::DELTA;
  constexpr int C = SCAN_CHUNK, AR = SCAN_AR;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int s = blockIdx.z, g = blockIdx.y, ci = blockIdx.x;
  const int first = a.cu_q[s], len = a.cu_q[s + 1] - first, t0 = ci * C;
  if (t0 >= len || len < a.line) return;                // (the whole workgroup)
  const int nt = min(C, len - t0), rep = a.H / a.G;
  const int chunk = scan_chunk_id(first, s, ci);
  const int Dp = c.Dp, row = Dp + 4, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, gq = lane >> 4;
  float* qs = lds;                                      // [C][row]; delta rule: then k with a head's decays
  float* ks = qs + C * row;                             // [C][row]
  float* qk = ks + C * row;                             // [C][AR] sums of q k
  float* kk = qk + C * AR;                              // [C][AR] sums of k k (delta rule)
  float* As = kk + (DELTA ? C * AR : 0);                // [C][AR] a head's
  float* Ms = As + C * AR;                              // [C][AR] (delta rule)
  float* la = Ms + (DELTA ? C * AR : 0);                // [C] logarithm of a token's decay | what it adds | beta | decay so far
  float* add = la + C;
  float* beta = add + C;
  float* sofar = beta + C;

  scan_rows(Dp, tid, [&](int tt, int d, float* x) {
    x[0] = x[1] = 0.f;
    if (tt < nt && d < a.D) {
      const float* src = a.src + (size_t)(first + t0 + tt) * a.src_stride + g * a.D + d;
      x[0] = src[a.q_col];
      x[1] = src[a.k_col];
    }
  }, [&](int tt, int d, const float* x) {
    qs[tt * row + d] = x[0];
    ks[tt * row + d] = x[1];
  });
  __syncthreads();
  for (int b = wave; b < (DELTA ? 6 : 3); b += 4) {     // 16 x 16 blocks, the one above the diagonal left out
    const int bt = b % 3 == 0 ? 0 : 1, bs = b % 3 == 2 ? 1 : 0;
    const float* x = (b >= 3 ? ks : qs) + (16 * bt + n) * row + 4 * gq;
    const float* y = ks + (16 * bs + n) * row + 4 * gq;
    scan_v4 sums[4] = {};                               // (four sums of every fourth piece: shorter chains of roundings)
    for (int d = 0; d < Dp; d += 64)
#pragma unroll
      for (int b4 = 0; b4 < 4; ++b4) {
        const scan_v4 xv = *(const scan_v4*)(x + d + 16 * b4), yv = *(const scan_v4*)(y + d + 16 * b4);
#pragma unroll
        for (int i = 0; i < 4; ++i) sums[b4] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[i], yv[i], sums[b4], 0, 0, 0);
      }
    const scan_v4 acc = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    float* out = (b >= 3 ? kk : qk) + (16 * bt + 4 * gq) * AR + 16 * bs + n;
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i * AR] = acc[i];
  }
  {
    const size_t at = ((size_t)chunk * a.G + g) * (Dp / 16) * 512;
    for (int idx = tid; idx < Dp * 8; idx += 256) {
      const int l = idx & 63, r = (idx >> 6) & 1, blk = idx >> 7;
      *(scan_v4*)(c.q + at + (size_t)idx * 4) = *(const scan_v4*)(qs + (16 * r + (l & 15)) * row + 16 * blk + 4 * (l >> 4));
      scan_v4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = ks[(16 * r + 4 * (l >> 4) + i) * row + 16 * blk + (l & 15)];
      *(scan_v4*)(c.kt + at + (size_t)idx * 4) = v;
    }
  }
  for (int h = g * rep; h < (g + 1) * rep; ++h) {
    float m_end = 0.f, floor_ = 0.f;
    __syncthreads();                                    // (the head before this one is done with what follows)
    if (MODE == SCAN_LSTM) {
      if (wave == 0) {
        // the running maximum at the chunk's start from what the chunks before it do to it, 64 of them at a time
        const bool fresh = a.positions[first] == 0;
        const float* slot = a.state + (size_t)a.slots[s] * a.state_stride + (size_t)a.H * a.Dv * a.D + (size_t)a.H * a.D;
        float m = fresh ? 0.f : slot[h];
        for (int c0 = 0; c0 < ci; c0 += 64) {
          float F = 0.f, M = -INFINITY;
          if (c0 + lane < ci) {
            const float* gr = c.gates + ((size_t)(chunk - ci + c0 + lane) * a.H + h) * (2 * C + 2);
            F = gr[2 * C];
            M = gr[2 * C + 1];
          }
#pragma unroll
          for (int o = 1; o < 64; o <<= 1) {
            const float F2 = __shfl_down(F, o, SL_WAVE), M2 = __shfl_down(M, o, SL_WAVE);
            M = fmaxf(M + F2, M2);
            F += F2;
          }
          m = fmaxf(m + __shfl(F, 0, SL_WAVE), __shfl(M, 0, SL_WAVE));
        }
        const float* gr = c.gates + ((size_t)chunk * a.H + h) * (2 * C + 2);
        const float ig = gr[lane & 31], fg = gr[C + (lane & 31)];
        float before = 0.f, top = 0.f;
        for (int tt = 0; tt < nt; ++tt) {
          const float reach = fmaxf(__shfl(fg, tt, SL_WAVE) + m, __shfl(ig, tt, SL_WAVE));
          if (lane == tt) {
            before = m;
            top = reach;
          }
          m = reach;
        }
        m_end = m;
        floor_ = expf(-top);
        if (lane < C) {
          la[lane] = lane < nt ? fg + before - top : 0.f;
          add[lane] = lane < nt ? expf(ig - top) : 0.f;
        }
      }
    } else if (tid < C) {
      float l = 0.f, w = 0.f, b = 0.f;
      if (tid < nt) {
        const float* gr = a.gates + (size_t)(first + t0 + tid) * a.gate_stride;
        if (MODE == SCAN_SSD) {
          w = softplusf_(gr[a.i_col + h] + a.step_bias[h]);
          l = -expf(a.rates[h]) * w;
        } else {
          w = 1.f;
          b = sigmoidf_(gr[a.i_col + h]);
          l = -expf(a.rates[h]) * softplusf_(gr[a.f_col + h] + a.step_bias[h]);
        }
      }
      la[tid] = l;
      add[tid] = w;
      beta[tid] = b;
    }
    __syncthreads();
    {
      // this thread's row and four neighbouring columns: the sum of the logarithms grows from the diagonal down to them
      const int t = tid >> 3, u0 = 4 * (tid & 7);
      float sum = 0.f;
      for (int r = u0 + 4; r <= t; ++r) sum += la[r];
#pragma unroll
      for (int i = 3; i >= 0; --i) {
        const int u = u0 + i;
        const float e = t >= u ? expf(sum) : 0.f;
        As[t * AR + u] = t >= u ? qk[t * AR + u] * (e * a.q_scale * add[u]) : 0.f;
        if (DELTA) Ms[t * AR + u] = t > u ? kk[t * AR + u] * (e * beta[t]) : 0.f;
        if (t >= u) sum += la[u];
      }
    }
    if (tid < C) {
      float head = 0.f, tail = 0.f;
      for (int r = 0; r <= tid; ++r) head += la[r];
      for (int r = tid + 1; r < C; ++r) tail += la[r];
      float* out = c.keep + ((size_t)chunk * a.H + h) * (3 * C + 4);
      const float eh = expf(head);
      out[tid] = eh * a.q_scale;
      out[C + tid] = expf(tail) * add[tid];
      out[2 * C + tid] = floor_;
      if (tid == C - 1) out[3 * C] = eh;
      if (tid == 0) out[3 * C + 1] = m_end;
      sofar[tid] = eh;
    }
    __syncthreads();
    scan_square_out(As, c.a + ((size_t)chunk * a.H + h) * 1024, tid);
    if constexpr (DELTA) {
      for (int idx = tid; idx < C * Dp; idx += 256) {
        const int t = idx / Dp, d = idx - t * Dp;
        qs[t * row + d] = ks[t * row + d] * sofar[t];
      }
      __syncthreads();
      scan_delta_rows(a, c, As, Ms, qs, beta, chunk, h, first + t0, nt, tid);
    }
  }
}

// Decays per channel: a workgroup per (chunk, head, sequence).
template <int MODE>
__global__ __launch_bounds__(256) void scan_prepare_channel_kernel(const MatrixScan a, const ScanChunks c) {
  constexpr bool DELTA = ScanForm<MODE>::DELTA;
  constexpr int C = SCAN_CHUNK, AR = SCAN_AR;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int s = blockIdx.z, h = blockIdx.y, ci = blockIdx.x;
  const int first = a.cu_q[s], len = a.cu_q[s + 1] - first, t0 = ci * C;
  if (t0 >= len || len < a.line) return;                // (the whole workgroup)
  const int nt = min(C, len - t0), g = h / (a.H / a.G);
  const int chunk = scan_chunk_id(first, s, ci);
  const int Dp = c.Dp, row = Dp + 4, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, gq = lane >> 4;
  float* qs = lds;                                      // [C][row]
  float* ks = qs + C * row;                             // [C][row]
  float* ls = ks + C * row;                             // [C][row] logarithms of the decays; then k with its decay to its block's end
  float* As = ls + C * row;                             // [C][AR]
  float* Ms = As + C * AR;                              // [C][AR] (delta rule)
  float* beta = Ms + (DELTA ? C * AR : 0);              // [C]
  float* part = beta + C;                               // [4][C][8][DELTA ? 2 : 1]; then [4][Dp] decays of the blocks
  float* ahead = part + 4 * Dp;                         // [5][Dp] decays of the blocks before one; behind it [4][Dp] of those after it
  float* after = ahead + 5 * Dp;

  scan_rows(Dp, tid, [&](int tt, int d, float* x) {
    x[0] = x[1] = x[2] = 0.f;
    if (tt < nt && d < a.D) {
      const size_t t = first + t0 + tt;
      const float* src = a.src + t * a.src_stride + g * a.D + d;
      x[0] = src[a.q_col];
      x[1] = src[a.k_col];
      x[2] = MODE == SCAN_FORGET ? a.lower[h * a.D + d] : a.log_decay[(t * a.H + h) * a.D + d];
    }
  }, [&](int tt, int d, const float* x) {
    float q = x[0], k = x[1], l = x[2];
    if (MODE == SCAN_FORGET) {
      // f = l + (1 - l) sigmoid(z), 1 - f from its own side (as in matrix_scan_kernel)
      const float bound = x[2], en = expf(-fabsf(k)), big = 1.f / (1.f + en), small = en * big;
      const bool pos = k >= 0.f, in = tt < nt && d < a.D;
      l = in ? logf(fmaxf(bound + (1.f - bound) * (pos ? big : small), 1.1754944e-38f)) : 0.f;
      k = in ? (1.f - bound) * (pos ? small : big) : 0.f;
      q = q * sigmoidf_(q);
    } else {
      l = l < -110.f ? -110.f : l;                      // (e^-110 is 0 in float; NaN stays NaN)
    }
    qs[tt * row + d] = q * a.q_scale;
    ks[tt * row + d] = k;
    ls[tt * row + d] = l;
  });
  if (DELTA && tid < C) beta[tid] = tid < nt ? sigmoidf_(a.gates[(size_t)(first + t0 + tid) * a.gate_stride + a.i_col + h]) : 0.f;
  for (int i = tid; i < C * AR; i += 256) {
    As[i] = 0.f;
    if (DELTA) Ms[i] = 0.f;
  }
  __syncthreads();
  // Pairs inside a block of 8 tokens: thread (s, eighth of the channels) walks the tokens behind s with a running
  // sum of the logarithms.
  {
    const int u = tid & 31, dg = tid >> 5, per = Dp / 8;
    float pa[8], pm[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      pa[i] = 0.f;
      pm[i] = 0.f;
    }
    for (int d = dg * per; d < (dg + 1) * per; d += 4) {
      const scan_v4 kv = *(const scan_v4*)(ks + u * row + d), qv = *(const scan_v4*)(qs + u * row + d);
      pa[0] += (qv[0] * kv[0] + qv[1] * kv[1]) + (qv[2] * kv[2] + qv[3] * kv[3]);
      scan_v4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 1; i < 8; ++i) {
        const int r = min(u + i, C - 1);                // (a token beyond the block: summed up and left out below)
        const scan_v4 lv = *(const scan_v4*)(ls + r * row + d), qr = *(const scan_v4*)(qs + r * row + d);
        sum += lv;
        scan_v4 x;
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = kv[j] * expf(sum[j]);
        pa[i] += (qr[0] * x[0] + qr[1] * x[1]) + (qr[2] * x[2] + qr[3] * x[3]);
        if (DELTA) {
          const scan_v4 kr = *(const scan_v4*)(ks + r * row + d);
          pm[i] += (kr[0] * x[0] + kr[1] * x[1]) + (kr[2] * x[2] + kr[3] * x[3]);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      pa[i] += __shfl_xor(pa[i], 32, SL_WAVE);
      if (DELTA) pm[i] += __shfl_xor(pm[i], 32, SL_WAVE);
      if (lane < 32) {
        part[(wave * C + u) * 8 + i] = pa[i];
        if (DELTA) part[4 * C * 8 + (wave * C + u) * 8 + i] = pm[i];
      }
    }
  }
  __syncthreads();
  {
    const int u = tid >> 3, i = tid & 7, t = u + i;
    if ((u & 7) + i < 8) {
      float v[4], m[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        v[w] = part[(w * C + u) * 8 + i];
        if (DELTA) m[w] = part[4 * C * 8 + (w * C + u) * 8 + i];
      }
      As[t * AR + u] = (v[0] + v[1]) + (v[2] + v[3]);
      if (DELTA && i > 0) Ms[t * AR + u] = ((m[0] + m[1]) + (m[2] + m[3])) * beta[t];
    }
  }
  __syncthreads();
  // A block's rows take their decays from its start (q, and k for the delta rule) and to its end (k), in place: the
  // latter where the logarithms lay; `part` takes the sums of the four blocks.
  for (int idx = tid; idx < 4 * Dp; idx += 256) {
    const int b = idx / Dp, d = idx - b * Dp;
    float lv[8], sum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) lv[i] = ls[(8 * b + i) * row + d];
#pragma unroll
    for (int i = 7; i >= 0; --i) {
      ls[(8 * b + i) * row + d] = ks[(8 * b + i) * row + d] * expf(sum);
      sum += lv[i];
    }
    part[b * Dp + d] = sum;
    sum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      sum += lv[i];
      const float e = expf(sum);
      qs[(8 * b + i) * row + d] *= e;
      if (DELTA) ks[(8 * b + i) * row + d] *= e;
    }
  }
  __syncthreads();
  for (int d = tid; d < Dp; d += 256) {
    float sum = 0.f;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      ahead[b * Dp + d] = expf(sum);
      sum += part[b * Dp + d];
    }
    ahead[4 * Dp + d] = expf(sum);
    c.keep[((size_t)chunk * a.H + h) * Dp + d] = expf(sum);
    sum = 0.f;
#pragma unroll
    for (int b = 3; b >= 0; --b) {
      after[b * Dp + d] = expf(sum);
      sum += part[b * Dp + d];
    }
  }
  // Pairs of different blocks on the matrix cores: rows are the 8 tokens of block 1, 2 or 3 (q, then k), columns
  // 16 earlier tokens; a wavefront takes one of the four (block, columns) combinations.
  {
    const int bt = wave == 3 ? 3 : wave + 1, s0 = wave == 3 ? 16 : 0;
    const float* x = (n < 8 ? qs : ks) + (8 * bt + (n & 7)) * row + 4 * gq;
    const int col = s0 + n, bs = min(col >> 3, 3);
    const float* y = ls + col * row + 4 * gq;
    scan_v4 sums[4] = {};
    for (int d0 = 0; d0 < Dp; d0 += 64)
#pragma unroll
      for (int b4 = 0; b4 < 4; ++b4) {
        const int d = d0 + 16 * b4;
        const scan_v4 xv = *(const scan_v4*)(x + d);
        scan_v4 yv = *(const scan_v4*)(y + d), between = {0.f, 0.f, 0.f, 0.f};
        for (int b = bs + 1; b < bt; ++b) between += *(const scan_v4*)(part + b * Dp + d + 4 * gq);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          yv[i] *= bs + 1 < bt ? expf(between[i]) : 1.f;
          sums[b4] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[i], yv[i], sums[b4], 0, 0, 0);
        }
      }
    const scan_v4 acc = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    if (col < 8 * bt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 4 * gq + i;
        if (r < 8) As[(8 * bt + r) * AR + col] = acc[i];
        else if (DELTA) Ms[(8 * bt + r - 8) * AR + col] = acc[i] * beta[8 * bt + r - 8];
      }
    }
  }
  __syncthreads();
  {
    const size_t at = ((size_t)chunk * a.H + h) * (Dp / 16) * 512;
    for (int idx = tid; idx < Dp * 8; idx += 256) {
      const int l = idx & 63, r = (idx >> 6) & 1, blk = idx >> 7;
      const int t = 16 * r + (l & 15), d = 16 * blk + 4 * (l >> 4);
      *(scan_v4*)(c.q + at + (size_t)idx * 4) = *(const scan_v4*)(qs + t * row + d) * *(const scan_v4*)(ahead + (t >> 3) * Dp + d);
      const int u = 16 * r + 4 * (l >> 4), ch = 16 * blk + (l & 15);
      const float e = after[(u >> 3) * Dp + ch];
      scan_v4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = ls[(u + i) * row + ch] * e;
      *(scan_v4*)(c.kt + at + (size_t)idx * 4) = v;
    }
  }
  scan_square_out(As, c.a + ((size_t)chunk * a.H + h) * 1024, tid);
  if constexpr (DELTA) {
    __syncthreads();
    for (int idx = tid; idx < C * Dp; idx += 256) {
      const int t = idx / Dp, d = idx - t * Dp;
      ks[t * row + d] *= ahead[(t >> 3) * Dp + d];
    }
    __syncthreads();
    scan_delta_rows(a, c, As, Ms, ks, beta, chunk, h, first + t0, nt, tid);
  }
}

// A workgroup walks a head's chunks for 16 value channels (matrix LSTM: 15 and the normaliser).  Its four wavefronts
// share the key channels, TW blocks of 16 each, and keep their part of S in the matrix instruction's accumulators: lane
// (gq, n) holds rows 4 gq .. + 3 of a block for value channel n, which is also how the same instruction wants its second
// operand, so q^T S and W S need no exchange but the sum over the wavefronts (through LDS, one barrier a chunk).
// The operands of the chunks ahead are asked for while one is worked on.
template <int MODE, int TW>
__global__ __launch_bounds__(256, ScanForm<MODE>::DELTA && TW > 1 ? 1 : 2) void scan_walk_kernel(const MatrixScan a, const ScanChunks c, int S, int slices) {
  constexpr bool SCALAR = ScanForm<MODE>::SCALAR, DELTA = ScanForm<MODE>::DELTA;
  constexpr int C = SCAN_CHUNK, NP = DELTA ? 4 : 2;
  __shared__ scan_v4 part[2][4][NP][64];
  __shared__ bool again[2];
  // Workgroups go to the eight dies in turn: the slices of a head, which read the same operands, run on one of them.
  const int die = blockIdx.x & 7, rest = blockIdx.x >> 3, slice = rest % slices, hs = rest / slices * 8 + die;
  if (hs >= S * a.H) return;
  const int s = hs / a.H, h = hs - s * a.H, g = h / (a.H / a.G);
  const int first = a.cu_q[s], len = a.cu_q[s + 1] - first;
  if (len <= 0 || len < a.line) return;
  const int nchunks = (len + C - 1) / C, chunk0 = scan_chunk_id(first, s, 0);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, n = lane & 15, gq = lane >> 4;
  const int vcols = MODE == SCAN_LSTM ? 15 : 16;
  const bool is_n = MODE == SCAN_LSTM && n == 15;
  const int col = slice * vcols + n;
  const bool live = is_n || (col < a.Dv && n < vcols);
  const bool fresh = a.positions[first] == 0;
  float* slot = a.state + (size_t)a.slots[s] * a.state_stride;
  float* srow = is_n ? slot + (size_t)a.H * a.Dv * a.D + (size_t)h * a.D : slot + ((size_t)h * a.Dv + (live ? col : 0)) * a.D;
  const int blocks = c.Dp / 16, vblocks = (a.Dv + 15) / 16;
  scan_v4 st[TW];
  auto begin = [&]() {
#pragma unroll
    for (int b = 0; b < TW; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 16 * (wave * TW + b) + 4 * gq + i;
        st[b][i] = !fresh && live && d < a.D ? srow[d] : 0.f;
      }
  };
  begin();
  const float skip = MODE == SCAN_SSD ? a.skip[h] : 0.f;

  struct Chunk {
    scan_v4 q[TW][2], kt[TW][2], w[DELTA ? TW : 1][2], a[2], keep[SCALAR ? 5 : TW], v[2];
  };
  // (everything but the lane's own place is the same for the wavefront, so that it stays out of the vector registers)
  const int vcol = min(col, a.Dv - 1);
  auto ask = [&](int ci, Chunk& x) {
    const int chunk = chunk0 + ci;
    const size_t ah = (size_t)chunk * a.H + h;
    const float* q = c.q + ((size_t)chunk * (SCALAR ? a.G : a.H) + (SCALAR ? g : h)) * blocks * 512 + wave * TW * 512;
    const float* kt = c.kt + (q - c.q);
    const float* w = DELTA ? c.w + ah * blocks * 512 + wave * TW * 512 : nullptr;
#pragma unroll
    for (int b = 0; b < TW; ++b)
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        if (DELTA) x.w[b][r] = *(const scan_v4*)(w + b * 512 + r * 256 + lane * 4);
        x.q[b][r] = *(const scan_v4*)(q + b * 512 + r * 256 + lane * 4);
      }
    if (DELTA) {
      const float* vt = c.vt + (ah * vblocks + slice) * 512;
#pragma unroll
      for (int j = 0; j < 2; ++j) x.v[j] = *(const scan_v4*)(vt + j * 256 + lane * 4);
    } else {
      // (beyond the sequence's last token its row again: it is not used)
      const int t0 = ci * C, last = len - 1 - t0;
      const float* v = a.src + (size_t)(first + t0) * a.src_stride + a.v_col + h * a.Dv;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) x.v[j][i] = v[min(16 * j + 4 * gq + i, last) * a.src_stride + vcol];
    }
#pragma unroll
    for (int b = 0; b < TW; ++b)
#pragma unroll
      for (int j = 0; j < 2; ++j) x.kt[b][j] = *(const scan_v4*)(kt + b * 512 + j * 256 + lane * 4);
    if (SCALAR) {
      const float* k = c.keep + ah * (3 * C + 4);
      x.keep[2] = *(const scan_v4*)(k + C + 4 * gq);
      x.keep[3] = *(const scan_v4*)(k + C + 16 + 4 * gq);
      x.keep[4][0] = k[3 * C];
      x.keep[0] = *(const scan_v4*)(k + 16 * (wave & 1) + 4 * gq);
      if (MODE == SCAN_LSTM) x.keep[1] = *(const scan_v4*)(k + 2 * C + 16 * (wave & 1) + 4 * gq);
    } else {
#pragma unroll
      for (int b = 0; b < TW; ++b) x.keep[b] = *(const scan_v4*)(c.keep + ah * c.Dp + 16 * (wave * TW + b) + 4 * gq);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) x.a[j] = *(const scan_v4*)(c.a + ah * 1024 + (wave & 1) * 512 + j * 256 + lane * 4);
  };

  float odd = 0.f;
  auto step = [&](int ci, Chunk& now, auto careful) {
    scan_v4(*buf)[NP][64] = part[ci & 1];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      if (DELTA) {
        scan_v4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < TW; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(now.w[b][r][i], st[b][i], acc, 0, 0, 0);
        buf[wave][2 + r][lane] = acc;
      }
      scan_v4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < TW; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(now.q[b][r][i], st[b][i], acc, 0, 0, 0);
      buf[wave][r][lane] = acc;
    }
    __syncthreads();                                    // (the other half was read before the barrier ahead of this one)
    scan_v4 u[2] = {now.v[0], now.v[1]};
    if (is_n) u[0] = u[1] = scan_v4{1.f, 1.f, 1.f, 1.f};   // (tokens beyond the last: A and the factors of k are 0)
    if (careful && !DELTA) {                            // (the last row again may be infinite, which 0 does not take out)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (ci * C + 16 * j + 4 * gq + i >= len) u[j][i] = 0.f;
    }
    if (DELTA) {
#pragma unroll
      for (int j = 0; j < 2; ++j) u[j] -= (buf[0][2 + j][lane] + buf[1][2 + j][lane]) + (buf[2][2 + j][lane] + buf[3][2 + j][lane]);
    }
    // S' = keep S + k u^T
    scan_v4 us[2] = {u[0], u[1]};
    if (SCALAR) {
      us[0] *= now.keep[2];
      us[1] *= now.keep[3];
    }
#pragma unroll
    for (int b = 0; b < TW; ++b) {
      scan_v4 acc = {0.f, 0.f, 0.f, 0.f};               // (summed up by itself: S sees one rounding a chunk)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(now.kt[b][j][i], us[j][i], acc, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) st[b][i] = fmaf(st[b][i], SCALAR ? now.keep[4][0] : now.keep[b][i], acc[i]);
    }
    if (wave < 2) {                                     // rows 16 wave .. of the read-outs
      scan_v4 o = (buf[0][wave][lane] + buf[1][wave][lane]) + (buf[2][wave][lane] + buf[3][wave][lane]);
      if (SCALAR) o *= now.keep[0];
      scan_v4 own[2] = {};
#pragma unroll
      for (int j = 0; j < 2; ++j)
        if (j <= wave)
#pragma unroll
          for (int i = 0; i < 4; ++i) own[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.a[j][i], u[j][i], own[j], 0, 0, 0);
      if (careful && wave == 0) own[0] = scan_lower_only<true>(now.a[0], u[0], lane);
      if (careful && wave == 1) own[1] = scan_lower_only<true>(now.a[1], u[1], lane);
      o += own[0] + own[1];
      if (!careful) odd = scan_odd(odd, o);
      const int t = ci * C + 16 * wave;
      float* out = a.out + ((size_t)(first + t) * a.H + h) * a.Dv;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v = o[i];
        if (MODE == SCAN_LSTM) v /= fmaxf(fabsf(__shfl(v, 16 * gq + 15, SL_WAVE)), now.keep[1][i]) + 1e-6f;
        if (MODE == SCAN_SSD) v += skip * (wave == 0 ? u[0][i] : u[1][i]);
        if (t + 4 * gq + i < len && live && !is_n) (out + (size_t)i * a.H * a.Dv)[(4 * gq) * a.H * a.Dv + col] = v;
      }
    }
  };
  constexpr int AHEAD = TW <= 2 ? 3 : 2;                // (chunks asked for; a chunk's operands take up to 76 registers at TW 2)
  // (no branch around the loads, also at the end, where the last chunk is asked for again: values that meet behind a
  // branch would be waited for there)
  Chunk ring[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) ask(min(i, nchunks - 1), ring[i]);
  for (int c0 = 0;; c0 += AHEAD) {
    bool done = false;
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      if (c0 + i >= nchunks) {
        done = true;
        break;
      }
      step(c0 + i, ring[i], std::false_type{});
      ask(min(c0 + i + AHEAD, nchunks - 1), ring[i]);
    }
    if (done) break;
  }
  if (wave < 2) {
    const bool any = __ballot(odd != 0.f) != 0;
    if (lane == 0) again[wave] = any;
  }
  __syncthreads();
  if (again[0] || again[1]) {                           // from the start again, a chunk at a time, the read-outs with care
    begin();
#pragma unroll 1
    for (int ci = 0; ci < nchunks; ++ci) {
      ask(ci, ring[0]);
      step(ci, ring[0], std::true_type{});
    }
  }
  if (!a.write || !live) return;
  float* to = srow;
  if (is_n) {                                           // (every slice reads the old n when it starts: see normaliser_kernel)
    if (slice != 0) return;
    to = a.normaliser + ((size_t)s * a.H + h) * (a.D + 1);
    if (wave == 0 && gq == 0) to[a.D] = c.keep[((size_t)(chunk0 + nchunks - 1) * a.H + h) * (3 * C + 4) + 3 * C + 1];
  }
#pragma unroll
  for (int b = 0; b < TW; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 16 * (wave * TW + b) + 4 * gq + i;
      if (d < a.D) to[d] = st[b][i];
    }
}

// Floats of the workspace, laid out in the order of ScanChunks; 0: the heads do not fit this form.
static inline long long scan_chunks_layout(int mode, int T, int S, int H, int G, int D, int Dv, float* base, ScanChunks* out) {
  if (D > 64 * SCAN_MAX_TILES) return 0;
  const bool scalar = mode == SCAN_LSTM || mode == SCAN_SSD || mode == SCAN_DELTA_HEAD;
  const bool delta = mode == SCAN_DELTA || mode == SCAN_DELTA_HEAD;
  const long long chunks = T / SCAN_CHUNK + S, Dp = (D + 63) / 64 * 64, heads = scalar ? G : H;
  long long at = 0;
  auto take = [&](long long n) {
    float* p = base == nullptr ? nullptr : base + at;
    at += (n + 63) / 64 * 64;
    return p;
  };
  ScanChunks c;
  c.Dp = (int)Dp;
  c.q = take(chunks * heads * Dp * SCAN_CHUNK);
  c.kt = take(chunks * heads * Dp * SCAN_CHUNK);
  c.a = take(chunks * H * 1024);
  c.w = delta ? take(chunks * H * Dp * SCAN_CHUNK) : nullptr;
  c.vt = delta ? take(chunks * H * ((Dv + 15) / 16) * 512) : nullptr;
  c.keep = take(scalar ? chunks * H * (3 * SCAN_CHUNK + 4) : chunks * H * Dp);
  c.gates = mode == SCAN_LSTM ? take(chunks * H * (2 * SCAN_CHUNK + 2)) : nullptr;
  if (out != nullptr) *out = c;
  return at;
}

template <int MODE>
static const char* scan_in_chunks(const MatrixScan& a, const ScanChunks& c, int S, int max_len, hipStream_t stream) {
  constexpr bool SCALAR = ScanForm<MODE>::SCALAR, DELTA = ScanForm<MODE>::DELTA;
  const int row = c.Dp + 4, chunks = (max_len + SCAN_CHUNK - 1) / SCAN_CHUNK, square = SCAN_CHUNK * SCAN_AR;
  const size_t floats = SCALAR ? 2 * SCAN_CHUNK * row + (DELTA ? 4 : 2) * square + 4 * SCAN_CHUNK :
      3 * SCAN_CHUNK * row + (DELTA ? 2 : 1) * square + SCAN_CHUNK + max(13 * c.Dp, 4 * SCAN_CHUNK * 8 * (DELTA ? 2 : 1));
  const int lds = (int)(floats * sizeof(float));
  if constexpr (SCALAR) {
    if (lds > 65536) {
      hipError_t e = hipFuncSetAttribute((const void*)scan_prepare_scalar_kernel<MODE>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (e != hipSuccess) return hipGetErrorString(e);
    }
    if (MODE == SCAN_LSTM) scan_gates_kernel<<<dim3(chunks, S), 256, 0, stream>>>(a, c);
    scan_prepare_scalar_kernel<MODE><<<dim3(chunks, a.G, S), 256, lds, stream>>>(a, c);
  } else {
    if (lds > 65536) {
      hipError_t e = hipFuncSetAttribute((const void*)scan_prepare_channel_kernel<MODE>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (e != hipSuccess) return hipGetErrorString(e);
    }
    scan_prepare_channel_kernel<MODE><<<dim3(chunks, a.H, S), 256, lds, stream>>>(a, c);
  }
  const int vcols = MODE == SCAN_LSTM ? 15 : 16, slices = (a.Dv + vcols - 1) / vcols;
  const dim3 grid((unsigned)((long long)(S * a.H + 7) / 8 * 8 * slices));
  const int tiles = c.Dp / 64;
  if (tiles == 1) scan_walk_kernel<MODE, 1><<<grid, 256, 0, stream>>>(a, c, S, slices);
  else if (tiles == 2) scan_walk_kernel<MODE, 2><<<grid, 256, 0, stream>>>(a, c, S, slices);
  else if (tiles == 3) scan_walk_kernel<MODE, 3><<<grid, 256, 0, stream>>>(a, c, S, slices);
  else scan_walk_kernel<MODE, 4><<<grid, 256, 0, stream>>>(a, c, S, slices);
  return nullptr;
}
