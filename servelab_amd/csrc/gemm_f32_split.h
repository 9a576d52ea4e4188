// Float32 products of more than 64 rows on the bfloat16 matrix units: y[M, N] = x[M, K] W[N, K]^T, K % 32 == 0.  Included by gemm.hip.
//
// An operand is three bfloat16 terms, each what the ones before left over, rounded to nearest: 8 + 8 + 8 bits of significand, so
// that together they are the float itself.  They are terms of 2^24 times the operand, or what they leave of one below 2^-109 would lie below
// bfloat16's least value (left at its size, an operand of 2^-116 was 2^-19 off and one of 2^-135 gone).  A product is the
// six products of terms down to 2^-18 of it; the three left out are at most 2^-26 of it together, a quarter of a float's rounding.
// Products of bfloat16 are exact in float, and a matrix instruction adds 32 of them to the running sum at once.  It rounds that sum down,
// not to nearest: left so, every result lay 5e-8 to 6e-7 of their spread too low, and the logits of a 6-layer model 3.1e-6 off
// instead of 2.8e-6.  Hence runs of chunks are summed apart, every other one with x's sign turned, whose sums are
// subtracted; runs of either sign are equally many and long, or but one chunk.  Mean offset of two million results, in their spread, no more
// than that of float32 instructions, 3e-10 (an odd number of chunks: 4e-10 at 544 values of k); with runs of 8 chunks at every k
// 8.0e-9 at 768, 6.1e-9 at 1,280, 4.6e-9 at 896.  Error of a result against 64 bits 2.4e-7 to 2.6e-7 for 3.7e-7 to 4.1e-7 with float32 instructions
// and sums of 512 terms, of those logits 2.4e-6 for 2.9e-6.
// A result that is not finite, as a sum of 2^48 times itself, is worked out again by float32 instructions: an infinite operand's rests are NaN.
//
// Bound by the matrix units, six instructions of 16 cycles in the place of eight of 32 (16 x 16 results, 32 terms), and their power:
// 2.3 us a chunk of 32 k on all CUs, 1.9 on one.  A workgroup of eight wavefronts, one a CU, owns 128 rows of x by 256 of W, a
// wavefront 64 x 64.  A chunk goes from memory to registers, is split there once for the workgroup, and lies in LDS as three planes of
// rows of 64 bytes (a wavefront's read of an operand is 1 KB in a row); two stages.  The order of a chunk is laid down
// instruction by instruction: left to itself the compiler converts in front of all products and loads behind them (294 us
// below, 272 laid down).  A lane stores its four results at once (one by one 266 products
// took 1.13 times as long, 2,048 rows of 8192 x 256 115 us instead of 56).  849 rows, 17920 x 1536 444 -> 272 us (172 TFLOP/s), 1536 x 8960 in six shares 205 -> 128; 2,048 rows, 37888 x
// 3584 4,380 -> 2,620 (212); 266 products of 65 to 2,048 rows take 0.72 of the time on average, 0.97 at worst, against
// v_mfma_f32_32x32x2_f32.
#pragma once
#include <utility>

typedef __bf16 split_bf16x8 __attribute__((ext_vector_type(8)));
typedef float split_f32x4 __attribute__((ext_vector_type(4)));
typedef float split_f32x4_at_4 __attribute__((ext_vector_type(4), aligned(4)));
typedef float split_f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 split_bf16x2 __attribute__((ext_vector_type(2)));

// Eight floats as three bfloat16 each, v = t0 + t1 + t2: every term is what the ones before left over, rounded to nearest.
__device__ __forceinline__ void split_terms(const split_f32x4 (&v)[2], split_bf16x8 (&t)[3]) {
  unsigned u[3][4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    split_f32x2 r = {v[e >> 1][2 * (e & 1)], v[e >> 1][2 * (e & 1) + 1]};
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      u[p][e] = __builtin_bit_cast(unsigned, __builtin_convertvector(r, split_bf16x2));
      if (p < 2) {
        r[0] -= __uint_as_float(u[p][e] << 16);
        r[1] -= __uint_as_float(u[p][e] & 0xffff0000u);
      }
    }
  }
#pragma unroll
  for (int p = 0; p < 3; ++p) __builtin_memcpy(&t[p], u[p], 16);
}

// f(0), f(1), ..: each with its number as a constant.
template <class F, int... I> __device__ __forceinline__ void in_order(F f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F> __device__ __forceinline__ void in_order(F f) { in_order(f, std::make_integer_sequence<int, N>{}); }

// B: tiles of 16 columns a wavefront takes, 4 or 2: a workgroup 256 columns or 128.
template <int B, bool SHARES>
__global__ __launch_bounds__(512, 2) void gemm_f32_split_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    float* __restrict__ y, int M, int N, int K, int nsplit) {
  constexpr int BM = 128, BN = 64 * B, CK = 32, ITEMS = 1 + B / 2, ROWS = BM + BN, PLANE = ROWS * 64, STAGE = 3 * PLANE;
  __shared__ __attribute__((aligned(1024))) char stages[2 * STAGE];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6), wm = wave >> 2, wn = wave & 3;
  // a chiplet takes a contiguous eighth of the (share, column tile, row tile) triples, row tiles fastest
  const int gx = (N + BN - 1) / BN, gy = (M + BM - 1) / BM, total = gx * gy * nsplit, per = (total + 7) / 8;
  const int triple = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || triple >= total) return;        // (the whole workgroup)
  const int share = triple / (gx * gy), m0 = triple % gy * BM, n0 = triple / gy % gx * BN;
  constexpr int SEG = SEGMENT_K / CK;
  const int chunks = K / CK, segs = (chunks + SEG - 1) / SEG;
  const int first = SHARES ? (int)((unsigned)segs * share / (unsigned)nsplit) * SEG : 0;
  const int behind = SHARES ? (int)((unsigned)segs * (share + 1) / (unsigned)nsplit) * SEG : segs * SEG;
  const int last = behind < chunks ? behind : chunks;
  if (SHARES) {
    y += (size_t)share * M * N;
    bias = nullptr;
  }
  // what this thread brings of every chunk: eight values of k, t % 4, of rows t / 4 + 128 j; rows past the end: the last
  const float* src[ITEMS];
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    const int r = (t >> 2) + 128 * j;
    src[j] = (j == 0 ? x + (size_t)(m0 + r < M ? m0 + r : M - 1) * K : w + (size_t)(n0 + r - BM < N ? n0 + r - BM : N - 1) * K) +
             8 * (t & 3) + CK * (size_t)first;
  }
  split_f32x4 v[ITEMS][2];
  auto load = [&](int j) {
    v[j][0] = *(const split_f32x4*)src[j];
    v[j][1] = *(const split_f32x4*)(src[j] + 4);
    src[j] += CK;
  };
  // Runs of RUN chunks, every other one multiplied with -x, from the first on; the chunks behind the last pair of such runs make a
  // pair of half as many each, an odd one at the end a run of its own.
  constexpr int RUN = 8;
  const int paired = first + (last - first) / (2 * RUN) * (2 * RUN), half = (last - paired) / 2;
  auto run_end = [&](int c) { return c < paired ? c + RUN : c < paired + half ? paired + half : c < paired + 2 * half ? paired + 2 * half : last; };
  constexpr float SCALE = 1 << 24;
  auto store = [&](int stage, int j) {
    split_bf16x8 terms[3];
    const float scale = j == 0 ? -SCALE : SCALE;
    v[j][0] *= scale, v[j][1] *= scale;
    split_terms(v[j], terms);
#pragma unroll
    for (int p = 0; p < 3; ++p) *(split_bf16x8*)(stages + stage * STAGE + p * PLANE + 8192 * j + 16 * t) = terms[p];
  };
  split_f32x4 acc[4][B], sum[4][B];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < B; ++b) acc[a][b] = sum[a][b] = split_f32x4{0.f, 0.f, 0.f, 0.f};
  const int at = 64 * (lane & 15) + 16 * (lane >> 4), x_at = at + 4096 * wm, w_at = at + 64 * BM + 1024 * B * wn;
  int asked = first;                                   // chunks asked for; past the last one that one again
  auto ask = [&](int j) {
    load(j);
    if (asked + 1 >= last) src[j] -= CK;
  };
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) ask(j);
  ++asked;
#pragma unroll
  for (int j = 0; j < ITEMS; ++j) {
    store(0, j);
    ask(j);
  }
  ++asked;
  __syncthreads();
  int c = first, stage = 0;
  for (float sign = -1.f; c < last; sign = -sign) {
    const int c1 = run_end(c);
    for (; c < c1; ++c, stage ^= 1) {
      const char* from = stages + stage * STAGE;
      char* to = stages + (stage ^ 1) * STAGE + 16 * t;
      split_bf16x8 x0[4], x1[4], w0[B], w1[B];
      auto read = [&](int p, int where, int a) { return *(const split_bf16x8*)(from + p * PLANE + where + 1024 * a); };
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        if (a < B) w0[a] = read(0, w_at, a);
        x0[a] = read(0, x_at, a);
      }
      constexpr int P = 24 * B, S = 12 * ITEMS, S0 = 3 * B / 2, SPAN = P - 2 * B;      // products; steps of the conversion, the first one's place
      const float scale_next = c + 1 < c1 ? SCALE * sign : -SCALE * sign;
      unsigned u[3][4];
      split_f32x2 r;
      in_order<P>([&](auto slot) __attribute__((always_inline)) {
        constexpr int i = decltype(slot)::value;
        // products of the terms: 0 0, 0 1, 1 1, 1 0, 0 2, 2 0 of x and W; the third terms take the second ones' registers
        constexpr int part = i / (4 * B), a = i / B % 4, b = a & 1 ? B - 1 - i % B : i % B;
        if constexpr (i < B) w1[i] = read(1, w_at, i);
        if constexpr (i >= 4 * B && i < 4 * B + 4) x1[i - 4 * B] = read(1, x_at, i - 4 * B);
        if constexpr (i >= 12 * B && i < 13 * B) w1[i - 12 * B] = read(2, w_at, i - 12 * B);
        if constexpr (i >= 16 * B && i < 16 * B + 4) x1[i - 16 * B] = read(2, x_at, i - 16 * B);
        constexpr int s = (S * (i - S0) + SPAN - 1) / SPAN;              // the next chunk's conversion: item s / 12, pair s / 3 % 4, term s % 3
        if constexpr (i >= S0 && s < S && S0 + s * SPAN / S == i) {
          constexpr int q = s / 12, e = s / 3 % 4, p = s % 3;
          if constexpr (p == 0) {
            r = split_f32x2{v[q][e >> 1][2 * (e & 1)], v[q][e >> 1][2 * (e & 1) + 1]};
            r *= q == 0 ? scale_next : SCALE;
          }
          u[p][e] = __builtin_bit_cast(unsigned, __builtin_convertvector(r, split_bf16x2));
          if constexpr (p < 2) {
            r[0] -= __uint_as_float(u[p][e] << 16);
            r[1] -= __uint_as_float(u[p][e] & 0xffff0000u);
          }
          if constexpr (e == 3) __builtin_memcpy(to + p * PLANE + 8192 * q, u[p], 16);
          if constexpr (e == 3 && p == 2) ask(q);
        }
        const split_bf16x8 xv = part == 0 || part == 1 || part == 4 ? x0[a] : x1[a], wv = part == 0 || part == 3 || part == 5 ? w0[b] : w1[b];
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, xv, acc[a][b], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      });
      ++asked;
      __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < B; ++b) {
        sum[a][b] += sign * acc[a][b];
        acc[a][b] = split_f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
  // lane: row lane % 16 of x's tile, four rows of W's from 4 (lane / 16) on
  unsigned long long again = 0;                        // bit 4 (B a + b) + e: a result that is not finite
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int m = m0 + 64 * wm + 16 * a + (lane & 15);
    if (m >= M) continue;
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int n = n0 + 16 * B * wn + 16 * b + 4 * (lane >> 4);
      if (n >= N) continue;
      split_f32x4 s = sum[a][b] * (1 / (SCALE * SCALE));
      unsigned odd = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        odd |= fabsf(s[e]) < INFINITY ? 0u : 1u << e;
        if (bias != nullptr) s[e] += bias[n + e < N ? n + e : N - 1];
      }
      float* to = y + (size_t)m * N + n;
      if (odd == 0 && n + 4 <= N) {
        *(split_f32x4_at_4*)to = s;                    // (one store: rows of 64 to 256 values are bound by them)
        continue;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N && !(odd >> e & 1)) to[e] = s[e];
      again |= (unsigned long long)(n + 4 <= N ? odd : odd & ((1u << (N - n)) - 1)) << 4 * (B * a + b);
    }
  }
  // An operand that is not finite, or 2^24 times it beyond the largest bfloat16, or a sum past 2^80: by float32 instructions and sums of
  // SEGMENT_K terms.  Sixteen rows of x at a time; what is finite beside them stays.
  for (int a = 0; a < 4; ++a) {
    const unsigned row = (unsigned)(again >> (4 * B * a)) & ((1u << 4 * B) - 1);
    if (__builtin_amdgcn_ballot_w64(row != 0) == 0) continue;          // (the whole wavefront)
    const int mine = m0 + 64 * wm + 16 * a + (lane & 15), wrow = n0 + 16 * B * wn + (lane & 15);
    const float *xr = x + (size_t)min(mine, M - 1) * K + 4 * (lane >> 4), *wr[B];
#pragma unroll
    for (int b = 0; b < B; ++b) wr[b] = w + (size_t)min(wrow + 16 * b, N - 1) * K + 4 * (lane >> 4);
    split_f32x4 total[B], part[B];
#pragma unroll
    for (int b = 0; b < B; ++b) total[b] = part[b] = split_f32x4{0.f, 0.f, 0.f, 0.f};
    for (int k = CK * first; k < CK * last; k += CK) {
      split_f32x4 xv[2], wv[2][B];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        xv[u] = *(const split_f32x4*)(xr + k + 16 * u);
#pragma unroll
        for (int b = 0; b < B; ++b) wv[u][b] = *(const split_f32x4*)(wr[b] + k + 16 * u);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int b = 0; b < B; ++b) part[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[u][b][j], xv[u][j], part[b], 0, 0, 0);
      if ((k + CK) % SEGMENT_K != 0 && k + CK < CK * last) continue;
#pragma unroll
      for (int b = 0; b < B; ++b) {
        total[b] += part[b];
        part[b] = split_f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int n = n0 + 16 * B * wn + 16 * b + 4 * (lane >> 4);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (row >> (4 * b + e) & 1) y[(size_t)mine * N + n + e] = total[b][e] + (bias != nullptr ? bias[n + e] : 0.f);
    }
  }
}
