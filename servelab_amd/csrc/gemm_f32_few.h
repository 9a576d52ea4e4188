#pragma once

// y[M, N] = x[M, K] W[N, K]^T + bias, float32, three to sixteen rows of x; K % 4 == 0.
//
// Bound by the stream of W from memory.  v_mfma_f32_4x4x1_16b_f32 is sixteen products of four columns by four rows side by side, each of
// values of k of its own: a lane takes 16 bytes of one row of W and of one row of x (lane 4 b + i: row i, values 4 b .. + 3 of a step of
// 64), a load is 256 bytes in a row of four rows, and what multiplies lies where it was loaded.  One such product takes eight
// cycles for the 256 bytes of W that meet four rows of x; as FMAs, three rows took 27 us of 17920 x 1536 and sixteen 62.
//  - A wavefront owns 4 C columns, whose loads of x it shares, and one of KW parts of K; U steps' loads are asked for together, in front of
//    their products (a barrier of the scheduler holds them there), W past the caches: a model reads every matrix once a step.
//  - Running sums: sixteen blocks, KW parts and E of the four values of a step apart, so that each is as short as in FMAs of a
//    wavefront or four (64 or 256 sums of K / 64 or K / 256 terms): the error against 64 bits stays what it was, 0.9 to 1.2e-7 of a result, or
//    shrinks (16 rows of 3584 x 18944 3.2e-7 -> 1.8e-7).
// us with FMAs / here (matrices in turn, 1.3 GB in all): 17920 x 1536 at 3 / 5 / 16 rows 27 / 37 / 62 -> 22 / 27 / 43; 1536 x 8960 16 / 22 / 94 -> 16
// / 20 / 31; 1536 x 1536 5.5 / 8.0 / 27 -> 5.3 / 6.3 / 8.7; 151936 x 1536 167 / 196 / 338 -> 152 / 159 / 291 (6.1 TB/s at three rows); 896 x 4864 8.1 / 11 / 53
// -> 7.9 / 8.8 / 15; 3584 x 18944 58 / 78 / 186 -> 50 / 57 / 84.
template <int MB, int C, int KW, int U, int E>
__global__ __launch_bounds__(KW == 8 ? 512 : 256) void gemm_f32_few_kernel(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, float* __restrict__ y, int M, int N, int K) {
  typedef float few_v4 __attribute__((ext_vector_type(4)));
  constexpr int WAVES = KW == 8 ? 8 : 4, G = WAVES / KW;  // wavefronts, and their groups of columns
  static_assert(KW > 1 && WAVES % KW == 0 && (E == 1 || E == 2 || E == 4), "parts of K among a workgroup's wavefronts");
  __shared__ few_v4 part[WAVES][MB * C][4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), kw = wave % KW;
  const int i = lane & 3, b = lane >> 2, n0 = (blockIdx.x * G + wave / KW) * 4 * C;
  const int steps = (K + 63) / 64, s1 = steps * (kw + 1) / KW, whole = min(s1, K / 64);
  few_v4 sums[E][MB][C];
#pragma unroll
  for (int e = 0; e < E; ++e)
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int c = 0; c < C; ++c) sums[e][m][c] = few_v4{0.f, 0.f, 0.f, 0.f};
  const float *wr[C], *xr[MB];                            // (rows past the last: that one again, never stored)
#pragma unroll
  for (int c = 0; c < C; ++c) wr[c] = w + (size_t)min(n0 + 4 * c + i, N - 1) * K + 4 * b;
#pragma unroll
  for (int m = 0; m < MB; ++m) xr[m] = x + (size_t)min(4 * m + i, M - 1) * K + 4 * b;
  auto trip = [&](int s, auto count, auto last) {         // last: a step that may end past K, whose lanes there read the row's start
    constexpr int T = decltype(count)::value;
    few_v4 wv[T][C], xv[T][MB];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int at = decltype(last)::value && 64 * (s + t) + 4 * b >= K ? -4 * b : 64 * (s + t);
#pragma unroll
      for (int c = 0; c < C; ++c) wv[t][c] = __builtin_nontemporal_load((const few_v4*)(wr[c] + at));
#pragma unroll
      for (int m = 0; m < MB; ++m) xv[t][m] = *(const few_v4*)(xr[m] + at);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (decltype(last)::value && 64 * s + 4 * b >= K) {
#pragma unroll
      for (int c = 0; c < C; ++c) wv[0][c] = few_v4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < MB; ++m) xv[0][m] = few_v4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
          for (int c = 0; c < C; ++c)
            sums[e % E][m][c] = __builtin_amdgcn_mfma_f32_4x4x1f32(wv[t][c][e], xv[t][m][e], sums[e % E][m][c], 0, 0, 0);
  };
  int s = steps * kw / KW;
  for (; s + U <= whole; s += U) trip(s, std::integral_constant<int, U>{}, std::false_type{});
  if constexpr (U > 2)
    for (; s + 2 <= whole; s += 2) trip(s, std::integral_constant<int, 2>{}, std::false_type{});
  for (; s < s1; ++s) trip(s, std::integral_constant<int, 1>{}, std::true_type{});
  // the blocks' sums: lane i of four holds columns n0 + 4 c .. + 3 of row 4 m + i
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int c = 0; c < C; ++c) {
      few_v4 v;
      if constexpr (E == 4) v = (sums[0][m][c] + sums[1][m][c]) + (sums[2][m][c] + sums[3][m][c]);
      else if constexpr (E == 2) v = sums[0][m][c] + sums[1][m][c];
      else v = sums[0][m][c];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float s = v[e];
        s += lane_xor<4>(s);
        s += lane_xor<8>(s);
        v[e] = column_meet(s, add_f);
      }
      if (lane < 4) part[wave][m * C + c][lane] = v;
    }
  __syncthreads();
  for (int q = threadIdx.x; q < G * MB * C * 4; q += 64 * WAVES) {
    const int g = q / (MB * C * 4), mc = q / 4 % (MB * C), row = 4 * (mc / C) + q % 4, n = (blockIdx.x * G + g) * 4 * C + 4 * (mc % C);
    few_v4 v = part[g * KW][mc][q % 4];
#pragma unroll
    for (int k = 1; k < KW; ++k) v += part[g * KW + k][mc][q % 4];
    if (row >= M) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) y[(size_t)row * N + n + e] = v[e] + (bias != nullptr ? bias[n + e] : 0.f);
  }
}

// Which of them, measured for 37 matrices of 64 to 151,936 rows and rows of 64 to 18,944 values: of few columns a wavefront takes four or
// eight, so that every CU has some; of long rows eight wavefronts share K, and of more than 2,048 such columns each takes sixteen (3584 x 18944 at 3 / 16 rows
// in eight 57 / 111 us, in sixteen 50 / 84; up to eight rows of 2560 x 3072 and 4096 x 4096 sixteen lose up to 7 %), of up to 1,024 four (1024 x 4096 at 3 / 8
// rows in eight 8.2 / 10.9, in four 6.4 / 8.5); up to four rows of up to 768 columns, from 512 values on, eight wavefronts as well (128 x 896 3.7 -> 3.3, 128 x 2560 4.8 ->
// 4.7); of many columns 8 or 16 read a load of x, and of very many two
// wavefronts share K (151936 x 896 at three rows 104 us for 91, 17920 x 1536 21 for 22).
template <int MB>
static void gemm_f32_few(const float* x, const float* w, const float* bias, float* y, int M, int N, int K, hipStream_t stream) {
#define SL_FEW(C, KW, U, E)                                                                                                      \
  gemm_f32_few_kernel<MB, C, KW, U, E>                                                                                           \
      <<<(unsigned)((N + 4 * C * (KW == 2 ? 2 : 1) - 1) / (4 * C * (KW == 2 ? 2 : 1))), KW == 8 ? 512 : 256, 0, stream>>>(x, w, bias, y, M, N, K)
  const bool few = N <= 4096, lengthy = K >= 3072;
  if constexpr (MB <= 2) {
    if (few && lengthy && N <= 1024) SL_FEW(1, 8, 2, 4);
    else if (few && lengthy && (N <= 2048 || K < 8192)) SL_FEW(2, 8, 2, 4);
    else if (few && lengthy) SL_FEW(4, 8, 2, 4);
    else if (MB == 1 && N <= 768 && K >= 512) SL_FEW(1, 8, 4, 4);
    else if (few) SL_FEW(1, 4, 4, 4);
    else if (N <= 32768) SL_FEW(2, 4, 4, (MB == 1 ? 4 : 2));
    else if constexpr (MB == 1) {
      if (K <= 2048) SL_FEW(2, 2, 4, 4);
      else SL_FEW(2, 4, 4, 4);
    } else SL_FEW(4, 2, 2, 2);
  } else {
    if (few && lengthy && N <= 1024) SL_FEW(1, 8, 2, 2);
    else if (few && lengthy && N <= 2048) SL_FEW(2, 8, 2, 2);
    else if (few && lengthy) SL_FEW(4, 8, 2, 2);
    else if (N <= 16384) SL_FEW(2, 4, 2, 1);
    else SL_FEW(4, 4, 2, 1);
  }
#undef SL_FEW
}
