// y[M, N] = x[M, K] W[N, K]^T for prompts: both operands row-major, tiles of 64 T rows of x by 256 rows of W, on eight
// wavefronts that stay and walk their tiles (at most a workgroup a CU).  A wavefront owns 32 T rows of x by 64 of W.
//
// What bounds it: power.  The matrix units alone, on random data, run 2.0 PFLOP/s at 2.1 GHz with v_mfma_f32_16x16x32 and
// 1.7 at 1.75 GHz with v_mfma_f32_32x32x16 (2.43 at 2.4 GHz on zeros), so what counts beside the cycles is what else moves.
// A chunk of 64 values of k (2,048 cycles of matrix work for T = 4) takes 2,350 to 2,450 cycles at 1.8 to 1.9 GHz; without
// the loads it takes 2,130, without the LDS reads as well 2,080.  2,048 rows: 37888 x 3584 gated 512 -> 465 us (1.20
// PFLOP/s; 1.30 on another card), 13 us of them the activation, which nothing runs beside, 3584 x 18944 in two shares of K 247 -> 220 us, against sixteen wavefronts of 64 x 64 each, which loaded, read and
// multiplied a chunk in turn behind one barrier.
//
//  - The order of a chunk is laid down instruction by instruction: products of operands that arrived before the last
//    barrier, between them the reads of the operands that come next and the loads two chunks ahead.  Left to itself the
//    compiler reads late and the loads stand in a row in front of the products (2,700 cycles a chunk).  Loads that each
//    wavefront makes at a place of its own cost more in branches than they save (3,400).
//  - The ring: a chunk is two halves of 32 KB (T = 4), first x's first rows and half of W's, then the rest.  A half's operands
//    are read into registers while the half before it is multiplied, and the half four further on is loaded into
//    its slot during the next one; a barrier a half.  Five slots (all of the LDS) gain nothing, nor do four
//    wavefronts of 128 x 128, which read a third less from the LDS.
//  - Consecutive products differ in one operand only (2 % of the power).
//  - The rows of W lie in a tile so that four lanes' results are 64 bytes of a row of y in one store of 16 bytes each, and a gate
//    and its up product are in one lane.
//  - A workgroup's loads run on over the end of its tile, so the next tile starts without waiting for memory.
#pragma once

__device__ __forceinline__ const __bf16* same_in_all_lanes(const __bf16* p) {
  const unsigned long long v = (unsigned long long)p;
  const unsigned long long hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(v >> 32));
  return (const __bf16*)((hi << 32) | (unsigned)__builtin_amdgcn_readfirstlane((int)v));
}
enum { ROUNDS_BF16 = 0, ROUNDS_F32 = 1, ROUNDS_GATED = 2 };            // what is written: KIND; N % 8, 4 and 16 == 0

template <int T, int KIND>
__global__ __launch_bounds__(512, 2) void gemm_rounds_kernel(
    const __bf16* __restrict__ x, const __bf16* __restrict__ w, const float* __restrict__ bias,
    void* __restrict__ y, int M, int N, int K, int act, int KS) {
  constexpr int T0 = (T + 1) / 2, T1 = T / 2, BM = 64 * T, BN = 256;   // halves of the tile: 64 T0 and 64 T1 rows of x, 128 of W
  constexpr int SLOT = 8192 * (T0 + 2), SLOTS = T == 2 ? 6 : 4;
  constexpr int HALF0 = T0 + 2, HALF1 = T1 + 2;                        // loads a wavefront makes of a half
  constexpr int AHEAD = (HALF0 + HALF1) * (SLOTS - 2) / 2;             // that are younger than those of the half read next
  __shared__ __attribute__((aligned(1024))) char ring[SLOTS * SLOT];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  // chiplet c takes a contiguous eighth of the (share, column tile, row tile) items, row tiles fastest, so that the
  // workgroups of a round that read the same rows share an L2; a workgroup takes every `step`-th of its chiplet's
  const int gx = (N + BN - 1) / BN, gy = (M + BM - 1) / BM, total = gx * gy * KS;
  const int per = (total + 7) / 8, first = (int)(blockIdx.x & 7) * per, step = (int)gridDim.x >> 3;
  const int end = first + per < total ? first + per : total;
  int item = first + (int)(blockIdx.x >> 3);
  if (item >= end) return;                                             // (the whole workgroup)
  const int chunks = K / 64;
  const unsigned ring_at = (unsigned)(size_t)(__attribute__((address_space(3))) char*)ring + 1024 * wave;

  // what is loaded next: the item, its chunks left, where they lie, and this lane's rows of it
  int load_item = item, load_left;
  const __bf16 *load_x, *load_w;
  unsigned at_x[T], at_w[4];
  auto open = [&](int it) {
    const int share = it / (gx * gy), m0 = it % gy * BM, n0 = it / gy % gx * BN;
    const int c0 = chunks * share / KS;
    load_left = __builtin_amdgcn_readfirstlane(chunks * (share + 1) / KS - c0);
    load_x = same_in_all_lanes(x + (size_t)m0 * K + 64 * (size_t)c0);
    load_w = same_in_all_lanes(w + (size_t)n0 * K + 64 * (size_t)c0);
    const int last_m = M - m0 - 1, last_n = N - n0 - 1, lane = lane_here();      // rows past the end: the last one again
#pragma unroll
    for (int j = 0; j < T; ++j) {
      const int r = 8 * (wave + 8 * j) + (lane >> 3);
      at_x[j] = (unsigned)(r < last_m ? r : last_m) * (unsigned)(2 * K) + 16 * ((lane & 7) ^ lds_place(r));
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {          // row s of half j / 2: tile u of a wavefront's four, row r of the matrix instruction
      const int s = 8 * (wave + 8 * (j & 1)) + (lane >> 3), r = s & 15, u = 2 * (j >> 1) + (s >> 4 & 1);
      const int n = 64 * (s >> 5) + (KIND == ROUNDS_GATED ? 16 * (r >> 2) + 4 * u + (r & 3)
                                     : KIND == ROUNDS_BF16 ? 32 * (u >> 1) + 8 * (r >> 2) + 4 * (u & 1) + (r & 3) : 16 * u + r);
      at_w[j] = (unsigned)(n < last_n ? n : last_n) * (unsigned)(2 * K) + 16 * ((lane & 7) ^ lds_place(s));
    }
  };
  auto load = [&](int half, int j, unsigned slot) {
    const int nx = half ? T1 : T0;
    if (j < nx) load_to_lds(at_x[(half ? T0 : 0) + j], load_x, slot + 8192 * j);
    else load_to_lds(at_w[2 * half + j - nx], load_w, slot + 8192 * (T0 + j - nx));
  };
  auto advance = [&]() {
    if (--load_left > 0) {
      load_x += 64;
      load_w += 64;
    } else if (load_item + step < end) {
      load_item += step;
      open(load_item);
    }                                      // (past the last chunk: that one again, which nothing reads)
  };
  auto barrier = [&]() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
  };
  open(item);
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
#pragma unroll
    for (int j = 0; j < (s & 1 ? HALF1 : HALF0); ++j) load(s & 1, j, ring_at + SLOT * s);
    if (s & 1) advance();
  }
  bf16x8 x0[2 * T0][2], x1[2 * T1][2], w0[2][2], w1[2][2];             // [tile of 16 rows][k-step of 32]
  f32x4 acc[2 * T][4];
#pragma unroll
  for (int a = 0; a < 2 * T; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  int at_x0[2], at_x1[2], at_wt[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const int lane = threadIdx.x & 63, i = lane & 15;
    const int at = 128 * i + 16 * ((4 * kk + (lane >> 4)) ^ lds_place(i));
    at_x0[kk] = at + 4096 * T0 * wm;
    at_x1[kk] = at + 4096 * T1 * wm;
    at_wt[kk] = at + 4096 * wn + 8192 * T0;
  }
  auto operand = [&](int at) { return *(const bf16x8*)(ring + at); };
  wait_loads<AHEAD + HALF1>();
  barrier();
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
    for (int b = 0; b < 2; ++b) w0[b][kk] = operand(at_wt[kk] + 2048 * b);
#pragma unroll
    for (int a = 0; a < 2 * T0; ++a) x0[a][kk] = operand(at_x0[kk] + 2048 * a);
  }
  asm volatile("" : : : "memory");
  wait_loads<AHEAD>();
  barrier();
  int read_at = SLOT;                      // slot of the half that is read next
  unsigned load_at = 0;                    // slot of the half that is loaded next: the one read before
  auto next = [&](unsigned at) { return at == SLOT * (SLOTS - 1) ? 0u : at + SLOT; };

  while (true) {
    const int share = item / (gx * gy), m0 = item % gy * BM, n0 = item / gy % gx * BN;
    const int tile_chunks = __builtin_amdgcn_readfirstlane(chunks * (share + 1) / KS - chunks * share / KS);
    for (int c = 0; c < tile_chunks; ++c) {
      // x's first rows; the second halves of x and W arrive in registers, the first of the chunk after next in the ring
      constexpr int P0 = 16 * T0, R0 = 4 + 4 * T1;                     // products, reads
#pragma unroll
      for (int i = 0; i < P0; ++i) {
#pragma unroll
        for (int r = 0; r < R0; ++r) {
          if (r * (P0 * 3 / 4) / R0 != i) continue;
          const int q = r - 4;
          if (r < 4) w1[r & 1][r >> 1] = operand(at_wt[r >> 1] + read_at + 2048 * (r & 1));
          else x1[q % (2 * T1)][q / (2 * T1)] = operand(at_x1[q / (2 * T1)] + read_at + 2048 * (q % (2 * T1)));
        }
#pragma unroll
        for (int j = 0; j < HALF0; ++j)
          if (j * P0 / HALF0 == i) load(0, j, ring_at + load_at);
        const int h = i / (8 * T0), j = i % (8 * T0), kk = j / (4 * T0), a = j / 2 % (2 * T0), b = (j ^ a) & 1;
        acc[a][2 * h + b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h ? w1[b][kk] : w0[b][kk], x0[a][kk], acc[a][2 * h + b], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("" : : : "memory");
      wait_loads<AHEAD>();         // the half that is read next is there: of the loads, one of each half is younger
      barrier();
      read_at = next(read_at);
      load_at = next(load_at);
      // x's second rows; the first halves of the next chunk arrive
      constexpr int P1 = 16 * T1, R1 = 4 * T0;
#pragma unroll
      for (int i = 0; i < P1; ++i) {
#pragma unroll
        for (int r = 0; r < R1; ++r)
          if (r * (P1 / 2) / R1 == i) x0[r % (2 * T0)][r / (2 * T0)] = operand(at_x0[r / (2 * T0)] + read_at + 2048 * (r % (2 * T0)));
#pragma unroll
        for (int r = 0; r < 4; ++r)        // (their first half's products are done)
          if (P1 / 2 + r * (P1 / 4) / 4 == i) w0[r & 1][r >> 1] = operand(at_wt[r >> 1] + read_at + 2048 * (r & 1));
#pragma unroll
        for (int j = 0; j < HALF1; ++j)
          if (j * P1 / HALF1 == i) load(1, j, ring_at + load_at);
        const int h = i / (8 * T1), j = i % (8 * T1), kk = j / (4 * T1), a = j / 2 % (2 * T1), b = (j ^ a) & 1;
        acc[2 * T0 + a][2 * h + b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h ? w1[b][kk] : w0[b][kk], x1[a][kk], acc[2 * T0 + a][2 * h + b], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("" : : : "memory");
      wait_loads<AHEAD>();
      barrier();
      read_at = next(read_at);
      load_at = next(load_at);
      advance();
    }

    // lane: row m of x; of tile b the four rows of W from column(b) on
    const int lane = lane_here(), g = lane >> 4, nw = n0 + 64 * wn;
    auto column = [&](int b) {
      return nw + (KIND == ROUNDS_GATED ? 16 * g + 4 * b : KIND == ROUNDS_BF16 ? 32 * (b >> 1) + 8 * g + 4 * (b & 1) : 16 * b + 4 * g);
    };
#pragma unroll
    for (int a = 0; a < 2 * T; ++a) {
      const int m = m0 + (a < 2 * T0 ? 32 * T0 * wm + 16 * a : 64 * T0 + 32 * T1 * wm + 16 * (a - 2 * T0)) + (lane & 15);
      f32x4 r[4];
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        r[b] = acc[a][b];
        acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (bias != nullptr) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (column(b) < N) r[b][e] += bias[column(b) + e];
        }
      }
      if (m >= M) continue;
      if constexpr (KIND == ROUNDS_GATED) {
        const int n = column(0);
        bf16x8 h;                          // (gate and up rows lie in blocks of eight: gates first, then their ups)
        if (act == SL_ACT_SILU) {
#pragma unroll
          for (int e = 0; e < 8; ++e) h[e] = (__bf16)(sl_act(r[e >> 2][e & 3], SL_ACT_SILU) * r[2 + (e >> 2)][e & 3]);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) h[e] = (__bf16)(sl_act(r[e >> 2][e & 3], act) * r[2 + (e >> 2)][e & 3]);
        }
        if (n < N) *(bf16x8*)((__bf16*)y + (size_t)m * (N / 2) + n / 2) = h;
      } else if constexpr (KIND == ROUNDS_F32) {
        float* o = (float*)y + ((size_t)share * M + m) * N;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int n = column(b);
          if (n < N) *(f32x4*)(o + n) = r[b];
        }
      } else {
        __bf16* o = (__bf16*)y + (size_t)m * N;
        if (act) {
#pragma unroll
          for (int e = 0; e < 16; ++e) r[e >> 2][e & 3] = sl_act(r[e >> 2][e & 3], act);
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int n = column(2 * p);
          bf16x8 h;
#pragma unroll
          for (int e = 0; e < 8; ++e) h[e] = (__bf16)r[2 * p + (e >> 2)][e & 3];
          if (n < N) *(bf16x8*)(o + n) = h;
        }
      }
    }
    item += step;
    if (item >= end) break;
  }
  wait_loads<0>();                         // (loads past the last chunk still land in this workgroup's LDS)
}
