#pragma once

enum { EVEN_BF16 = 0, EVEN_F32 = 1 };                                  // what is written; N % 4 == 0

// y[M, N] = x[M, K] W[N, K]^T for prompts and matrices of few rows (q/k/v, o): x row-major, W in the tiled layout (sl_tile_weight),
// K % 64 == 0.  A workgroup owns 128 rows of x by 32 B of W, with B from 3 to 7 so that the tiles go round the CUs evenly, once at best
// (HipOps._even_columns): 2,048 rows of 3584 x 3584 are 112 tiles of 256 x 256 and 256 of 128 x 224.
//
// Bound by what a CU pulls, 50 to 60 KB a us of tiles whose W comes from memory (73 to 94 out of the caches): 128 x 224 at 2,048 rows of
// 3584 x 18944 take 134 us without their loads (2.07 PFLOP/s), 212 with them.  So W comes in its tiled copy, 2 KB in a row
// a tile of 16 rows and chunk; out of the rows, 128 bytes each, 225 (2048 x 11008 111, here 95).
// us, the library / here: 2,048 rows of 2048 x 2048 22.5 / 20.3, 3584 x 3584 52 / 48; 527 rows of 4608 x 3584 30 / 25.
//  - Four wavefronts: two halves of the columns, two of every chunk's k, so that a wavefront has 128 rows by 16 B columns and reads
//    8 + B operands of the LDS for 8 B products; the halves' sums meet at the end through the LDS.
//  - The accumulators are 32 B registers of 512: they are named as accumulation registers in the instruction, or the compiler
//    moves them to and fro (2,048 x 2,048 x 2,048 26 us instead of 20).
//  - A ring of three to six chunks; the next chunk's operands are read into registers while one is multiplied; the order is laid down.
template <int B, int KIND>
__global__ __launch_bounds__(256, 1) void gemm_even_kernel(
    const __bf16* __restrict__ x, const __bf16* __restrict__ wt, const float* __restrict__ bias,
    void* __restrict__ y, int M, int N, int K) {
  constexpr int BM = 128, BN = 32 * B, ROWS = BM + BN, SLOT = 128 * ROWS;
  constexpr int SLOTS = 160 * 1024 / SLOT < 6 ? 160 * 1024 / SLOT : 6;
  constexpr int LOADS = 4 + B;                                         // of a wavefront for a chunk
  constexpr int P = 8 * B, R = 8 + B;                                  // products and reads of a wavefront for a chunk
  static_assert(16384 * B <= SLOT * SLOTS, "the exchanged sums fit the ring");
  __shared__ __attribute__((aligned(1024))) char ring[SLOTS * SLOT];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), wn = wave & 1, wk = wave >> 1;
  const int gx = (N + BN - 1) / BN, gy = (M + BM - 1) / BM, total = gx * gy, per = (total + 7) / 8;
  const int item = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (item >= total || (int)(blockIdx.x >> 3) >= per) return;          // (the whole workgroup)
  const int panel = item / (8 * gx), in_panel = gy - 8 * panel < 8 ? gy - 8 * panel : 8, place = item - panel * 8 * gx;
  const int m0 = BM * (8 * panel + place % in_panel), n0 = BN * (place / in_panel);
  const int chunks = K / 64;
  const unsigned ring_at = (unsigned)(size_t)(__attribute__((address_space(3))) char*)ring + 1024 * wave;
  const __bf16* load_x = same_in_all_lanes(x + (size_t)m0 * K);
  const __bf16* load_w = same_in_all_lanes(wt + (size_t)n0 * K);        // (whole tiles of 16 rows)
  unsigned at_row[LOADS];                                              // of x for the first four loads, of W behind them
  {
    const int last_m = M - m0 - 1, last_tile = (N + 15) / 16 - n0 / 16 - 1, lane = threadIdx.x & 63;   // past the end: the last one again
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = 8 * (wave + 4 * j) + (lane >> 3);
      at_row[j] = (unsigned)(s < last_m ? s : last_m) * (unsigned)(2 * K) + 16 * ((lane & 7) ^ lds_place(s));
    }
#pragma unroll
    for (int j = 4; j < LOADS; ++j) {                                  // k-step q / (2 B) of tile q % (2 B)
      const int q = wave + 4 * (j - 4), u = q % (2 * B);
      at_row[j] = (unsigned)(u < last_tile ? u : last_tile) * (unsigned)(32 * K) + 1024 * (q / (2 * B)) + 16 * lane;
    }
  }
  auto load = [&](int j, unsigned slot) { load_to_lds(at_row[j], j < 4 ? load_x : load_w, slot + 4096 * j); };
  auto barrier = [&]() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
  };
  int ahead = 0;                                                       // chunks asked for
  auto advance = [&]() {
    if (++ahead < chunks) {
      load_x += 64;
      load_w += 1024;
    }                                                                  // (past the last chunk: that one again, which nothing reads)
  };
#pragma unroll
  for (int s = 0; s < SLOTS; ++s) {
#pragma unroll
    for (int j = 0; j < LOADS; ++j) load(j, ring_at + SLOT * s);
    advance();
  }
  int at_x, at_w;
  {
    const int lane = threadIdx.x & 63, i = lane & 15;
    at_x = 128 * i + 16 * ((4 * wk + (lane >> 4)) ^ lds_place(i));
    at_w = 128 * BM + 1024 * (2 * B * wk + B * wn) + 16 * lane;
  }
  // (rows 16 a + i: lds_place of them is that of i)
  f32x4 acc[8][B];
#pragma unroll
  for (int a = 0; a < 8; ++a)
#pragma unroll
    for (int b = 0; b < B; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 ops[2][R];                                                    // x's eight tiles, then W's
  auto read = [&](int set, int r, int slot) {
    ops[set][r] = *(const bf16x8*)(ring + slot + (r < 8 ? at_x + 2048 * r : at_w + 1024 * (r - 8)));
  };
  wait_loads<(SLOTS - 1) * LOADS>();
  barrier();
#pragma unroll
  for (int r = 0; r < R; ++r) read(0, r, 0);
  asm volatile("" : : : "memory");
  wait_loads<(SLOTS - 2) * LOADS>();
  barrier();
  int read_at = SLOT;
  unsigned load_at = 0;
  auto next = [&](unsigned at) { return at == SLOT * (SLOTS - 1) ? 0u : at + SLOT; };
  auto chunk = [&](auto set_tag) {
    constexpr int set = decltype(set_tag)::value;
#pragma unroll
    for (int i = 0; i < P; ++i) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        if (q * (P * 3 / 4) / R != i) continue;
        const int r = q == 0 ? 0 : q <= B ? 7 + q : q - B;             // x's first tile, W's, the others of x: as they are used
        read(set ^ 1, r, read_at);
      }
#pragma unroll
      for (int j = 0; j < LOADS; ++j)
        if (j * P / LOADS == i) load(j, ring_at + load_at);
      const int a = i / B, b = a & 1 ? B - 1 - i % B : i % B;          // (consecutive products differ in one operand)
      asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[a][b]) : "v"(ops[set][8 + b]), "v"(ops[set][a]));
      __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("" : : : "memory");
    wait_loads<(SLOTS - 2) * LOADS>();
    barrier();
    read_at = next(read_at);
    load_at = next(load_at);
    advance();
  };
  int c = 0;
  for (; c + 2 <= chunks; c += 2) {
    chunk(std::integral_constant<int, 0>{});
    chunk(std::integral_constant<int, 1>{});
  }
  if (c < chunks) chunk(std::integral_constant<int, 0>{});
  // The two halves of every chunk's k meet: a wavefront hands the sums of the rows of x that are the other's to it, by way of the
  // ring's LDS once all loads into it are done.
  wait_loads<0>();
  barrier();
  // (the last products' results, which the compiler does not see coming: read by none before the waits)
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
  for (int a = 0; a < 8; ++a)
#pragma unroll
    for (int b = 0; b < B; ++b) asm volatile("" : "+a"(acc[a][b]));
  f32x4* mail = (f32x4*)ring;
  const int lane = threadIdx.x & 63, g = lane >> 4;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < B; ++b) mail[((wave * 4 + a) * B + b) * 64 + lane] = wk ? acc[a][b] : acc[4 + a][b];
  __syncthreads();
  const int from = (wave ^ 2) * 4;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int m = m0 + 64 * wk + 16 * a + (lane & 15);
    f32x4 r[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
      r[b] = wk ? acc[4 + a][b] : acc[a][b];
      const f32x4 o = mail[((from + a) * B + b) * 64 + lane];
      r[b] = wk ? o + r[b] : r[b] + o;
      const int n = n0 + 16 * B * wn + 16 * b + 4 * g;
      if (bias != nullptr && n < N) {
#pragma unroll
        for (int e = 0; e < 4; ++e) r[b][e] += bias[n + e];
      }
    }
    if (m >= M) continue;
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int n = n0 + 16 * B * wn + 16 * b + 4 * g;
      if (n >= N) continue;
      if constexpr (KIND == EVEN_F32) {
        *(f32x4*)((float*)y + (size_t)m * N + n) = r[b];
      } else {
        bf16x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = (__bf16)r[b][e];
        *(bf16x4*)((__bf16*)y + (size_t)m * N + n) = h;
      }
    }
  }
}
