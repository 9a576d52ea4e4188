// y[M, N] = x[M, K] W[N, K]^T for at most 16 rows of x in bfloat16, W in the tiled layout (see sl_tile_weight): a decode step of
// one to sixteen requests.  Included by gemm.hip, whose comments on the few-rows products say what GATED, PRODUCER, CONSUMER and
// ROPE add to the product.
//
// Bound by streaming W once and, where W is small, by the chain launch -> loads -> sums across the wavefronts -> store.  A workgroup
// of eight wavefronts owns a tile of W (16 columns of y), half of one, or two (TILES 1, 0, 2), each wavefront an eighth of K.
//   * Up to 8 rows of x (WIDE false): the matrix instruction has 16 columns for them; the lanes of columns 8..15 hold the same rows
//     one k-step further on, so that one load of x serves two k-steps (a load takes a place in the CU's queue of outstanding
//     requests whatever its size, and that queue is what these kernels run on).  Whole tiles: the even k-steps' products are
//     valid in columns 0..7 of one accumulator, the odd ones' in columns 8..15 of another.
//   * Half a tile: a load of W is 8 rows at two k-steps, whole cache lines of 128 bytes out of the same layout; up to 8 rows of x
//     one instruction then multiplies both k-steps (two quadrants of its result are valid).
//   * Two tiles share every load of x: with 9 to 16 rows those loads are up to half of what a CU pulls.  Their consumers are held to 80
//     registers, three workgroups a CU: with 82 and two, the 560 of 17920 x 896 took 11.4 us at 16 rows, now 9.8.
//   * All loads of U pairs of k-steps are asked for before the first product, held there by a scheduling barrier.  Without it the
//     compiler moves the loads of x down to their products, and a wavefront makes a trip to memory for each of them.
// Measured in chains of a graph, W cold (us; before: loads left to the compiler, whole tiles; in brackets a plain read of W):
// 2048 x 11008 at 1 / 4 rows 15.2 / 15.5 -> 9.3 / 9.8 (9.2), 2048 x 2048 4.6 / 4.8 -> 3.5 / 3.7 (3.2), 64 x 2048 4.1 -> 2.9 (1.7),
// 3584 x 18944 at 8 rows 27.7 -> 24.1 (24.4), 18944 x 3584 23.7 -> 22.5, gated 22016 x 2048 at 4 rows 17.7 -> 15.9 (16.7),
// 32000 x 2048 at one row 23.5 -> 21.4, 2048 x 11008 at 16 rows 19.4 -> 15.2, 37888 x 3584 at 16 rows (two tiles) 48.0 -> 46.2.
// Tried: rings that refill a register as it is used (0.1 to 1 us slower), 16 wavefronts (as fast at 3584 x 18944, slower at many
// tiles), plain instead of streaming loads of W (0.2 to 1.7 us slower).
struct FewRows {
  const __bf16* x;
  const __bf16* wt;
  const float* bias;
  void* y;
  int M, N, K, out_f32;
  NormFusion F;
  RopeStore R;
  KeyShares S;
};

template <bool WIDE, int TILES, bool GATED, bool CONSUMER, bool PRODUCER, int PARTS, bool ROPE, int U, int WAVES = 8, bool SHARES = false>
__global__ __launch_bounds__(64 * WAVES, TILES == 2 && CONSUMER && !ROPE && PARTS == 8 ? 6 : 1) void gemm_few_kernel(const FewRows A) {
  constexpr bool HALF = TILES == 0;
  constexpr int NT = TILES == 2 ? 2 : 1;
  static_assert(NT == 1 || WIDE, "two tiles a workgroup share their loads of nine and more rows of x");
  static_assert(!HALF || (!GATED && !ROPE), "a gate and its up, a channel and its partner lie in one tile");
  static_assert(!SHARES || PRODUCER, "shares of keys: added to the stream");
  static_assert(!CONSUMER || WAVES == 8, "the shares of the sums of squares are laid out for 512 threads");
  constexpr int C = HALF ? 8 : 16;                           // columns of y a workgroup owns
  constexpr int RM = WIDE ? 16 : 8;                          // rows of x
  constexpr int LW = HALF ? 1 : 2, LX = WIDE ? 2 : 1;        // loads of W and of x for two k-steps
  __shared__ f32x4 red[NT][WAVES][WIDE ? 64 : 32];
  __shared__ float wsum[CONSUMER ? WAVES : 1][16];
  const NormFusion& F = A.F;
  const RopeStore& R = A.R;
  const int M = A.M, N = A.N, K = A.K;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int lane = threadIdx.x % 64, i = lane & 15, gq = lane >> 4, hi = i >> 3;
  const int th = PRODUCER && !HALF ? F.th : 16;
  const int KT = K / 32, KP = KT / 2;                        // pairs of k-steps; an odd one at the end is the last wavefront's
  const int p0 = first_k_step(KP, wave, WAVES), p1 = first_k_step(KP, wave + 1, WAVES);
  const int ntiles = (N + th - 1) / th;
  const int tile0 = HALF ? blockIdx.x >> 1 : blockIdx.x * NT, half = HALF ? blockIdx.x & 1 : 0;
  const int wstep = 32 * th;                                 // values of W from one k-step of a tile to the next
  const __bf16* wtile[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wtile[t] = A.wt + (size_t)(tile0 + t < ntiles ? tile0 + t : ntiles - 1) * KT * wstep;
  // (lanes of rows a lower tile does not have read its last row; their columns of the result are dropped)
  const int wlane = HALF ? hi * 512 + (gq * 16 + half * 8 + (i & 7)) * 8 : (gq * th + (i < th ? i : th - 1)) * 8;
  const int xcol = WIDE ? i : i & 7;
  int xrow = xcol < M ? xcol : M - 1;
  if (CONSUMER && F.rows != nullptr) xrow = F.rows[xrow];
  const int xstep = !SHARES && F.x_tiled ? F.x_tiled * 32 : 32;       // values of x from one k-step of a row to the next
  const int xlane = xrow * (!SHARES && F.x_tiled ? 32 : K) + 8 * gq + (WIDE ? 0 : hi * xstep);
  // what only the epilogue needs, asked for first
  float pv[PARTS];
  if (CONSUMER) {
#pragma unroll
    for (int j = 0; j < PARTS; ++j) {
      const int p = threadIdx.x / 16 + 32 * j;
      pv[j] = p < F.in_nparts ? F.in_parts[p * 16 + lane % 16] : 0.f;
    }
  }
  const int em = threadIdx.x / C, ec = threadIdx.x % C;      // row and column of a thread of the epilogue
  const bool row_live = threadIdx.x < RM * C && em < M;
  float r_old[NT], g_next[NT], b_pre[NT], c_pre[NT], s_pre[NT];
  int slot = 0;
  if (ROPE && row_live && R.slots != nullptr) slot = R.slots[em];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int en = HALF ? tile0 * 16 + half * 8 + ec : (tile0 + t) * th + ec;
    r_old[t] = g_next[t] = b_pre[t] = s_pre[t] = 0.f;
    c_pre[t] = 1.f;
    if (!row_live || en >= N || (!HALF && ec >= th)) continue;
    if (PRODUCER) {
      r_old[t] = F.resid[(size_t)em * N + en];
      g_next[t] = F.next_w[en];
    }
    if (ROPE) {
      if (A.bias != nullptr) b_pre[t] = A.bias[en];
      const int hd = en / R.D, p = en % R.D;
      if (R.cosv != nullptr && hd < R.nh + R.nkv && p < R.rot) {
        const int j = 8 * (p / 16) + p % 8, half_rot = R.rot / 2;
        c_pre[t] = R.cosv[(size_t)em * half_rot + j];
        s_pre[t] = R.sinv[(size_t)em * half_rot + j];
      }
    }
  }
  // Running sums: a producer's, whose results are added to the float stream, of every other pair of k-steps apart, so that they are as
  // short as with the sixteen wavefronts it had (error of a delta of 2048 x 11008 at 8 / 16 rows 1.30e-7 / 1.66e-7; one sum 1.58e-7 / 2.24e-7).
  constexpr int SUMS = PRODUCER && !SHARES && !(HALF && WIDE) ? 2 : 1;
  f32x4 acc[SUMS][NT], odd[SUMS];
#pragma unroll
  for (int s = 0; s < SUMS; ++s) {
    odd[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  bf16x8 a[NT][LW * U], b[LX * U];
  auto load_w = [&](int u, int p) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const __bf16* w = wtile[t] + (size_t)p * (2 * wstep);
      a[t][LW * u] = stream_load(w + wlane);
      if (!HALF) a[t][LW * u + LW - 1] = stream_load(w + wstep + wlane);
    }
  };
  auto load_x = [&](int u, const __bf16* x, int p) {
    b[LX * u] = *(const bf16x8*)(x + 2 * p * xstep + xlane);
    if (WIDE) b[LX * u + LX - 1] = *(const bf16x8*)(x + (2 * p + 1) * xstep + xlane);
  };
  auto multiply = [&](int u) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x4& even = acc[u % SUMS][t];
      even = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t][LW * u], b[LX * u], even, 0, 0, 0);
      f32x4& other = WIDE && !HALF ? even : odd[u % SUMS];   // (whole tiles of 16 rows of x: all of one accumulator is valid)
      if (WIDE || !HALF) other = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t][LW * u + LW - 1], b[LX * u + LX - 1], other, 0, 0, 0);
    }
  };
  const __bf16* x = A.x;
  if constexpr (SHARES) {
    // x is attention that is still in shares of its keys.  A thread merges the shares of a channel, everything it needs asked for
    // at once behind the first of W, into rows of bfloat16 in LDS.  (Merged by the lanes that multiply, sixteen (row, share) pairs
    // to a load, it took 7 us a layer of the 0.5B shape more than the merging kernel that it saves.)
    extern __shared__ __bf16 merged[];                       // [M][K]
    constexpr int J = SL_MAX_SHARES;
    const KeyShares& S = A.S;
    ask_ahead<U>(p0, p1, load_w);
    for (int c = threadIdx.x; c < M * K; c += 64 * WAVES) {
      const size_t at = (size_t)(c >> S.head_bits) * S.shares;        // (rows of K values: whole heads)
      const float* o = S.o + (at << S.head_bits) + (c & ((1 << S.head_bits) - 1));
      float v[J], top = -INFINITY, sum = 0.f, all = 0.f;
      float2 ml[J];
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int q = j < S.shares ? j : S.shares - 1;
        v[j] = o[(size_t)q << S.head_bits];
        ml[j] = S.ml[at + q];
      }
#pragma unroll
      for (int j = 0; j < J; ++j) top = fmaxf(top, ml[j].x);
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const float wgt = j < S.shares && ml[j].x != -INFINITY ? __builtin_amdgcn_exp2f(ml[j].x - top) : 0.f;   // (maxima are in units of log 2)
        all += wgt * ml[j].y;
        sum += wgt * v[j];
      }
      merged[c] = (__bf16)(sum * (1.f / all));
    }
    __syncthreads();
    x = merged;
    for (int p = p0; p < p1; p += U) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (p + u >= p1) break;
        if (p != p0) load_w(u, p + u);
        load_x(u, x, p + u);
        multiply(u);
      }
    }
  } else {
    int p = p0;
    for (; p + U <= p1; p += U) {
#pragma unroll
      for (int u = 0; u < U; ++u) load_w(u, p + u), load_x(u, x, p + u);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u) multiply(u);
    }
    if (p < p1) {
#pragma unroll
      for (int u = 0; u < U - 1; ++u)
        if (p + u < p1) load_w(u, p + u), load_x(u, x, p + u);
#pragma unroll
      for (int u = 0; u < U - 1; ++u)
        if (p + u < p1) multiply(u);
    }
  }
  if ((KT & 1) && wave == WAVES - 1) {                       // the odd k-step: its operands in the lanes of even ones alone
    const bf16x8 none = {};
    bf16x8 aw[NT], bx = none;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      aw[t] = none;
      if (!HALF || hi == 0) aw[t] = stream_load(wtile[t] + (size_t)KP * (2 * wstep) + wlane);
    }
    if (WIDE || hi == 0) bx = *(const bf16x8*)(x + 2 * KP * xstep + xlane);
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aw[t], bx, acc[0][t], 0, 0, 0);
  }
  if constexpr (SUMS == 2) {
    odd[0] += odd[1];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[0][t] += acc[1][t];
  }
  // Element r of lane (column of x, quarter of the tile's rows) is a sum of row 4 (quarter) + r of the tile.
  constexpr int QS = WIDE ? 16 : 8;                          // places a quarter takes in LDS: valid columns only
  if (HALF && WIDE) red[0][wave][lane] = gq < 2 ? acc[0][0] : odd[0];      // rows 0..7 of the even k-steps' sums, rows 8..15 of the odd ones'
  else if (HALF) {
    if ((gq >> 1) == hi) red[0][wave][gq * 8 + (i & 7)] = acc[0][0];
  } else if (WIDE) {
#pragma unroll
    for (int t = 0; t < NT; ++t) red[t][wave][lane] = acc[0][t];
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[0][0][r] += lane_xor<8>(odd[0][r]);      // (columns 0..7 are used)
    if (hi == 0) red[0][wave][gq * 8 + i] = acc[0][0];
  }
  if (CONSUMER) {                                            // this wavefront's share of the sums of squares, by row
    float sacc = 0.f;
#pragma unroll
    for (int j = 0; j < PARTS; ++j) sacc += pv[j];
    sacc = column_meet(sacc, add_f);
    if (lane < 16) wsum[wave][lane] = sacc;
  }
  __syncthreads();
  if (threadIdx.x >= RM * C) return;
  auto sum_of = [&](int t, int m, int n) {                   // row n of the tile (HALF: and the same row of the odd k-steps)
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float even = red[t][w][(n / 4) * QS + m][n % 4];
      s += HALF ? even + red[t][w][(2 + n / 4) * QS + m][n % 4] : even;
    }
    return s;
  };
  auto inv_of = [&](int m) {                                 // rsqrt(mean x^2 + eps) of the row of x behind result row m
    const int tok = F.rows != nullptr ? F.rows[m] : m;
    float ss = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) ss += wsum[w][tok];
    return rsqrtf(ss / (float)K + F.eps);
  };
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int tile = tile0 + t;
    if (NT > 1 && tile >= ntiles) break;
    if constexpr (GATED) {
      const int m = threadIdx.x / 8, j = threadIdx.x % 8, n = tile * 8 + j;
      if (m >= M || n >= N / 2) continue;
      float g = sum_of(t, m, j), u = sum_of(t, m, j + 8);
      if (CONSUMER) {
        const float inv = inv_of(m);
        g *= inv;
        u *= inv;
      }
      if (A.bias != nullptr) {                               // (the bias lies as the rows do: 8 gates, their 8 ups)
        g += A.bias[tile * 16 + j];
        u += A.bias[tile * 16 + 8 + j];
      }
      const size_t at = F.y_tiled ? (size_t)(n / 32) * (M * 32) + m * 32 + n % 32 : (size_t)m * (N / 2) + n;
      ((__bf16*)A.y)[at] = (__bf16)(sl_act(g, F.gate_act) * u);
      continue;
    }
    const int en = HALF ? tile * 16 + half * 8 + ec : tile * th + ec;
    const bool live = em < M && en < N && (HALF || ec < th);
    float s = sum_of(t, em, ec);
    if (CONSUMER && live) s *= inv_of(em);
    if constexpr (ROPE) {
      s += b_pre[t];
      const float partner = lane_xor<8>(s);                  // the other half of the pair, same row
      if (!live) continue;
      const int hd = en / R.D, q = en % R.D;
      if (hd < R.nh + R.nkv) {
        float val = s;
        if (R.cosv != nullptr && q < R.rot) val = q % 16 < 8 ? s * c_pre[t] - partner * s_pre[t] : s * c_pre[t] + partner * s_pre[t];
        if (hd < R.nh) ((__bf16*)A.y)[(size_t)em * N + en] = (__bf16)(val * R.qscale);
        else if (R.slots != nullptr)
          R.kc[(((size_t)(slot / R.page) * R.nkv + (hd - R.nh)) * R.page + slot % R.page) * R.D + q] = (__bf16)val;
      } else if (R.slots != nullptr) {
        R.vc[(((size_t)(slot / R.page) * R.nkv + (hd - R.nh - R.nkv)) * R.D + q) * R.page + slot % R.page] = (__bf16)s;
      }
      continue;
    }
    if (live && A.bias != nullptr) s += A.bias[en];
    const size_t at = !CONSUMER && F.y_tiled ? (size_t)(en / 32) * (M * 32) + em * 32 + en % 32 : (size_t)em * N + en;
    if (PRODUCER) {
      float sq = 0.f;
      if (live) {
        const float r = r_old[t] + s;
        F.resid[(size_t)em * N + en] = r;
        ((__bf16*)A.y)[at] = (__bf16)(r * g_next[t]);
        sq = r * r;
      }
      if (C == 16) sq += lane_xor<8>(sq);                    // over the workgroup's columns of row em
      sq += lane_xor<4>(sq);
      sq += lane_xor<2>(sq);
      sq += lane_xor<1>(sq);
      if (ec == 0) {
        float* parts = F.out_parts + (size_t)(HALF ? blockIdx.x : tile) * 16 + em;
        parts[0] = sq;
        if (!WIDE) parts[8] = 0.f;                           // (rows that the stream does not have: sixteen are laid down)
      }
    } else if (live) {
      if (!CONSUMER && F.gate_act) s = sl_act(s, F.gate_act);
      if (A.out_f32) ((float*)A.y)[at] = s;
      else ((__bf16*)A.y)[at] = (__bf16)s;
    }
  }
}

// TILES: 0 half a tile a workgroup, 1, 2.  U: pairs of k-steps asked for together.  One tile and 9 to 16 rows: four, and three where there are
// more than two tiles a CU, so that no more than 80 registers (of consumers of up to 4,096 values and of plain rows) leave room for three
// workgroups, all tiles at once: 12288 x 1024 7.6 to 9.5 us with four, 6.6 to 7.9 with three, 9728 x 896 6.8 to 8.0 and 5.7 to 6.8; 2048 x 2048, whose
// wavefronts have four pairs, 5.2 and 5.5.  Halves: 9 or 10 pairs in one trip, in fours / tens at one row and
// at 8: 896 x 4224 4.5 / 4.0 and 5.6 / 5.2, 1536 x 4864 5.0 / 4.7 and 6.1 / 5.9, 2048 x 4864 5.8 / 5.5 and 6.4 / 6.2, 2048 x 5056 5.9 / 5.8 and 6.4 / 6.5,
// 2048 x 5120, ten pairs for every wavefront, 5.6 / 5.5 and 6.5 / 6.7; products that add to the stream 1536 x 4864 5.3 / 5.1 and 6.3 / 6.2, 2048 x 4864
// 6.0 / 5.9 and 6.6 / 6.5, 2048 x 4992 6.2 / 6.2 and 6.6 / 6.9, 2048 x 5120 5.9 / 6.2 and 6.8 / 7.2.  9 to 16 rows and more than four pairs, in twos (in
// fours / twos at 9 and 16 rows: 896 x 4864 6.3 / 6.2 and 8.0 / 7.5, 2048 x 3072 5.2 / 5.2 and 6.3 / 5.9, 1536 x 8960 11.4 / 11.3 and 13.1 / 12.8).
template <bool WIDE, int TILES, int U>
static void launch_few_rows(const FewRows& A, bool gated, bool rope, hipStream_t stream) {
  const bool consumer = A.F.in_parts != nullptr, producer = A.F.resid != nullptr, few = A.F.in_nparts <= 32 * 8;
  const int tiles = (A.N + A.F.th - 1) / A.F.th;
  const dim3 grid(TILES == 0 ? 2 * tiles : TILES == 1 ? tiles : (tiles + 1) / 2);
#define SL_FEW(GATED, CONSUMER, PRODUCER, PARTS, ROPE) \
  gemm_few_kernel<WIDE, TILES, GATED, CONSUMER, PRODUCER, PARTS, ROPE, U><<<grid, 512, 0, stream>>>(A)
  if constexpr (TILES > 0) {
    if (rope && consumer && few) return SL_FEW(false, true, false, 8, true);
    if (rope && consumer) return SL_FEW(false, true, false, 16, true);
    if (rope) return SL_FEW(false, false, false, 1, true);
    if (consumer && gated && few) return SL_FEW(true, true, false, 8, false);
    if (consumer && gated) return SL_FEW(true, true, false, 16, false);
    if (consumer && few) return SL_FEW(false, true, false, 8, false);
    if (consumer) return SL_FEW(false, true, false, 16, false);
    if (gated) return SL_FEW(true, false, false, 1, false);
  }
  if constexpr (U % 2 == 0) {                                // (a producer's two running sums: of pairs in turn)
    if (producer) return SL_FEW(false, false, true, 1, false);
  }
  SL_FEW(false, false, false, 1, false);
#undef SL_FEW
}
