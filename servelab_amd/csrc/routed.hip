// Routed experts: every token goes through the `top` experts with the largest router logits,
// weighted by the softmax over those logits only; or (shares over all experts) with the largest
// softmax shares plus a correction per expert, weighted by their shares, divided by their sum
// and multiplied by a constant; or with the largest logits, weighted by their sigmoids, which
// multiply an expert's input instead of its output (as a factor of its first products' sums:
// W (s x) = s (W x)).  The last experts may be ones without matrices that hand their
// input through.
//
//   route       per token the chosen experts and their shares (float), one wavefront a token
//   group       the step's (token, choice) pairs sorted by expert, on the device: where each
//               expert's rows start, the list of row tiles (expert, first row, rows) that the
//               grouped products walk, and each pair's place in the sorted order
//   grouped     y[row] = W[expert of row] x[row]: one launch over all experts, a workgroup per
//               (row tile, column tile); the gated form computes act(gate) * up of an expert's
//               stacked [gate; up] matrix, the activated form act(W x) of a single one
//   combine     out[token] = g base[token] + sum over its choices of share * y[place of the pair],
//               g = 1 or the sigmoid of one number per token
//
// No launch depends on the routing: the grids are sized for the worst case (pairs / tile rows
// + experts tiles) and workgroups beyond the tiles in use leave at once, so a step is a fixed
// list of launches that a captured graph can replay.
#include "common.h"
#include "lds_loads.h"

#define RT_ROWS 16           // rows of a tile of the plain grouped product; a row tile holds 16, 128 or 256 rows

// ------------------------------------------------------------------ route
// One wavefront per token; lane k < top gets the expert of the k-th choice.  Largest first; among equal logits the lower
// index wins.  NaN counts as -infinity there, so that a choice is an expert whatever the row holds; its share is NaN.
// over_all: the numbers compared are softmax(z)[e] + correction[e] over all E, and a chosen
// expert's share is softmax(z)[e] / (sum over the chosen + 1e-20) * scale.  sigmoid: the logits are
// compared, and a chosen expert's share is the sigmoid of its own.
struct Route {
  const float* logits;
  int stride, E, top;
  int* chosen;
  float* shares;
  int over_all;
  const float* correction;
  float scale;
  int sigmoid;
};

__device__ __forceinline__ int route_token(const Route& r, size_t t, int lane) {
  const int E = r.E, top = r.top, over_all = r.over_all;
  const float* __restrict__ correction = r.correction;
  int* __restrict__ chosen = r.chosen;
  float* __restrict__ shares = r.shares;
  const float* __restrict__ z = r.logits + t * r.stride;
  float zmax = 0.f, inv_sum = 1.f;
  if (over_all) {
    float mx = -INFINITY;
    for (int e = lane; e < E; e += 64) mx = fmaxf(mx, z[e]);
    zmax = wave_max(mx);
    float sm = 0.f;
    for (int e = lane; e < E; e += 64) sm += expf(z[e] - zmax);
    inv_sum = 1.f / wave_sum(sm);
  }
  unsigned long long taken = 0ull;             // bit u: element lane + 64 u is chosen already (E <= 4096)
  float mine = 0.f;                            // lane k keeps the k-th largest logit
  int mine_e = 0;
  auto number = [&](int e) -> float {          // what the experts are compared by
    const float v = z[e], c = over_all ? expf(v - zmax) * inv_sum + (correction != nullptr ? correction[e] : 0.f) : v;
    return c == c ? c : -INFINITY;
  };
  float kept[4];                               // a lane's first four numbers stay in registers (E <= 256: all)
#pragma unroll
  for (int u = 0; u < 4; ++u) kept[u] = lane + 64 * u < E ? number(lane + 64 * u) : -INFINITY;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int at = 0x7fffffff;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = lane + 64 * u;
      if (e < E && !((taken >> u) & 1ull) && (kept[u] > best || (kept[u] == best && e < at))) {
        best = kept[u];
        at = e;
      }
    }
    for (int u = 4, e = lane + 256; e < E; ++u, e += 64) {
      const float v = number(e);
      if (!((taken >> u) & 1ull) && (v > best || (v == best && e < at))) {
        best = v;
        at = e;
      }
    }
    const float most = wave_max(best);
    unsigned long long holders = __ballot(best == most);
    if (__popcll(holders) == 1) {
      at = __builtin_amdgcn_readlane(at, __ffsll(holders) - 1);
    } else {
      if (best != most) at = 0x7fffffff;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) at = min(at, __shfl_xor(at, o, SL_WAVE));
    }
    best = most == -INFINITY && !over_all ? z[at] : most;
    if (at % 64 == lane) taken |= 1ull << (at / 64);
    if (lane == k) {
      mine = best;
      mine_e = at;
    }
  }
  if (over_all) {
    const float w = lane < top ? expf(z[mine_e] - zmax) * inv_sum : 0.f;
    const float sum = wave_sum(w);
    if (lane < top) {
      chosen[t * top + lane] = mine_e;
      shares[t * top + lane] = w / (sum + 1e-20f) * r.scale;
    }
    return mine_e;
  }
  if (r.sigmoid) {
    if (lane < top) {
      chosen[t * top + lane] = mine_e;
      shares[t * top + lane] = 1.f / (1.f + expf(-mine));
    }
    return mine_e;
  }
  const float top1 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(mine)));
  const float w = lane < top ? expf(mine - top1) : 0.f;
  const float sum = wave_sum(w);
  if (lane < top) {
    chosen[t * top + lane] = mine_e;
    shares[t * top + lane] = w / sum;
  }
  return mine_e;
}

// The same for up to 64 experts: a lane has one, and what is compared stays in its register.
__device__ __forceinline__ int route_token_64(const Route& r, size_t t, int lane) {
  const int E = r.E, top = r.top;
  const bool there = lane < E;
  const float raw = r.logits[t * r.stride + (there ? lane : 0)], add = r.correction != nullptr ? r.correction[there ? lane : 0] : 0.f;
  float share = 0.f, number = raw;
  if (r.over_all) {
    const float zmax = wave_max(there ? raw : -INFINITY);
    share = there ? expf(raw - zmax) : 0.f;
    share *= 1.f / wave_sum(share);
    number = share + add;
  }
  number = number == number ? number : -INFINITY;
  unsigned long long left = __ballot(there);
  float mine = 0.f;
  int mine_e = 0;
  for (int k = 0; k < top; ++k) {
    const bool in = left >> lane & 1;
    const float most = wave_max(in ? number : -INFINITY);
    const int at = __ffsll(__ballot(in && number == most)) - 1;      // (the lowest index among equals)
    left &= ~(1ull << at);
    // (a chosen expert's logit, or its share of all; NaN stays what it is)
    const float v = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.over_all ? share : raw), at));
    if (lane == k) {
      mine = v;
      mine_e = at;
    }
  }
  float w;
  if (r.over_all) {
    w = lane < top ? mine : 0.f;
    w = w / (wave_sum(w) + 1e-20f) * r.scale;
  } else if (r.sigmoid) {
    w = 1.f / (1.f + expf(-mine));
  } else {
    const float top1 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(mine)));
    w = lane < top ? expf(mine - top1) : 0.f;
    w = w / wave_sum(w);
  }
  if (lane < top) {
    r.chosen[t * top + lane] = mine_e;
    r.shares[t * top + lane] = w;
  }
  return mine_e;
}

__global__ __launch_bounds__(64) void route_kernel(const Route r) {
  if (r.E <= 64) route_token_64(r, blockIdx.x, threadIdx.x);
  else route_token(r, blockIdx.x, threadIdx.x);
}

// ------------------------------------------------------------------ group
// One workgroup sorts the n = tokens * top pairs by expert (counting sort in LDS: 3 E numbers at `sh`).
//   order[place] = pair (token * top + choice);  place_of[pair] = place
//   tiles[i] = {expert, first row, rows} for i < tiles in use; rows 0 beyond; used[0] = tiles in use
// Experts from E_real on have no matrices: their pairs get places but no tiles.
struct Group {
  int n, E, E_real, max_tiles, tile_rows;
  int* order;
  int* place_of;
  int* tiles;
  int* used;
};

__device__ __forceinline__ void group_pairs(const Group& g, const int* chosen, int* sh) {
  const int n = g.n, E = g.E, E_real = g.E_real, tile_rows = g.tile_rows;
  int* __restrict__ tiles = g.tiles;
  int* count = sh;               // [E]
  int* start = sh + E;           // [E] first row of the expert
  int* tile0 = sh + 2 * E;       // [E] first tile of the expert
  const int tid = threadIdx.x;
  for (int e = tid; e < E; e += blockDim.x) count[e] = 0;
  __syncthreads();
  for (int i = tid; i < n; i += blockDim.x) atomicAdd(&count[chosen[i]], 1);
  __syncthreads();
  if (tid < 64) {                // one wavefront adds up 64 experts at a time
    int rows = 0, nt = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + tid, c = e < E ? count[e] : 0, tl = e < E_real ? (c + tile_rows - 1) / tile_rows : 0;
      const int up_rows = sum_up_to(c), up_tiles = sum_up_to(tl);
      if (e < E) {
        start[e] = rows + up_rows - c;
        tile0[e] = nt + up_tiles - tl;
      }
      rows += __builtin_amdgcn_readlane(up_rows, 63);
      nt += __builtin_amdgcn_readlane(up_tiles, 63);
    }
    if (tid == 0) *g.used = nt;
    for (int i = nt + tid; i < g.max_tiles; i += 64) {
      tiles[3 * i] = 0;
      tiles[3 * i + 1] = 0;
      tiles[3 * i + 2] = 0;
    }
  }
  __syncthreads();
  for (int e = tid; e < E; e += blockDim.x) {
    const int c = count[e], first = start[e];
    if (e < E_real)
      for (int i = 0; i * tile_rows < c; ++i) {
        int* tl = tiles + 3 * (tile0[e] + i);
        tl[0] = e;
        tl[1] = first + i * tile_rows;
        tl[2] = min(tile_rows, c - i * tile_rows);
      }
    count[e] = first;                                                 // now the next free row
  }
  __syncthreads();
  for (int i = tid; i < n; i += blockDim.x) {
    const int place = atomicAdd(&count[chosen[i]], 1);
    g.order[place] = i;
    g.place_of[i] = place;
  }
}

__global__ __launch_bounds__(1024) void group_kernel(const int* __restrict__ chosen, const Group g) {
  extern __shared__ int sh[];
  group_pairs(g, chosen, sh);
}

// Both for a step of up to 16 tokens, a wavefront each: the work is a few microseconds of one workgroup, and a second
// launch costs as much again (2 tokens, 64 experts, 8 choices: 7.5 + 8.3 us in two kernels; 6.2 here with four experts a lane in a loop
// over all of them, 3.2 with an expert's number in its lane's register).  Pairs placed by looking at all the others, in place of the
// counters of the sort, took 4.2, and 32 pairs 5.4 against 3.4.
__global__ __launch_bounds__(1024) void route_group_kernel(const Route r, const Group g) {
  extern __shared__ int sh[];
  int* chosen = sh + 3 * g.E;    // [n]
  const int wave = threadIdx.x / 64, lane = threadIdx.x & 63;
  const int e = r.E <= 64 ? route_token_64(r, wave, lane) : route_token(r, wave, lane);
  if (lane < r.top) chosen[wave * r.top + lane] = e;
  __syncthreads();
  group_pairs(g, chosen, sh);
}

extern "C" const char* sl_route_tokens(const float* logits, int stride, int T, int E, int top, int* chosen,
                                       float* shares, int* order, int* place_of, int* tiles, int* used, int max_tiles,
                                       int tile_rows, int over_all, const float* correction, float scale,
                                       int E_real, int sigmoid, hipStream_t stream) {
  SL_CHECK(!(over_all && sigmoid), "route_tokens: shares over all or sigmoids");
  SL_CHECK(T >= 0 && E >= 1 && E <= 4096 && top >= 1 && top <= 64 && top <= E && E <= stride,
           "route_tokens: at most 4096 experts within the rows, at most 64 choices");
  SL_CHECK(E_real >= 0 && E_real <= E && (over_all || correction == nullptr),
           "route_tokens: the experts with matrices are the first of all; a correction needs shares over all");
  SL_CHECK(tile_rows == 16 || tile_rows == 128 || tile_rows == 256, "route_tokens: row tiles hold 16, 128 or 256 rows");
  SL_CHECK(max_tiles >= ((long long)T * top + tile_rows - 1) / tile_rows + E, "route_tokens: too few tile entries");
  if (T == 0) return nullptr;
  const Route r{logits, stride, E, top, chosen, shares, over_all, correction, scale, sigmoid};
  const Group g{T * top, E, E_real, max_tiles, tile_rows, order, place_of, tiles, used};
  if (T <= 16 && E <= 1024) {
    route_group_kernel<<<1, 64 * T, (3 * E + T * top) * sizeof(int), stream>>>(r, g);
  } else {
    route_kernel<<<T, 64, 0, stream>>>(r);
    group_kernel<<<1, 1024, 3 * E * sizeof(int), stream>>>(chosen, g);
  }
  return sl_launch_status();
}

// ------------------------------------------------------------------ grouped products
struct Grouped {
  const act_t* x;            // row r reads x + src(r) * K, src(r) = order[r] / top when order is given, else r
  const int* order;
  int top;
  const act_t* w;            // [experts][N_w][K]; gated: N_w = 2 N, gate rows before up rows
  int w_tiled;               // an expert's matrix lies as [N_w / 16][K / 32][64 lanes][8], lane = 16 (k / 8 % 4) + n % 16:
                             // the first operand of mfma 16x16x32 as it sits in registers, 1 KB a wavefront's load
  const int* tiles;          // [max_tiles][3]
  int sub;                   // row tiles hold 16 * sub rows
  int N, K;
  act_t* out_act;            // gated and activated: [rows][N]
  float* out_f32;            // plain: [rows][N]
  int act;                   // the activation (common.h); 0 with out_f32
  float limit;               // the clamped gate's bound
  const float* row_scale;    // with order: the sums of row r are multiplied by row_scale[order[r]] first; or nullptr
  const int* used;           // how many of the tiles are in use, which then come first; nullptr: any of them may be
  int max_tiles, col_blocks; // the matrix-core kernels' launch: max_tiles x col_blocks workgroups in a row
};

// Which (row tile, column block) a workgroup of a one-dimensional launch takes.  Workgroups go to the
// chip's eight dies in turn (number % 8), and each die has an L2 of its own: a die gets a contiguous
// run of the list ordered by column block, then row tile, so the row tiles of one expert, which read
// the same columns of the same matrices, run on one die at about the same time and the matrices
// come from memory once.
__device__ __forceinline__ bool grouped_place(const Grouped& a, int& tile, int& cb) {
  const int total = a.max_tiles * a.col_blocks, run = (total + 7) / 8;
  const int m = (blockIdx.x & 7) * run + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= run || m >= total) return false;
  cb = m / a.max_tiles;
  tile = m - cb * a.max_tiles;
  return true;
}

// 256 threads: thread (row = tid / 16, lane16 = tid % 16) owns columns lane16 + 16 u, u < 4, of a
// 16 x 64 tile.  x and W go through LDS in chunks of 32 values of k; sums are float.
template <bool GATED>
__global__ __launch_bounds__(256) void grouped_product_kernel(const Grouped a) {   // (not GATED: plain or activated)
  const int* tl = a.tiles + 3 * (blockIdx.x / a.sub);
  const int part = blockIdx.x % a.sub;                  // which 16 rows of the row tile
  const int rows = min(RT_ROWS, tl[2] - RT_ROWS * part);
  if (rows <= 0) return;
  const int e = tl[0], row0 = tl[1] + RT_ROWS * part;
  const int n0 = blockIdx.y * 64;
  __shared__ float xs[RT_ROWS][33];
  __shared__ float ws[GATED ? 128 : 64][33];
  const int tid = threadIdx.x, r = tid / 16, l = tid % 16;
  const size_t n_w = GATED ? 2 * (size_t)a.N : (size_t)a.N;
  const act_t* we = a.w + (size_t)e * n_w * a.K;
  float acc[4] = {0.f, 0.f, 0.f, 0.f}, acc2[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < a.K; k0 += 32) {
    __syncthreads();
    for (int i = tid; i < RT_ROWS * 32; i += 256) {
      const int rr = i / 32, kk = i % 32;
      float v = 0.f;
      if (rr < rows && k0 + kk < a.K) {
        const size_t src = a.order != nullptr ? (size_t)(a.order[row0 + rr] / a.top) : (size_t)(row0 + rr);
        v = to_f(a.x[src * a.K + k0 + kk]);
      }
      xs[rr][kk] = v;
    }
    for (int i = tid; i < (GATED ? 128 : 64) * 32; i += 256) {
      const int c = i / 32, kk = i % 32;
      const int n = n0 + (c % 64);
      float v = 0.f;
      if (n < a.N && k0 + kk < a.K) v = to_f(we[((size_t)(c / 64) * a.N + n) * a.K + k0 + kk]);
      ws[c][kk] = v;
    }
    __syncthreads();
#pragma unroll 8
    for (int kk = 0; kk < 32; ++kk) {
      const float xv = xs[r][kk];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        acc[u] += xv * ws[l + 16 * u][kk];
        if (GATED) acc2[u] += xv * ws[64 + l + 16 * u][kk];
      }
    }
  }
  if (r >= rows) return;
  const float rs = a.row_scale != nullptr ? a.row_scale[a.order[row0 + r]] : 1.f;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int n = n0 + l + 16 * u;
    if (n >= a.N) continue;
    const size_t at = (size_t)(row0 + r) * a.N + n;
    acc[u] *= rs;
    if (GATED) acc2[u] *= rs;
    if (GATED) a.out_act[at] = from_f<act_t>(sl_gated(acc[u], acc2[u], a.act, a.limit));
    else if (a.act) a.out_act[at] = from_f<act_t>(sl_act(acc[u], a.act));
    else a.out_f32[at] = acc[u];
  }
}

#if !defined(SL_F32)
typedef __bf16 rt_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 rt_bf16x4 __attribute__((ext_vector_type(4)));
typedef float rt_f32x4 __attribute__((ext_vector_type(4)));

// The same on the matrix cores (bfloat16, K in steps of 32, N in steps of 16): a wavefront owns
// NT x 16 rows of a row tile by NU x 16 columns and reads its operands straight from
// memory, eight values a lane: rows of W are the first operand of mfma 16x16x32, rows of x the
// second; the gated form keeps gate and up sums of the same columns.  Rows past the tile's last are
// computed like the last and never stored.
template <int NT, int NU, bool GATED, int WR, int WC>
__global__ __launch_bounds__(64 * WR * WC) void grouped_product_mfma_kernel(const Grouped a) {
  // WR x WC wavefronts a workgroup: WR along the rows of the row tile, WC along the columns; those
  // that read the same rows of x or of W find them in the CU's cache after the first has asked
  int tile, cb;
  if (!grouped_place(a, tile, cb)) return;
  const int* tl = a.tiles + 3 * tile;
  const int wave = threadIdx.x / 64, wr = wave % WR, wc = wave / WR;
  const int rows = min(16 * NT, tl[2] - 16 * NT * wr);
  const int n0 = (cb * WC + wc) * 16 * NU;
  if (rows <= 0 || n0 >= a.N) return;
  const int e = tl[0], row0 = tl[1] + 16 * NT * wr;
  const int lane = threadIdx.x & 63, i = lane & 15, gq = lane >> 4;
  const size_t n_w = GATED ? 2 * (size_t)a.N : (size_t)a.N;
  const __bf16* we = a.w + (size_t)e * n_w * a.K;
  const __bf16* xp[NT];
#pragma unroll
  for (int v = 0; v < NT; ++v) {
    const int rr = row0 + min(16 * v + i, rows - 1);
    const size_t src = a.order != nullptr ? (size_t)(a.order[rr] / a.top) : (size_t)rr;
    xp[v] = a.x + src * a.K + 8 * gq;
  }
  const __bf16* wp[NU];
  const int wstep = a.w_tiled ? 512 : 32;               // elements from one k-step to the next
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    if (a.w_tiled) wp[u] = we + (size_t)(min(n0 + 16 * u, a.N - 16) / 16) * (a.K / 32) * 512 + lane * 8;
    else wp[u] = we + (size_t)min(n0 + 16 * u + i, a.N - 1) * a.K + 8 * gq;
  }
  const size_t up = (size_t)a.N * a.K;                  // from a gate row to its up row (N in steps of 16)
  rt_f32x4 acc[NT][NU], acc2[NT][GATED ? NU : 1];
#pragma unroll
  for (int v = 0; v < NT; ++v)
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      acc[v][u] = rt_f32x4{0.f, 0.f, 0.f, 0.f};
      if (GATED) acc2[v][u] = rt_f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll 4
  for (int k = 0; k < a.K; k += 32) {
    rt_bf16x8 b[NT], w1[NU], w2[GATED ? NU : 1];
    const size_t kw = (size_t)(k / 32) * wstep;
#pragma unroll
    for (int v = 0; v < NT; ++v) b[v] = *(const rt_bf16x8*)(xp[v] + k);
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      w1[u] = *(const rt_bf16x8*)(wp[u] + kw);
      if (GATED) w2[u] = *(const rt_bf16x8*)(wp[u] + up + kw);
    }
#pragma unroll
    for (int v = 0; v < NT; ++v)
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        acc[v][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1[u], b[v], acc[v][u], 0, 0, 0);
        if (GATED) acc2[v][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w2[u], b[v], acc2[v][u], 0, 0, 0);
      }
  }
  // this lane holds columns n0 + 16 u + 4 gq .. + 3 of rows 16 v + i
#pragma unroll
  for (int v = 0; v < NT; ++v) {
    if (16 * v + i >= rows) continue;
    const size_t at = (size_t)(row0 + 16 * v + i) * a.N + n0 + 4 * gq;
    if (a.row_scale != nullptr) {
      const float rs = a.row_scale[a.order[row0 + 16 * v + i]];
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        acc[v][u] *= rs;
        if (GATED) acc2[v][u] *= rs;
      }
    }
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      if (n0 + 16 * u >= a.N) continue;
      if (GATED) {
        rt_bf16x4 r;
#pragma unroll
        for (int c = 0; c < 4; ++c) r[c] = (__bf16)sl_gated(acc[v][u][c], acc2[v][u][c], a.act, a.limit);
        *(rt_bf16x4*)(a.out_act + at + 16 * u) = r;
      } else if (a.act) {
        rt_bf16x4 r;
#pragma unroll
        for (int c = 0; c < 4; ++c) r[c] = (__bf16)sl_act(acc[v][u][c], a.act);
        *(rt_bf16x4*)(a.out_act + at + 16 * u) = r;
      } else {
        *(rt_f32x4*)(a.out_f32 + at + 16 * u) = acc[v][u];
      }
    }
  }
}


// Row tiles of 16 rows where an expert has few of them, bound by the stream of the experts' matrices: a
// workgroup takes a row tile by 16 NU columns and its eight wavefronts cut K among themselves, so that the few
// (expert, column block) pairs of such a step still put enough loads in flight on every CU (one token of 8
// experts of 1,024 x 2,048 was 128 wavefronts that each walked all of K).  The partial sums meet in LDS and are
// added in the order of K.  Two products and the combine, 64 experts of 1,024 over rows of 2,048, 8 a token,
// at 1 / 2 / 4 / 8 / 32 tokens: 48 / 51 / 78 / 113 / 146 -> 23 / 39 / 58 / 89 / 128 us (5.5 TB/s at 8 tokens).
// Four wavefronts or 64 columns a workgroup: 27 us at one token, 103 at 8.
constexpr int FEW_WAVES = 8;
template <int NU, bool GATED>
__global__ __launch_bounds__(64 * FEW_WAVES) void grouped_product_few_kernel(const Grouped a) {
  constexpr int KW = FEW_WAVES;
  constexpr int MATS = GATED ? 2 : 1;
  __shared__ rt_f32x4 part[KW][NU * MATS][64];
  int tile, cb;
  if (!grouped_place(a, tile, cb)) return;
  const int* tl = a.tiles + 3 * tile;
  const int rows = min(16, tl[2]);
  const int n0 = cb * 16 * NU;
  if (rows <= 0 || n0 >= a.N) return;                   // (the whole workgroup)
  const int e = tl[0], row0 = tl[1];
  const int wave = threadIdx.x / 64, lane = threadIdx.x & 63, i = lane & 15, gq = lane >> 4;
  const size_t n_w = GATED ? 2 * (size_t)a.N : (size_t)a.N;
  const __bf16* we = a.w + (size_t)e * n_w * a.K;
  const int rr = row0 + min(i, rows - 1);
  const size_t src = a.order != nullptr ? (size_t)(a.order[rr] / a.top) : (size_t)rr;
  const __bf16* xp = a.x + src * a.K + 8 * gq;
  const __bf16* wp[NU];
  const int wstep = a.w_tiled ? 512 : 32;               // elements from one k-step to the next
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    if (a.w_tiled) wp[u] = we + (size_t)(min(n0 + 16 * u, a.N - 16) / 16) * (a.K / 32) * 512 + lane * 8;
    else wp[u] = we + (size_t)min(n0 + 16 * u + i, a.N - 1) * a.K + 8 * gq;
  }
  const size_t up = (size_t)a.N * a.K;
  rt_f32x4 acc[NU * MATS];
#pragma unroll
  for (int u = 0; u < NU * MATS; ++u) acc[u] = rt_f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = a.K / 32, s1 = steps * (wave + 1) / KW;
#pragma unroll 4
  for (int s = steps * wave / KW; s < s1; ++s) {
    const rt_bf16x8 b = *(const rt_bf16x8*)(xp + 32 * s);
    const size_t kw = (size_t)s * wstep;
    rt_bf16x8 w[NU * MATS];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      w[u] = __builtin_nontemporal_load((const rt_bf16x8*)(wp[u] + kw));
      if (GATED) w[NU + u] = __builtin_nontemporal_load((const rt_bf16x8*)(wp[u] + up + kw));
    }
#pragma unroll
    for (int u = 0; u < NU * MATS; ++u) acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u], b, acc[u], 0, 0, 0);
  }
#pragma unroll
  for (int u = 0; u < NU * MATS; ++u) part[wave][u][lane] = acc[u];
  __syncthreads();
  if (i >= rows) return;
  const float rs = a.row_scale != nullptr ? a.row_scale[a.order[row0 + i]] : 1.f;
  for (int u = wave; u < NU; u += KW) {
    if (n0 + 16 * u >= a.N) continue;
    rt_f32x4 v = part[0][u][lane];
#pragma unroll
    for (int w = 1; w < KW; ++w) v += part[w][u][lane];
    v *= rs;
    const size_t at = (size_t)(row0 + i) * a.N + n0 + 16 * u + 4 * gq;
    if (GATED) {
      rt_f32x4 z = part[0][NU + u][lane];
#pragma unroll
      for (int w = 1; w < KW; ++w) z += part[w][NU + u][lane];
      z *= rs;
      rt_bf16x4 r;
#pragma unroll
      for (int c = 0; c < 4; ++c) r[c] = (__bf16)sl_gated(v[c], z[c], a.act, a.limit);
      *(rt_bf16x4*)(a.out_act + at) = r;
    } else if (a.act) {
      rt_bf16x4 r;
#pragma unroll
      for (int c = 0; c < 4; ++c) r[c] = (__bf16)sl_act(v[c], a.act);
      *(rt_bf16x4*)(a.out_act + at) = r;
    } else {
      *(rt_f32x4*)(a.out_f32 + at) = v;
    }
  }
}


// Row tiles of R = 128 or 256 rows, both operands through LDS: eight wavefronts take a row tile by 256 rows of W (256
// columns, or 128 of the gate and the same 128 of the up matrix), a wavefront R / 2 by 64 of it, and walk their (row tile, column
// block) items, at most a workgroup a CU.  As in the products of whole prompts (gemm_rounds.h) a chunk of 64 values of k is
// two halves, R / 2 rows of x and half of W each; a half's operands are read into registers while the one before it is multiplied,
// in an order laid down instruction by instruction, and six halves of 24 KB, or four of 32, are on the way in the ring.  What
// bounds it at 128 rows is that ring: the matrices come from memory, two microseconds away, and three chunks of 512 ns of matrix
// work ahead do not cover that (about 1.1 us a chunk whatever the order of the items; a chunk of 256 rows takes 1.3).
// The trips that start an item (its row tile, where its rows lie, the rows) are as long as several chunks, so a workgroup
// looks up BATCH items ahead and its loads run on from one item into the next.
// A prompt of 2,048 tokens, 8 of 64 experts of 1,024 over rows of 2,048 a token: gate/up 232 -> 177 us, down 134 -> 109 (of which
// its 134 MB of float rows and 268 MB of matrices are 70), against an item a workgroup, 128 rows each, and a ring of three whole chunks
// behind one barrier; 128 rows walked like this: 209 and 126.
// Halves of the rows without a pair are not multiplied.  HALF: results in bfloat16, and the rows of W are picked from two tiles
// so that a lane holds eight columns in a row; odd tiles lie in LDS with their rows four places on, off the other's banks.
template <int R, bool GATED, bool HALF>
__global__ __launch_bounds__(512, 2) void grouped_product_walk_kernel(const Grouped a) {
  constexpr int X_BYTES = 64 * R, SLOT = X_BYTES + 16384, SLOTS = R == 128 ? 6 : 4, BATCH = 12;
  constexpr int XL = R / 128, LOADS = XL + 2;            // loads of 64 rows a half holds, a wavefront's loads of a half
  constexpr int XT = R / 64;                            // a wavefront's tiles of 16 rows in a half
  static_assert(R == 128 || R == 256, "row tiles of 128 or 256 rows");
  __shared__ __attribute__((aligned(1024))) char ring[SLOTS * SLOT];
  __shared__ int from[BATCH][R];                      // of an item's rows: the row of x
  __shared__ float scale[BATCH][R];                   // and the factor of its sums
  __shared__ int what[BATCH][4];                        // expert, first row, rows, column block
  __shared__ int found;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), wm = wave >> 2, wn = wave & 3;
  // Only the tiles in use, every column block of a tile before the next tile: a die, whose items are a contiguous run, reads a tile's
  // rows of x once for all of its columns and has two or three experts' matrices under way.  A workgroup takes every `step`-th.
  const int total = (a.used != nullptr ? min(*a.used, a.max_tiles) : a.max_tiles) * a.col_blocks, run = (total + 7) / 8;
  const int first = (int)(blockIdx.x & 7) * run, end = min(first + run, total), step = (int)gridDim.x >> 3;
  const int chunks = a.K / 64;
  const unsigned ring_at = (unsigned)(size_t)(__attribute__((address_space(3))) char*)ring + 1024 * wave;
  int at_x[2], at_wt;                                   // where this lane reads its operands in a slot
  {
    const int lane = threadIdx.x & 63, i = lane & 15, gq = lane >> 4;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) at_x[kk] = 128 * (16 * XT * wm + i) + 16 * ((4 * kk + gq) ^ lds_place(i));
    const int odd = HALF ? i >> 3 : 0, row = HALF ? (8 * (i >> 2 & 1) + (i & 3)) ^ (4 * odd) : i;
    at_wt = X_BYTES + 2048 * (2 * wn + odd) + 16 * (16 * gq + row);
  }
  auto operand = [&](int at) { return *(const rt_bf16x8*)(ring + at); };
  auto w_at = [&](int b, int kk) { return HALF ? (at_wt ^ (64 * b)) + 1024 * kk : at_wt + 2048 * b + 1024 * kk; };
  auto barrier = [&]() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
  };
  auto next = [&](unsigned at) { return at == SLOT * (SLOTS - 1) ? 0u : at + SLOT; };

  for (int base = first + (int)(blockIdx.x >> 3); base < end; base += BATCH * step) {
    if (wave == 0) {                                    // the next items that have rows
      const int lane = threadIdx.x & 63, it = base + lane * step;
      int e = 0, row0 = 0, rows = 0, cb = 0;
      if (lane < BATCH && it < end) {
        const int tile = it / a.col_blocks;
        cb = it - tile * a.col_blocks;
        e = a.tiles[3 * tile], row0 = a.tiles[3 * tile + 1], rows = min(R, a.tiles[3 * tile + 2]);
      }
      const unsigned long long live = __ballot(rows > 0);
      if (rows > 0) {
        const int p = __popcll(live & ((1ull << lane) - 1));
        what[p][0] = e, what[p][1] = row0, what[p][2] = rows, what[p][3] = cb;
      }
      if (lane == 0) found = __popcll(live);
    }
    __syncthreads();
    const int items = __builtin_amdgcn_readfirstlane(found);
    for (int q = threadIdx.x; q < items * R; q += 512) {
      const int k = q / R, r = q % R, rr = what[k][1] + min(r, what[k][2] - 1);
      const int pair = a.order != nullptr ? a.order[rr] : rr;
      from[k][r] = a.order != nullptr ? pair / a.top : rr;
      scale[k][r] = a.row_scale != nullptr ? a.row_scale[pair] : 1.f;
    }
    __syncthreads();
    if (items == 0) continue;

    int load_item = 0, load_left;
    const __bf16 *load_x, *load_w;
    unsigned from_x[2 * XL], from_w[4];                 // of each half
    auto open = [&](int k) {
      const int lane = lane_here();
      const int e = __builtin_amdgcn_readfirstlane(what[k][0]), cb = __builtin_amdgcn_readfirstlane(what[k][3]);
      const int n0 = cb * (GATED ? 128 : 256);
      load_left = chunks;
      load_x = a.x;
      load_w = a.w + (size_t)e * (GATED ? 2 * (size_t)a.N : (size_t)a.N) * a.K;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int j = 0; j < XL; ++j) {
          const int r = 64 * j + 8 * wave + (lane >> 3);
          from_x[XL * h + j] = (unsigned)from[k][R / 2 * h + r] * (unsigned)(2 * a.K) + 16 * ((lane & 7) ^ lds_place(r));
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {                   // 1 KB: a tile of 16 rows of W by 32 of k, tiles 2 h and 2 h + 1 of each wn
          const int piece = wave + 8 * j, t = piece >> 1;
          const int col = GATED ? n0 + 32 * (t >> 1) + 16 * (t & 1) : n0 + 64 * (t >> 1) + 32 * h + 16 * (t & 1);
          from_w[2 * h + j] = ((unsigned)(min(col, a.N - 16) / 16) * (unsigned)(a.K / 32) + (piece & 1)) * 1024u
                              + 16 * (HALF && (t & 1) ? lane ^ 4 : lane) + (GATED && h ? 2u * (unsigned)a.N * (unsigned)a.K : 0u);
        }
      }
    };
    auto load = [&](int h, int j, unsigned slot) {
      if (j < XL) load_to_lds(from_x[XL * h + j], load_x, ring_at + slot + 8192 * j);
      else load_to_lds(from_w[2 * h + j - XL], load_w, ring_at + slot + X_BYTES + 8192 * (j - XL));
    };
    auto advance = [&]() {
      if (--load_left > 0) {
        load_x += 64;
        load_w += 1024;
      } else if (load_item + 1 < items) {
        open(++load_item);
      }                                                 // (past the last chunk: that one again, which nothing reads)
    };
    open(0);
#pragma unroll
    for (int s = 0; s < SLOTS; ++s) {
#pragma unroll
      for (int j = 0; j < LOADS; ++j) load(s & 1, j, SLOT * s);
      if (s & 1) advance();
    }
    rt_bf16x8 x0[XT][2], x1[XT][2], w0[2][2], w1[2][2]; // [tile of 16 rows][k-step of 32]
    rt_f32x4 acc[2 * XT][4];                            // [tile of 16 rows, of the first half, then the second][tile of W]
#pragma unroll
    for (int v = 0; v < 2 * XT; ++v)
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[v][u] = rt_f32x4{0.f, 0.f, 0.f, 0.f};
    wait_loads<LOADS * (SLOTS - 1)>();
    barrier();
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
      for (int b = 0; b < 2; ++b) w0[b][kk] = operand(w_at(b, kk));
#pragma unroll
      for (int v = 0; v < XT; ++v) x0[v][kk] = operand(at_x[kk] + 2048 * v);
    }
    asm volatile("" : : : "memory");
    wait_loads<LOADS * (SLOTS - 2)>();
    barrier();
    int read_at = SLOT;                                 // slot of the half that is read next
    unsigned load_at = 0;                               // slot of the half that is loaded next: the one read before

    for (int item = 0; item < items; ++item) {
      const int rows = __builtin_amdgcn_readfirstlane(what[item][2]);
      auto chunk = [&](auto both) {                     // (a loop of its own for each: the registers do not reach for one that branches)
        // the first half of the rows; W's second half and the other rows arrive in registers
        constexpr int P = 8 * XT, R0 = 4 + 2 * XT;      // products, reads
#pragma unroll
        for (int p = 0; p < P; ++p) {
#pragma unroll
          for (int r = 0; r < R0; ++r) {
            if (r * (P * 3 / 4) / R0 != p) continue;
            const int q = r < 4 ? 0 : r - 4;
            if (r < 4) w1[r & 1][r >> 1] = operand(w_at(r & 1, r >> 1) + read_at);
            else x1[q % XT][q / XT] = operand(at_x[q / XT] + read_at + 2048 * (q % XT));
          }
#pragma unroll
          for (int j = 0; j < LOADS; ++j)
            if (j * P / LOADS == p) load(0, j, load_at);
          const int h = p / (4 * XT), j = p % (4 * XT), kk = j / (2 * XT), v = j / 2 % XT, b = (j ^ v) & 1;
          acc[v][2 * h + b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h ? w1[b][kk] : w0[b][kk], x0[v][kk], acc[v][2 * h + b], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("" : : : "memory");
        wait_loads<LOADS * (SLOTS - 2)>();                  // the half that is read next is there
        barrier();
        read_at = (int)next(read_at);
        load_at = next(load_at);
        // the other rows; the first halves of the next chunk arrive
#pragma unroll
        for (int p = 0; p < P; ++p) {
#pragma unroll
          for (int r = 0; r < 2 * XT; ++r)
            if (r * (P / 2) / (2 * XT) == p) x0[r % XT][r / XT] = operand(at_x[r / XT] + read_at + 2048 * (r % XT));
#pragma unroll
          for (int r = 0; r < 4; ++r)                 // (their first half's products are done)
            if (P / 2 + r * (P / 4) / 4 == p) w0[r & 1][r >> 1] = operand(w_at(r & 1, r >> 1) + read_at);
#pragma unroll
          for (int j = 0; j < LOADS; ++j)
            if (j * P / LOADS == p) load(1, j, load_at);
          const int h = p / (4 * XT), j = p % (4 * XT), kk = j / (2 * XT), v = j / 2 % XT, b = (j ^ v) & 1;
          if (decltype(both)::value)
            acc[XT + v][2 * h + b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h ? w1[b][kk] : w0[b][kk], x1[v][kk], acc[XT + v][2 * h + b], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("" : : : "memory");
        wait_loads<LOADS * (SLOTS - 2)>();
        barrier();
        read_at = (int)next(read_at);
        load_at = next(load_at);
        advance();
      };
      if (rows > R / 2) {
        for (int c = 0; c < chunks; ++c) chunk(std::true_type{});
      } else {
        for (int c = 0; c < chunks; ++c) chunk(std::false_type{});
      }
      // this lane: row i of a tile of rows; of W rows 4 gq .. + 3 of each tile, or (HALF) 8 gq .. + 7 of each two
      const int lane = lane_here(), i = lane & 15, gq = lane >> 4, row0 = __builtin_amdgcn_readfirstlane(what[item][1]);
      const int n0 = __builtin_amdgcn_readfirstlane(what[item][3]) * (GATED ? 128 : 256);
#pragma unroll
      for (int v = 0; v < 2 * XT; ++v) {
        const int r = R / 2 * (v / XT) + 16 * XT * wm + 16 * (v % XT) + i;
        const float rs = scale[item][r];
        const size_t at = (size_t)(row0 + r) * a.N;
        rt_f32x4 z[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          z[u] = acc[v][u] * rs;
          acc[v][u] = rt_f32x4{0.f, 0.f, 0.f, 0.f};
        }
        if (r >= rows) continue;
        if constexpr (GATED) {
          const int n = n0 + 32 * wn + 8 * gq;
          rt_bf16x8 h;
          auto gate = [&](int act) {
#pragma unroll
            for (int c = 0; c < 8; ++c) h[c] = (__bf16)sl_gated(z[c >> 2][c & 3], z[2 + (c >> 2)][c & 3], act, a.limit);
          };
          if (a.act == SL_ACT_SILU) gate(SL_ACT_SILU);  // (no branches between the eight chains of operations)
          else gate(a.act);
          if (n < a.N) *(rt_bf16x8*)(a.out_act + at + n) = h;
        } else if constexpr (HALF) {
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const int n = n0 + 64 * wn + 32 * q + 8 * gq;
            rt_bf16x8 h;
#pragma unroll
            for (int c = 0; c < 8; ++c) h[c] = (__bf16)sl_act(z[2 * q + (c >> 2)][c & 3], a.act);
            if (n < a.N) *(rt_bf16x8*)(a.out_act + at + n) = h;
          }
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int n = n0 + 64 * wn + 16 * u + 4 * gq;
            if (n < a.N) *(rt_f32x4*)(a.out_f32 + at + n) = z[u];
          }
        }
      }
    }
    wait_loads<0>();                                    // (loads past the last chunk still land in the ring)
    __syncthreads();
  }
}
#endif

extern "C" const char* sl_grouped_product(const void* x, const int* order, int top, const void* w, const int* tiles,
                                          const int* used, int w_tiled, int max_tiles, int tile_rows, int pairs, int experts,
                                          int N, int K, int gated, int act, float limit, const float* row_scale, void* out, hipStream_t stream) {
  // gated: act(gate) * up into the activation type; else act != 0: act(W x) into the activation type;
  // else plain float sums
  SL_CHECK(max_tiles >= 0 && N > 0 && K > 0 && top >= 1, "grouped_product: sizes must be positive");
  SL_CHECK(act >= 0 && act <= SL_ACT_CLAMPED_SWISH && (!gated || act) && (gated || act != SL_ACT_CLAMPED_SWISH),
           "grouped_product: unknown activation, a gate without one, or the clamped form without a gate");
  SL_CHECK(row_scale == nullptr || order != nullptr, "grouped_product: factors per row go with the pairs' order");
  SL_CHECK(tile_rows == 16 || tile_rows == 128 || tile_rows == 256, "grouped_product: row tiles hold 16, 128 or 256 rows");
  SL_CHECK(pairs >= 0 && experts >= 0, "grouped_product: sizes must be positive");
  if (max_tiles == 0 || pairs == 0) return nullptr;
  if (used != nullptr) max_tiles = min(max_tiles, pairs);         // (the tiles in use come first, and each holds a pair)
  Grouped a{(const act_t*)x, order, top, (const act_t*)w, w_tiled, tiles, tile_rows / RT_ROWS, N, K,
            act ? (act_t*)out : nullptr, act ? nullptr : (float*)out, act, limit, row_scale, used, max_tiles, 1};
#if !defined(SL_F32)
  if (K % 32 == 0 && N % 16 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0 && (uintptr_t)out % 16 == 0) {
    // (a one-dimensional launch of max_tiles x col_blocks workgroups, rounded up to the eight dies)
    auto blocks = [&](int cols) {
      a.col_blocks = (N + cols - 1) / cols;
      return dim3(8 * (unsigned)((max_tiles * a.col_blocks + 7) / 8));
    };
    const unsigned long long rows = order != nullptr ? pairs / top : pairs;
    if (tile_rows >= 128 && w_tiled && K % 64 == 0 && rows * K < (1ull << 31) && (gated ? 2ull : 1ull) * N * K < (1ull << 31)) {
      // (operands' offsets in 32 bits)
      const int cus = device_cus() & ~7;
      dim3 grid = blocks(gated ? 128 : 256);
      if (cus >= 8 && grid.x > (unsigned)cus) grid.x = cus;
      if (tile_rows == 128) {
        if (gated) grouped_product_walk_kernel<128, true, true><<<grid, 512, 0, stream>>>(a);
        else if (act) grouped_product_walk_kernel<128, false, true><<<grid, 512, 0, stream>>>(a);
        else grouped_product_walk_kernel<128, false, false><<<grid, 512, 0, stream>>>(a);
      } else {
        if (gated) grouped_product_walk_kernel<256, true, true><<<grid, 512, 0, stream>>>(a);
        else if (act) grouped_product_walk_kernel<256, false, true><<<grid, 512, 0, stream>>>(a);
        else grouped_product_walk_kernel<256, false, false><<<grid, 512, 0, stream>>>(a);
      }
    } else if (tile_rows == 256) {                      // four wavefronts along the rows
      if (gated) grouped_product_mfma_kernel<4, 4, true, 4, 1><<<blocks(64), 256, 0, stream>>>(a);
      else grouped_product_mfma_kernel<4, 4, false, 4, 1><<<blocks(64), 256, 0, stream>>>(a);
    } else if (tile_rows == 128) {                      // two wavefronts along the rows, two along the columns
      if (gated) grouped_product_mfma_kernel<4, 4, true, 2, 2><<<blocks(128), 256, 0, stream>>>(a);
      else grouped_product_mfma_kernel<4, 4, false, 2, 2><<<blocks(128), 256, 0, stream>>>(a);
    } else if (pairs <= 8 * (long long)experts) {
      // (few rows an expert: the launch is bound by the matrices' stream, see the kernel.  Under six rows an
      // expert every one of its tiles is narrow; from there on the rows of x, read again by every column block,
      // count: 64 experts of 1,792, 8 rows each, 433 us in blocks of 16 columns and 400 in blocks of 32.  From
      // twelve rows on it is the kernel below that is faster: 12 rows of the 2,048 x 1,024 experts 152 against 160 us.)
      if (pairs < 6 * (long long)experts) {
        if (gated) grouped_product_few_kernel<1, true><<<blocks(16), 64 * FEW_WAVES, 0, stream>>>(a);
        else grouped_product_few_kernel<1, false><<<blocks(16), 64 * FEW_WAVES, 0, stream>>>(a);
      } else {
        if (gated) grouped_product_few_kernel<2, true><<<blocks(32), 64 * FEW_WAVES, 0, stream>>>(a);
        else grouped_product_few_kernel<2, false><<<blocks(32), 64 * FEW_WAVES, 0, stream>>>(a);
      }
    } else {
      if (gated) grouped_product_mfma_kernel<1, 4, true, 1, 1><<<blocks(64), 64, 0, stream>>>(a);
      else grouped_product_mfma_kernel<1, 4, false, 1, 1><<<blocks(64), 64, 0, stream>>>(a);
    }
    return sl_launch_status();
  }
#endif
  SL_CHECK(!w_tiled, "grouped_product: tiled matrices need K in steps of 32, N in steps of 16 and aligned operands");
  const dim3 grid(max_tiles * (tile_rows / RT_ROWS), (N + 63) / 64);
  if (gated) grouped_product_kernel<true><<<grid, 256, 0, stream>>>(a);
  else grouped_product_kernel<false><<<grid, 256, 0, stream>>>(a);
  return sl_launch_status();
}

// ------------------------------------------------------------------ combine
// out[t] = g[t] base[t] + sum_k shares[t][k] * y[place_of[t top + k]], float sums, choices in their order;
// g[t] = sigmoid(base_gate[t * gate_stride]) when base_gate is given, else 1 (shares == nullptr: all 1).  A choice from
// E_real on (chosen given) is an expert that hands its input through: it adds share * x[t].
__global__ __launch_bounds__(256) void routed_combine_kernel(const float* __restrict__ y,
                                                             const int* __restrict__ place_of,
                                                             const float* __restrict__ shares, int top,
                                                             const act_t* __restrict__ base,
                                                             const float* __restrict__ base_gate, int gate_stride,
                                                             int H, act_t* __restrict__ out,
                                                             const int* __restrict__ chosen, int E_real,
                                                             const act_t* __restrict__ x) {
  __shared__ int place[64];
  __shared__ float share[64];
  const size_t t = blockIdx.x;
  if (threadIdx.x < top) {
    const bool through = chosen != nullptr && chosen[t * top + threadIdx.x] >= E_real;
    place[threadIdx.x] = through ? -1 : place_of[t * top + threadIdx.x];
    share[threadIdx.x] = shares != nullptr ? shares[t * top + threadIdx.x] : 1.f;
  }
  __syncthreads();
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= H) return;
  float v = base != nullptr ? to_f(base[t * H + c]) : 0.f;
  if (base_gate != nullptr) v *= 1.f / (1.f + expf(-base_gate[t * gate_stride]));
  for (int k = 0; k < top; ++k)
    v += share[k] * (place[k] < 0 ? to_f(x[t * H + c]) : y[(size_t)place[k] * H + c]);
  out[t * H + c] = from_f<act_t>(v);
}

// The same, four channels a thread with 16-byte loads, eight choices' rows asked for at once: rows of a multiple of four values and
// aligned operands.  2,048 tokens of 8 choices, 2,048 channels, 150 MB: 39 us with a channel a thread, 26 here.  Few tokens are a chain of two
// trips in either, and the places of eight choices in registers are a longer one than two or ten of them in LDS: from 400,000 values
// on, and with five to eight choices (us, a channel a thread / here: 64 tokens of 2,048 channels, 2 choices 3.0 / 3.2, 10 3.8 / 3.9, 8 3.5 / 3.2; 200 tokens, 2
// choices 3.5 / 3.5, 10 4.6 / 4.3; 300 of 896, 2 choices 3.3 / 3.4, 500 3.6 / 3.5; 2,048 of 2,048, 2 choices 18.7 / 9.8).
struct __attribute__((aligned(16))) rc_f4 { float v[4]; };
struct __attribute__((aligned(4 * sizeof(act_t)))) rc_a4 { act_t v[4]; };
template <bool THROUGH>
__global__ __launch_bounds__(256) void routed_combine_vec_kernel(const float* __restrict__ y, const int* __restrict__ place_of,
                                                                 const float* __restrict__ shares, int top,
                                                                 const act_t* __restrict__ base, const float* __restrict__ base_gate,
                                                                 int gate_stride, int H, act_t* __restrict__ out,
                                                                 const int* __restrict__ chosen, int E_real,
                                                                 const act_t* __restrict__ x) {
  const size_t t = blockIdx.x;
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (c >= H) return;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  if (base != nullptr) {
    const rc_a4 b = *(const rc_a4*)(base + t * H + c);
    const float g = base_gate != nullptr ? 1.f / (1.f + expf(-base_gate[t * gate_stride])) : 1.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = base_gate != nullptr ? to_f(b.v[j]) * g : to_f(b.v[j]);
  }
  for (int k0 = 0; k0 < top; k0 += 8) {
    rc_f4 r[8];
    float share[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = min(k0 + u, top - 1);                                               // (the same for the whole workgroup)
      share[u] = shares != nullptr ? shares[t * top + k] : 1.f;
      if (THROUGH && chosen[t * top + k] >= E_real) {
        const rc_a4 a = *(const rc_a4*)(x + t * H + c);
#pragma unroll
        for (int j = 0; j < 4; ++j) r[u].v[j] = to_f(a.v[j]);
      } else r[u] = *(const rc_f4*)(y + (size_t)place_of[t * top + k] * H + c);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k0 + u < top)
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] += share[u] * r[u].v[j];
  }
  rc_a4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) o.v[j] = from_f<act_t>(v[j]);
  *(rc_a4*)(out + t * H + c) = o;
}

extern "C" const char* sl_routed_combine(const float* y, const int* place_of, const float* shares, int T, int top,
                                         const void* base, const float* base_gate, int gate_stride, int H,
                                         void* out, const int* chosen, int E_real, const void* x,
                                         hipStream_t stream) {
  SL_CHECK(T >= 0 && top >= 1 && top <= 64 && H > 0, "routed_combine: sizes must be positive, at most 64 choices");
  SL_CHECK(chosen == nullptr || x != nullptr, "routed_combine: experts that hand their input through need the input");
  if (T == 0) return nullptr;
  const bool vec = (long long)T * H >= 400000 || top % 8 == 0 || top % 8 > 4;
  if (vec && H % 4 == 0 && (uintptr_t)y % 16 == 0 && ((uintptr_t)base | (uintptr_t)out | (uintptr_t)x) % sizeof(rc_a4) == 0) {
    const int n = H >= 1024 ? 256 : (H / 4 + 63) / 64 * 64;
    auto run = [&](auto kernel) {
      kernel<<<dim3(T, (H / 4 + n - 1) / n), n, 0, stream>>>(y, place_of, shares, top, (const act_t*)base, base_gate, gate_stride, H,
                                                             (act_t*)out, chosen, E_real, (const act_t*)x);
    };
    if (chosen != nullptr) run(routed_combine_vec_kernel<true>);
    else run(routed_combine_vec_kernel<false>);
    return sl_launch_status();
  }
  routed_combine_kernel<<<dim3(T, (H + 255) / 256), 256, 0, stream>>>(y, place_of, shares, top, (const act_t*)base,
                                                                    base_gate, gate_stride, H, (act_t*)out,
                                                                    chosen, E_real, (const act_t*)x);
  return sl_launch_status();
}
