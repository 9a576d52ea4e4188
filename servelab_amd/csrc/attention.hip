// Attention over the paged cache: general kernel.
//
// For every query token t of the batch (sequence s = tok_seq[t], position
// p = positions[t]) and every query head h: keys r in [lo, p] of sequence s,
// lo = max(0, p - window + 1) with a window, else 0, found through the
// sequence's block table; score = (q . k_r) * scale; softmax over r; output
// sum_r P_r v_r; all in float with a running maximum and sum.  kv head of h is
// h / (nh / nkv).
//
// Reference: the per-sequence loop of servelab/parallel/tp_model.py:136-157
// (scores, causal mask, softmax, PV in float32) and the running-softmax form of
// servelab/attention/triton/paged_attention.py:39-74.  A prompt portion sees
// itself through the cache (its keys are written before this runs), so a
// decode token is just a portion of one token.  The window is this build's own.
//
// One wavefront per (token, head, share of the keys); lanes split 64 keys for
// the scores and the head's channels for the output.  With more than one share
// (few tokens, long contexts: a decode step) every wavefront leaves its
// unnormalised output, maximum and sum, and attention_general_combine_kernel
// merges them.  Any head size up to 256, any head counts,
// page sizes 16 / 32 / 64.  This is the kernel of the float32 path and the
// fallback of the bfloat16 path for sizes its matrix-core kernels refuse.
#include "common.h"

#define MAX_D 256

__global__ __launch_bounds__(64) void attention_general_kernel(
    const act_t* __restrict__ qkv, int row_stride, const act_t* __restrict__ kc,
    const act_t* __restrict__ vc, const int* __restrict__ block_tables, int max_pages,
    const int* __restrict__ tok_seq, const int* __restrict__ positions, int nh, int nkv, int D,
    int page, float scale, int window, act_t* __restrict__ out, int nsplit,
    float* __restrict__ part_o, float* __restrict__ part_ml) {
  __shared__ float qs[MAX_D];
  __shared__ float ps[64];
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const int s = tok_seq[t], p = positions[t];
  const int kvh = h / (nh / nkv);
  const int lo = window > 0 ? (p - window + 1 > 0 ? p - window + 1 : 0) : 0;
  const int* table = block_tables + (size_t)s * max_pages;
  const act_t* q = qkv + (size_t)t * row_stride + (size_t)h * D;
  for (int d = lane; d < D; d += 64) qs[d] = to_f(q[d]);
  __syncthreads();

  float m = -INFINITY, l = 0.f;
  float acc[MAX_D / 64];
#pragma unroll
  for (int i = 0; i < MAX_D / 64; ++i) acc[i] = 0.f;

  // blocks of 64 keys [first, p / 64]; this wavefront takes share blockIdx.z of them
  const int first = lo / 64, nblk = p / 64 + 1 - first;
  const int b0 = first + (int)((long long)nblk * blockIdx.z / nsplit);
  const int b1 = first + (int)((long long)nblk * (blockIdx.z + 1) / nsplit);
  for (int kb = b0 * 64; kb < b1 * 64; kb += 64) {
    const int r = kb + lane;
    const bool valid = r >= lo && r <= p;
    float sc = -INFINITY;
    if (valid) {
      const int pg = table[r / page];
      const act_t* kr = kc + (((size_t)pg * nkv + kvh) * page + r % page) * D;
      float dot = 0.f;
      for (int d = 0; d < D; ++d) dot += qs[d] * to_f(kr[d]);
      sc = dot * scale;
    }
    const float mn = fmaxf(m, wave_max(sc));       // every block holds a visible key
    const float alpha = expf(m - mn);              // exp(-inf) = 0 on the first block
    const float pr = valid ? expf(sc - mn) : 0.f;
    l = l * alpha + wave_sum(pr);
    m = mn;
    ps[lane] = pr;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < MAX_D / 64; ++i) acc[i] *= alpha;
    for (int pb = 0; pb < 64; pb += page) {
      const int r0 = kb + pb;
      if (r0 > p) break;
      if (r0 + page <= lo) continue;               // wholly before the window: may be released
      const int pg = table[r0 / page];
      const act_t* vbase = vc + ((size_t)pg * nkv + kvh) * D * page;
#pragma unroll
      for (int i = 0; i < MAX_D / 64; ++i) {
        const int d = lane + 64 * i;
        if (d < D) {
          const act_t* vr = vbase + (size_t)d * page;
          float a = acc[i];
          for (int j = 0; j < page; ++j) a += ps[pb + j] * to_f(vr[j]);
          acc[i] = a;
        }
      }
    }
    __syncthreads();
  }
  if (nsplit > 1) {
    const size_t pr = ((size_t)t * nh + h) * nsplit + blockIdx.z;
#pragma unroll
    for (int i = 0; i < MAX_D / 64; ++i) {
      const int d = lane + 64 * i;
      if (d < D) part_o[pr * D + d] = acc[i];
    }
    if (lane == 0) {
      part_ml[pr * 2] = m;
      part_ml[pr * 2 + 1] = l;
    }
    return;
  }
  const float inv = 1.f / l;
  act_t* o = out + ((size_t)t * nh + h) * D;
#pragma unroll
  for (int i = 0; i < MAX_D / 64; ++i) {
    const int d = lane + 64 * i;
    if (d < D) o[d] = from_f<act_t>(acc[i] * inv);
  }
}

// The same for up to GROUP_HEADS query heads of one kv head at a time: a decode
// row's heads of a group read the same keys and values, so one wavefront takes
// them together and every key row and value column is fetched once for all of
// them (the kernel above fetches it once per head).
constexpr int GROUP_HEADS = 8;
constexpr int PIECE = 16 / sizeof(act_t);
struct __attribute__((aligned(16))) att_piece { act_t v[PIECE]; };

__global__ __launch_bounds__(64) void attention_general_group_kernel(
    const act_t* __restrict__ qkv, int row_stride, const act_t* __restrict__ kc,
    const act_t* __restrict__ vc, const int* __restrict__ block_tables, int max_pages,
    const int* __restrict__ tok_seq, const int* __restrict__ positions, int nh, int nkv, int D,
    int page, float scale, int window, act_t* __restrict__ out, int nsplit,
    float* __restrict__ part_o, float* __restrict__ part_ml) {
  __shared__ float qs[GROUP_HEADS][MAX_D];
  __shared__ float ps[GROUP_HEADS][64];
  const int t = blockIdx.x, lane = threadIdx.x;
  const int g = nh / nkv, chunks = (g + GROUP_HEADS - 1) / GROUP_HEADS;
  const int kvh = blockIdx.y / chunks, h0 = kvh * g + (blockIdx.y % chunks) * GROUP_HEADS;
  const int nheads = kvh * g + g - h0 < GROUP_HEADS ? kvh * g + g - h0 : GROUP_HEADS;
  const int s = tok_seq[t], p = positions[t];
  const int lo = window > 0 ? (p - window + 1 > 0 ? p - window + 1 : 0) : 0;
  const int* table = block_tables + (size_t)s * max_pages;
  const bool aligned = ((uintptr_t)kc | (uintptr_t)vc) % 16 == 0, whole = aligned && D % PIECE == 0;
  for (int idx = lane; idx < GROUP_HEADS * D; idx += 64)      // rows past nheads: zeros, results never stored
    qs[idx / D][idx % D] = idx / D < nheads
        ? to_f(qkv[(size_t)t * row_stride + (size_t)(h0 + idx / D) * D + idx % D]) : 0.f;
  __syncthreads();

  float m[GROUP_HEADS], l[GROUP_HEADS], acc[GROUP_HEADS][MAX_D / 64];
#pragma unroll
  for (int h = 0; h < GROUP_HEADS; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int i = 0; i < MAX_D / 64; ++i) acc[h][i] = 0.f;
  }
  const int first = lo / 64, nblk = p / 64 + 1 - first;
  const int b0 = first + (int)((long long)nblk * blockIdx.z / nsplit);
  const int b1 = first + (int)((long long)nblk * (blockIdx.z + 1) / nsplit);
  for (int kb = b0 * 64; kb < b1 * 64; kb += 64) {
    const int r = kb + lane;
    const bool valid = r >= lo && r <= p;
    float dot[GROUP_HEADS];
#pragma unroll
    for (int h = 0; h < GROUP_HEADS; ++h) dot[h] = 0.f;
    if (valid) {
      const int pg = table[r / page];
      const act_t* kr = kc + (((size_t)pg * nkv + kvh) * page + r % page) * D;
      // (rows of whole 16-byte pieces: a lane's row is its own, so its loads are as wide as they can be, eight in flight)
      if (whole) {
#pragma unroll 8
        for (int d = 0; d < D; d += PIECE) {
          const att_piece kv = *(const att_piece*)(kr + d);
#pragma unroll
          for (int j = 0; j < PIECE; ++j)
#pragma unroll
            for (int h = 0; h < GROUP_HEADS; ++h) dot[h] += qs[h][d + j] * to_f(kv.v[j]);
        }
      } else {
        for (int d = 0; d < D; ++d) {
          const float kv = to_f(kr[d]);
#pragma unroll
          for (int h = 0; h < GROUP_HEADS; ++h) dot[h] += qs[h][d] * kv;
        }
      }
    }
    float alpha[GROUP_HEADS];
#pragma unroll
    for (int h = 0; h < GROUP_HEADS; ++h) {
      const float sc = valid ? dot[h] * scale : -INFINITY;
      const float mn = fmaxf(m[h], wave_max(sc));  // every block holds a visible key
      alpha[h] = expf(m[h] - mn);                  // exp(-inf) = 0 on the first block
      const float pr = valid ? expf(sc - mn) : 0.f;
      l[h] = l[h] * alpha[h] + wave_sum(pr);
      m[h] = mn;
      ps[h][lane] = pr;
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < GROUP_HEADS; ++h)
#pragma unroll
      for (int i = 0; i < MAX_D / 64; ++i) acc[h][i] *= alpha[h];
    for (int pb = 0; pb < 64; pb += page) {
      const int r0 = kb + pb;
      if (r0 > p) break;
      if (r0 + page <= lo) continue;               // wholly before the window: may be released
      const int pg = table[r0 / page];
      const act_t* vbase = vc + ((size_t)pg * nkv + kvh) * D * page;
#pragma unroll
      for (int i = 0; i < MAX_D / 64; ++i) {
        const int d = lane + 64 * i;
        if (d < D) {
          const act_t* vr = vbase + (size_t)d * page;
          // (a channel's keys of a page lie together: pages of 16, 32 or 64 keys are whole pieces)
          if (aligned) {
#pragma unroll 4
            for (int j = 0; j < page; j += PIECE) {
              const att_piece v = *(const att_piece*)(vr + j);
#pragma unroll
              for (int e = 0; e < PIECE; ++e)
#pragma unroll
                for (int h = 0; h < GROUP_HEADS; ++h) acc[h][i] += ps[h][pb + j + e] * to_f(v.v[e]);
            }
          } else {
            for (int j = 0; j < page; ++j) {
              const float v = to_f(vr[j]);
#pragma unroll
              for (int h = 0; h < GROUP_HEADS; ++h) acc[h][i] += ps[h][pb + j] * v;
            }
          }
        }
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int h = 0; h < GROUP_HEADS; ++h) {
    if (h >= nheads) break;
    const size_t row = (size_t)t * nh + h0 + h;
    if (nsplit > 1) {
#pragma unroll
      for (int i = 0; i < MAX_D / 64; ++i) {
        const int d = lane + 64 * i;
        if (d < D) part_o[(row * nsplit + blockIdx.z) * D + d] = acc[h][i];
      }
      if (lane == 0) {
        part_ml[(row * nsplit + blockIdx.z) * 2] = m[h];
        part_ml[(row * nsplit + blockIdx.z) * 2 + 1] = l[h];
      }
    } else {
      const float inv = 1.f / l[h];
#pragma unroll
      for (int i = 0; i < MAX_D / 64; ++i) {
        const int d = lane + 64 * i;
        if (d < D) out[row * D + d] = from_f<act_t>(acc[h][i] * inv);
      }
    }
  }
}

// The same for single tokens whose keys are shared out over wavefronts (and so are few a wavefront): blocks of 16 keys, four lanes a
// key, each a quarter of its channels, and everything of a block asked for at once, the next block's keys and values while this one's
// are multiplied.  A block of 64 keys, a lane each, is 10 trips to memory and a chain of 96 exchanges between lanes
// for one wavefront, and 333 keys make six of them a pair of heads, on 256 CUs.
// With its combine kernel, us a layer, before / here: 12 heads on 2 of 128, 1 request at 40 / 333 / 4,000 keys 26 / 16, 28 / 16 and 28 / 28,
// 3 at 333 29 / 17, 6 at 600 29 / 18; 14 on 2 of 64, 1 and 6 requests 18 / 11 and 19 / 12.  It takes most of a SIMD's registers, so
// that it pays while every wavefront has a SIMD to itself (16 requests at 4,000 keys, 2,048 wavefronts: 42 / 58); heads of 256
// do not fit them (1 request at 4,000: 46 / 57).
template <bool MAX> __device__ __forceinline__ float over_keys(float v) {      // 16 keys, the four lanes of a key alike
  auto meet = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
  v = meet(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, true)));   // the other key of two
  v = meet(v, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, true)));   // the other two of four
  return column_meet(v, meet);
}
template <int HD>
__global__ __launch_bounds__(64) void attention_few_keys_kernel(
    const act_t* __restrict__ qkv, int row_stride, const act_t* __restrict__ kc,
    const act_t* __restrict__ vc, const int* __restrict__ block_tables, int max_pages,
    const int* __restrict__ tok_seq, const int* __restrict__ positions, int nh, int nkv,
    int page, float scale, int window, int nsplit, float* __restrict__ part_o, float* __restrict__ part_ml) {
  constexpr int KU = HD / (4 * PIECE), VI = (HD + 63) / 64, VU = 16 / PIECE;   // pieces of a key a lane holds; channels, pieces of each
  static_assert(KU * 4 * PIECE == HD, "four lanes a key, whole pieces");
  __shared__ __attribute__((aligned(16))) float qs[GROUP_HEADS][HD];
  __shared__ __attribute__((aligned(16))) float ps[GROUP_HEADS][16];
  const int t = blockIdx.x, lane = threadIdx.x, key = lane >> 2, part = lane & 3;
  const int g = nh / nkv, chunks = (g + GROUP_HEADS - 1) / GROUP_HEADS;
  const int kvh = blockIdx.y / chunks, h0 = kvh * g + (blockIdx.y % chunks) * GROUP_HEADS;
  const int nheads = kvh * g + g - h0 < GROUP_HEADS ? kvh * g + g - h0 : GROUP_HEADS;
  const int s = tok_seq[t], p = positions[t];
  const int lo = window > 0 ? (p - window + 1 > 0 ? p - window + 1 : 0) : 0;
  const int* table = block_tables + (size_t)s * max_pages;
  const int first = lo / 16, nblk = p / 16 + 1 - first;
  const int b0 = first + (int)((long long)nblk * blockIdx.z / nsplit);
  const int b1 = first + (int)((long long)nblk * (blockIdx.z + 1) / nsplit);
  float m[GROUP_HEADS], l[GROUP_HEADS], acc[GROUP_HEADS][VI];
#pragma unroll
  for (int h = 0; h < GROUP_HEADS; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int i = 0; i < VI; ++i) acc[h][i] = 0.f;
  }
  struct block { att_piece k[KU], v[VI][VU]; };
  auto load = [&](int b) {                              // (16 keys lie in one page; every key of a page is there to be read)
    block r;
    const size_t row = (size_t)table[16 * b / page] * nkv + kvh;
    const int at = 16 * b % page;
    const act_t* kr = kc + (row * page + at + key) * HD + PIECE * part;
#pragma unroll
    for (int u = 0; u < KU; ++u) r.k[u] = *(const att_piece*)(kr + 4 * PIECE * u);
#pragma unroll
    for (int i = 0; i < VI; ++i) {
      const int d = lane + 64 * i < HD ? lane + 64 * i : HD - 1;
#pragma unroll
      for (int u = 0; u < VU; ++u) r.v[i][u] = *(const att_piece*)(vc + (row * HD + d) * page + at + PIECE * u);
    }
    return r;
  };
  block now;
  if (b0 < b1) {
    now = load(b0);
    // (asked for together and without conditions: a value a trip, this was most of the kernel's time)
    constexpr int NQ = GROUP_HEADS * HD / 64;
    act_t q[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int h = (lane + 64 * i) / HD, d = (lane + 64 * i) % HD;
      q[i] = qkv[(size_t)t * row_stride + (size_t)(h0 + (h < nheads ? h : nheads - 1)) * HD + d];
    }
#pragma unroll
    for (int i = 0; i < NQ; ++i)                                // (rows past nheads: the last again, results never stored)
      qs[(lane + 64 * i) / HD][(lane + 64 * i) % HD] = to_f(q[i]);
  }
  __syncthreads();
  for (int b = b0; b < b1; ++b) {
    block ahead = now;
    if (b + 1 < b1) ahead = load(b + 1);
    const int r = 16 * b + key;
    const bool valid = r >= lo && r <= p;
    float dot[GROUP_HEADS];
#pragma unroll
    for (int h = 0; h < GROUP_HEADS; ++h) dot[h] = 0.f;
#pragma unroll
    for (int u = 0; u < KU; ++u)
#pragma unroll
      for (int h = 0; h < GROUP_HEADS; ++h)
#pragma unroll
        for (int j = 0; j < PIECE; ++j) dot[h] += qs[h][PIECE * (part + 4 * u) + j] * to_f(now.k[u].v[j]);
#pragma unroll
    for (int h = 0; h < GROUP_HEADS; ++h) {
      float d = dot[h];
      d += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(d), 0xB1, 0xf, 0xf, true));
      d += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(d), 0x4E, 0xf, 0xf, true));
      const float sc = valid ? d * scale : -INFINITY;
      const float mn = fmaxf(m[h], over_keys<true>(sc));
      const float from = mn == -INFINITY ? 0.f : mn;            // (16 keys may well have no score above minus infinity: they weigh nothing)
      const float alpha = expf(m[h] - from), pr = valid ? expf(sc - from) : 0.f;  // exp(-inf) = 0 on the first block
      l[h] = l[h] * alpha + over_keys<false>(pr);
      m[h] = mn;
      if (part == 0) ps[h][key] = pr;
#pragma unroll
      for (int i = 0; i < VI; ++i) acc[h][i] *= alpha;
    }
    __syncthreads();
    const bool whole = 16 * b >= lo && 16 * b + 15 <= p;        // (a weight of 0 times what lies in an unseen place may be no number)
#pragma unroll
    for (int u = 0; u < VU; ++u)
#pragma unroll
      for (int e = 0; e < PIECE; ++e) {
        const int j = PIECE * u + e;
        const bool seen = whole || (16 * b + j >= lo && 16 * b + j <= p);
#pragma unroll
        for (int i = 0; i < VI; ++i) {
          const float v = seen ? to_f(now.v[i][u].v[e]) : 0.f;
#pragma unroll
          for (int h = 0; h < GROUP_HEADS; ++h) acc[h][i] += ps[h][j] * v;
        }
      }
    __syncthreads();
    now = ahead;
  }
#pragma unroll
  for (int h = 0; h < GROUP_HEADS; ++h) {
    if (h >= nheads) break;
    const size_t row = ((size_t)t * nh + h0 + h) * nsplit + blockIdx.z;
#pragma unroll
    for (int i = 0; i < VI; ++i) {
      const int d = lane + 64 * i;
      if (d < HD) part_o[row * HD + d] = acc[h][i];
    }
    if (lane == 0) {
      part_ml[row * 2] = m[h];
      part_ml[row * 2 + 1] = l[h];
    }
  }
}

// out[t, h, :] = sum_j w_j o_j / sum_j w_j l_j,  w_j = exp(m_j - max m); a share
// without keys has m = -inf and l = 0 and drops out.  One wavefront per (t, h, 64 channels).  Up to SHARES shares' outputs are
// asked for with their maxima, one trip to memory for all; behind the weights, sixteen at a time and the channels' halves one after the
// other, three requests of 333 tokens took 8.0 us, now 4.7.  Added in the order of the shares.
template <int SHARES>
__global__ __launch_bounds__(64) void attention_general_combine_kernel(
    const float* __restrict__ part_o, const float* __restrict__ part_ml, int nsplit, int nh, int D,
    act_t* __restrict__ out) {
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, d = blockIdx.z * 64 + lane, at = min(d, D - 1);
  const size_t base = ((size_t)t * nh + h) * nsplit, mine = (base + min(lane, nsplit - 1)) * 2;
  float m = part_ml[mine], l = part_ml[mine + 1], v[SHARES];
#pragma unroll
  for (int u = 0; u < SHARES; ++u) v[u] = part_o[(base + min(u, nsplit - 1)) * D + at];
  __builtin_amdgcn_sched_barrier(0);
  if (lane >= nsplit) m = -INFINITY, l = 0.f;
  const float mx = wave_max(m);
  const float w = m == -INFINITY ? 0.f : expf(m - mx);
  const float denom = wave_sum(w * l);
  float a = 0.f;
#pragma unroll
  for (int u = 0; u < SHARES; ++u)                     // (past the last: nothing, whatever came)
    a += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), u)) * (u < nsplit ? v[u] : 0.f);
  if (d < D) out[((size_t)t * nh + h) * D + d] = from_f<act_t>(a / denom);
}

// ---------------------------------------------------------------------------
// Prompt portions, general sizes.  The kernel above gives a wavefront to every
// (token, head) and lets it read its keys from the cache itself: for a prompt
// of thousands of tokens every key row is fetched thousands of times.  Here a
// workgroup of four wavefronts owns TILE_COLS columns, a column being a (token,
// head of the group) pair of one sequence and one kv head, and walks the key
// blocks its columns see: a block of KB keys and values is staged in LDS as
// floats once and serves all columns; 16 lanes share a column, splitting a
// block's keys for the scores and the head's channels for the output.  Float
// FMAs only, running maximum and sum per column as above.
// ---------------------------------------------------------------------------
constexpr int TILE_COLS = 16;
constexpr int TILE_THREADS = 256;

template <int KB>
__global__ __launch_bounds__(TILE_THREADS) void attention_general_tile_kernel(
    const act_t* __restrict__ qkv, int row_stride, const act_t* __restrict__ kc,
    const act_t* __restrict__ vc, const int* __restrict__ block_tables, int max_pages,
    const int* __restrict__ cu_q, const int* __restrict__ positions, int nh, int nkv, int D,
    int page, float scale, int window, act_t* __restrict__ out) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int KS = D + 4, VS = D + 1;                  // row strides: K rows are read 16 bytes at a time, by 16 rows at once
  float* qs = lds;                                   // [TILE_COLS][D]
  float* ks = qs + TILE_COLS * D;                    // [KB][KS]
  float* vs = ks + KB * KS;                          // [KB][VS]
  float* ps = vs + KB * VS;                          // [TILE_COLS][KB]
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int sub = lane & 15;                         // this lane's place among the 16 of its column
  const int col = 4 * wave + (lane >> 4);            // column of the tile
  const int seq = blockIdx.z, kvh = blockIdx.y;
  const int g = nh / nkv;
  const int q0 = cu_q[seq], qlen = cu_q[seq + 1] - q0;
  const int ncols = qlen * g;
  const int c0 = blockIdx.x * TILE_COLS;
  if (c0 >= ncols) return;
  const int pos0 = positions[q0];
  const int* table = block_tables + (size_t)seq * max_pages;

  // the tile's columns and the keys any of them sees
  const int c = c0 + col;
  const bool live = c < ncols;
  const int tok = live ? c / g : 0, head = kvh * g + (live ? c % g : 0);
  const int pos_c = live ? pos0 + tok : -1;
  const int lo_c = window > 0 && pos_c - window + 1 > 0 ? pos_c - window + 1 : 0;
  const int tok_first = c0 / g;
  const int c_last = c0 + TILE_COLS - 1 < ncols - 1 ? c0 + TILE_COLS - 1 : ncols - 1;
  const int kmax = pos0 + c_last / g;
  int kmin = 0;
  if (window > 0 && pos0 + tok_first - window + 1 > 0) kmin = pos0 + tok_first - window + 1;

  for (int idx = t; idx < TILE_COLS * D; idx += TILE_THREADS) {
    const int cc = c0 + idx / D, d = idx % D;
    qs[idx] = cc < ncols ? to_f(qkv[(size_t)(q0 + cc / g) * row_stride + (size_t)(kvh * g + cc % g) * D + d]) : 0.f;
  }

  float m = -INFINITY, l = 0.f;
  float acc[MAX_D / 16];
#pragma unroll
  for (int j = 0; j < MAX_D / 16; ++j) acc[j] = 0.f;
  const int nd16 = D / 16;

  for (int kb = kmin / KB; kb <= kmax / KB; ++kb) {
    const int kbase = kb * KB;
    __syncthreads();                                 // the last block's readers are done (and qs is written)
    for (int idx = t; idx < KB * D; idx += TILE_THREADS) {
      {                                              // K: consecutive threads along a key's channels
        const int key = kbase + idx / D, d = idx % D;
        float v = 0.f;
        if (key >= kmin && key <= kmax) {
          const int pg = table[key / page];
          v = to_f(kc[(((size_t)pg * nkv + kvh) * page + key % page) * D + d]);
        }
        ks[(idx / D) * KS + d] = v;
      }
      {                                              // V^T in the cache: consecutive threads along a channel's keys
        const int kk = idx % KB, d = idx / KB, key = kbase + kk;
        float v = 0.f;
        if (key >= kmin && key <= kmax) {
          const int pg = table[key / page];
          v = to_f(vc[(((size_t)pg * nkv + kvh) * D + d) * page + key % page]);
        }
        vs[kk * VS + d] = v;
      }
    }
    __syncthreads();
    // scores of this lane's keys sub, sub + 16, ... of the block
    float sc[KB / 16];
#pragma unroll
    for (int r = 0; r < KB / 16; ++r) sc[r] = 0.f;
    const float* qrow = qs + col * D;
    for (int d = 0; d < D; d += 4) {
      const float4 q4 = *(const float4*)(qrow + d);
#pragma unroll
      for (int r = 0; r < KB / 16; ++r) {
        const float4 k4 = *(const float4*)(ks + (sub + 16 * r) * KS + d);
        sc[r] += q4.x * k4.x + q4.y * k4.y + q4.z * k4.z + q4.w * k4.w;
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < KB / 16; ++r) {
      const int key = kbase + sub + 16 * r;
      sc[r] = key >= lo_c && key <= pos_c ? sc[r] * scale : -INFINITY;
      mx = fmaxf(mx, sc[r]);
    }
    mx = row_meet(mx, max_f);
    const float mn = fmaxf(m, mx);
    // a column that has seen no key yet keeps m = -inf: nothing to rescale, nothing to add
    const float alpha = mn == -INFINITY ? 1.f : expf(m - mn);
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < KB / 16; ++r) {
      const float pr = sc[r] == -INFINITY ? 0.f : expf(sc[r] - mn);
      psum += pr;
      ps[col * KB + sub + 16 * r] = pr;
    }
    psum = row_meet(psum, add_f);
    l = l * alpha + psum;
    m = mn;
    __syncthreads();                                 // ps is complete
#pragma unroll
    for (int j = 0; j < MAX_D / 16; ++j) acc[j] *= alpha;
    const float* prow = ps + col * KB;
    for (int kk = 0; kk < KB; ++kk) {
      const float pk = prow[kk];
      const float* vrow = vs + kk * VS + sub;
#pragma unroll
      for (int j = 0; j < MAX_D / 16; ++j)
        if (j < nd16) acc[j] += pk * vrow[16 * j];
    }
  }
  if (!live) return;
  const float inv = 1.f / l;
  act_t* o = out + ((size_t)(q0 + tok) * nh + head) * D + sub;
#pragma unroll
  for (int j = 0; j < MAX_D / 16; ++j)
    if (j < nd16) o[16 * j] = from_f<act_t>(acc[j] * inv);
}

#if defined(SL_F32)
// ---------------------------------------------------------------------------
// Prompt portions in float32 on the matrix cores (v_mfma_f32_16x16x4_f32: float32 factors and sums), for head sizes in
// steps of 16 fixed at compile time.  A workgroup of four wavefronts owns columns, (token, head of the group) pairs of one sequence and
// one kv head, a wavefront 16 of them: 64 columns, or 32 in two teams that walk every other block of keys and meet at the end.  Blocks
// are 32 keys, staged in LDS as K [32][D + 4] and V^T [D][36]; a team's next one travels from the pages to registers meanwhile.  S^T = K Q^T, softmax with a running
// maximum per column, O^T += V^T P^T: a lane's scores of a 16 x 16 block (keys 4 (lane / 16) .. + 3 of column lane % 16) are the
// second product's operand as they are.  What bounds it is the matrix instructions of the longest tile: 128 a block and
// wavefront at D 128, 1.7 us.  One prompt of 333 tokens and two shorter ones, 12 heads on 2, D 128: 287 us with the FMA tiles, 74 with
// four wavefronts over 64 columns and loads behind conditions, 45 without those, 41 with two teams over 64 columns, 31 with two over 32.  The second product multiplies the zero weights of keys that a column does not see too, which an infinite or NaN
// value turns into NaN: a wavefront with a result that is not finite takes its columns again key by key, over seen keys alone.
// ---------------------------------------------------------------------------
typedef float att_v4 __attribute__((ext_vector_type(4)));

template <int D, int TEAMS>
__global__ __launch_bounds__(256) void attention_f32_mfma_kernel(
    const float* __restrict__ qkv, int row_stride, const float* __restrict__ kc, const float* __restrict__ vc,
    const int* __restrict__ block_tables, int max_pages, const int* __restrict__ cu_q, const int* __restrict__ positions,
    int nh, int nkv, int page, float scale, int window, float* __restrict__ out) {
  constexpr int TEAM = 256 / TEAMS, COLS = 64 / TEAMS; // threads of a team, and the columns that all teams share
  constexpr int KR = D + 4, VR = 36, NP = 8 * D / TEAM;      // row lengths; 16-byte pieces of K and of V^T a thread stages of a block
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const int team = __builtin_amdgcn_readfirstlane(threadIdx.x / TEAM), tid = threadIdx.x % TEAM;
  float* ks = lds + team * (32 * KR + D * VR);         // [32][KR]
  float* vt = ks + 32 * KR;                            // [D][VR]
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, gq = lane >> 4;
  const int seq = blockIdx.z, kvh = blockIdx.y, g = nh / nkv;
  const int q0 = cu_q[seq], qlen = cu_q[seq + 1] - q0, ncols = qlen * g;
  // (tiles of late tokens see the most keys: they come first)
  const int tile = (int)gridDim.x - 1 - (int)blockIdx.x, c0 = tile * COLS;
  if (c0 >= ncols) return;
  const int pos0 = positions[q0];
  const int* table = block_tables + (size_t)seq * max_pages;
  const int c_last = min(c0 + COLS - 1, ncols - 1);
  const int kmax = pos0 + c_last / g;
  const int kmin = window > 0 ? max(0, pos0 + c0 / g - window + 1) : 0;
  const int cw = c0 + 16 * wave;
  const bool wave_live = cw < ncols;
  const int c = min(cw + n, ncols - 1);                // (a column past the last is computed like the last, never stored)
  const int tok = c / g, head = kvh * g + c % g, pos_c = pos0 + tok;
  const int lo_c = window > 0 ? max(0, pos_c - window + 1) : 0;
  att_v4 qf[D / 16];
  {
    const float* q = qkv + (size_t)(q0 + tok) * row_stride + (size_t)head * D + 4 * gq;
#pragma unroll
    for (int j = 0; j < D / 16; ++j) qf[j] = *(const att_v4*)(q + 16 * j);
  }
  att_v4 o[D / 16];
#pragma unroll
  for (int j = 0; j < D / 16; ++j) o[j] = att_v4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  att_v4 kr[NP], vr[NP];
  // A half of a block (16 keys, of one page) is read where it lies, its page asked for a block earlier, no load behind a condition (the
  // compiler waits for a load where the two ways meet: eight loads a thread, each behind its page's, were sixteen trips to memory a
  // block in turn).  A half of which no column sees a key may have no page: the other half stands for it.  Keys outside
  // [kmin, kmax] get no weight, and their values are staged as zeros: a slot that holds no visible key may hold anything.
  auto ask_pages = [&](int kbase) { return table[min(kbase + ((lane & 1) << 4), kmax) / page]; };
  auto fetch = [&](int kbase, int asked) {
    const int pgA = __builtin_amdgcn_readlane(asked, 0), pgB = __builtin_amdgcn_readlane(asked, 1);
    const bool seenA = kbase + 15 >= kmin, seenB = kbase + 16 <= kmax;
    const size_t headA = (size_t)(seenA ? pgA : pgB) * nkv + kvh, headB = (size_t)(seenB ? pgB : pgA) * nkv + kvh;
    const int inA = (seenA ? kbase : kbase + 16) % page, inB = (seenB ? kbase + 16 : kbase) % page;
    const float *keysA = kc + (headA * page + inA) * D, *keysB = kc + (headB * page + inB) * D;
    const float *valuesA = vc + headA * D * page + inA, *valuesB = vc + headB * D * page + inB;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int idx = tid + TEAM * i, kl = idx / (D / 4) & 15, d4 = idx % (D / 4);
      kr[i] = *(const att_v4*)((i >= NP / 2 ? keysB : keysA) + kl * D + 4 * d4);      // (the first NP / 2 pieces are 16 rows)
      vr[i] = *(const att_v4*)((idx & 4 ? valuesB : valuesA) + (idx / 8) * page + 4 * (idx & 3));
    }
  };
  const int b0 = kmin / 32, b1 = kmax / 32;
  const int mine = b0 + team;
  int asked = 0;
  if (mine <= b1) {
    fetch(32 * mine, ask_pages(32 * mine));
    if (mine + TEAMS <= b1) asked = ask_pages(32 * (mine + TEAMS));
  }
  for (int b = mine; b - team <= b1; b += TEAMS) {   // (as many rounds for both teams; the second may have no block in the last)
    const int kbase = 32 * b;
    __syncthreads();                                   // the last block's readers are done
    const bool all_seen = kbase >= kmin && kbase + 31 <= kmax;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int idx = tid + TEAM * i;
      if (!all_seen) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = kbase + 4 * (idx % 8) + e;
          vr[i][e] = (key >= kmin) & (key <= kmax) ? vr[i][e] : 0.f;
        }
      }
      *(att_v4*)(ks + (idx / (D / 4)) * KR + 4 * (idx % (D / 4))) = kr[i];
      *(att_v4*)(vt + (idx / 8) * VR + 4 * (idx % 8)) = vr[i];
    }
    __syncthreads();
    if (b + TEAMS <= b1) {
      fetch(kbase + 32 * TEAMS, asked);
      if (b + 2 * TEAMS <= b1) asked = ask_pages(kbase + 64 * TEAMS);
    }
    if (!wave_live || b > b1) continue;                          // (a wavefront without columns only helps staging)
    att_v4 s[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      att_v4 sum[2] = {};
      const float* kp = ks + (16 * kt + n) * KR + 4 * gq;
#pragma unroll
      for (int j = 0; j < D / 16; ++j) {
        const att_v4 kv = *(const att_v4*)(kp + 16 * j);
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[j & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[i], qf[j][i], sum[j & 1], 0, 0, 0);
      }
      s[kt] = sum[0] + sum[1];
    }
    float top = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = kbase + 16 * kt + 4 * gq + i;
        s[kt][i] = (key >= lo_c) & (key <= pos_c) ? s[kt][i] * scale : -INFINITY;      // (no branches)
        top = fmaxf(top, s[kt][i]);
      }
    top = column_meet(top, max_f);
    const float mn = fmaxf(m, top);
    // a column that has seen no key yet keeps m = -inf: nothing to rescale, nothing to add
    const float alpha = mn == -INFINITY ? 1.f : expf(m - mn);
    float psum = 0.f;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[kt][i] = s[kt][i] == -INFINITY ? 0.f : expf(s[kt][i] - mn);
        psum += s[kt][i];
      }
    l = l * alpha + psum;                              // (this lane's keys; the column's four lanes are added at the end)
    m = mn;
#pragma unroll
    for (int dd = 0; dd < D / 16; ++dd) {
      att_v4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const att_v4 vv = *(const att_v4*)(vt + (16 * dd + n) * VR + 16 * kt + 4 * gq);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[i], s[kt][i], acc, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) o[dd][i] = fmaf(o[dd][i], alpha, acc[i]);
    }
  }
  // the first team takes what the second has of its columns
  if constexpr (TEAMS == 2) {
    att_v4* os = (att_v4*)lds;                           // [D / 16][TEAM]
    float2* ml = (float2*)(os + TEAM * (D / 16));
    __syncthreads();
    if (team == 1) {
#pragma unroll
      for (int dd = 0; dd < D / 16; ++dd) os[TEAM * dd + tid] = o[dd];
      ml[tid] = make_float2(m, l);
    }
    __syncthreads();
    if (team == 1) return;
    const float2 other = ml[tid];
    const float both = fmaxf(m, other.x), ours = m == -INFINITY ? 0.f : expf(m - both), theirs = other.x == -INFINITY ? 0.f : expf(other.x - both);
#pragma unroll
    for (int dd = 0; dd < D / 16; ++dd) {
      const att_v4 x = os[TEAM * dd + tid];
#pragma unroll
      for (int i = 0; i < 4; ++i) o[dd][i] = fmaf(x[i], theirs, o[dd][i] * ours);
    }
    l = fmaf(other.y, theirs, l * ours);
    m = both;
  }
  l = column_meet(l, add_f);
  float odd = 0.f;                                     // (0, or NaN where a result is not finite)
#pragma unroll
  for (int dd = 0; dd < D / 16; ++dd) odd = fmaf((o[dd][0] + o[dd][1]) + (o[dd][2] + o[dd][3]), 0.f, odd);
  if (__ballot(odd != 0.f)) {
#pragma unroll
    for (int dd = 0; dd < D / 16; ++dd) o[dd] = att_v4{0.f, 0.f, 0.f, 0.f};
    m = -INFINITY;
    l = 0.f;
#pragma unroll 1
    for (int key = kmin; key <= kmax; ++key) {
      const size_t at = (size_t)table[key / page] * nkv + kvh;
      const float* kp = kc + (at * page + key % page) * D + 4 * gq;
      const float* vp = vc + (at * D + 4 * gq) * page + key % page;
      float sc = 0.f;                                  // this lane's quarter of the channels: those that it holds of q and o
#pragma unroll
      for (int j = 0; j < D / 16; ++j) {
        const att_v4 kv = *(const att_v4*)(kp + 16 * j);
#pragma unroll
        for (int i = 0; i < 4; ++i) sc = fmaf(qf[j][i], kv[i], sc);
      }
      sc = column_meet(sc, add_f);
      if (key < lo_c || key > pos_c) continue;
      sc *= scale;
      const float mn = fmaxf(m, sc), alpha = mn == -INFINITY ? 1.f : expf(m - mn), p = sc == -INFINITY ? 0.f : expf(sc - mn);
      l = fmaf(l, alpha, p);
      m = mn;
#pragma unroll
      for (int dd = 0; dd < D / 16; ++dd)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[dd][i] = fmaf(p, vp[(16 * dd + i) * page], o[dd][i] * alpha);
    }
  }
  if (cw + n >= ncols) return;
  const float inv = 1.f / l;
  float* to = out + ((size_t)(q0 + tok) * nh + head) * D + 4 * gq;
#pragma unroll
  for (int dd = 0; dd < D / 16; ++dd) *(att_v4*)(to + 16 * dd) = o[dd] * inv;
}
#endif

// Sequences [0, num_seqs) of the batch, prompt portions of at most max_q_len
// tokens each, `tokens` in all, that see at most `longest` keys (their tokens come first in the batch).  D % 16 == 0.
extern "C" const char* sl_attention_general_tiles(
    const void* qkv, int row_stride, const void* kc, const void* vc, const int* block_tables,
    int max_pages, const int* cu_q, const int* positions, int num_seqs, int max_q_len, int tokens, int longest, int nh,
    int nkv, int D, int page, float scale, int window, void* out, hipStream_t stream) {
  SL_CHECK(num_seqs >= 0 && max_q_len >= 1 && nh > 0 && nkv > 0 && nh % nkv == 0,
           "attention tiles: heads must be a positive multiple of kv heads");
  SL_CHECK(D > 0 && D <= MAX_D && D % 16 == 0, "attention tiles: head_dim must be a multiple of 16 up to 256");
  SL_CHECK(page == 16 || page == 32 || page == 64, "attention tiles: page size must be 16, 32 or 64");
  SL_CHECK(nkv <= 65535 && num_seqs <= 65535, "attention tiles: grid too large");
  SL_CHECK(window >= 0, "attention tiles: window must be >= 0 (0 = none)");
  if (num_seqs == 0) return nullptr;
  const long long cols = (long long)max_q_len * (nh / nkv);
  const long long tiles = (cols + TILE_COLS - 1) / TILE_COLS;
  SL_CHECK(tiles <= 1 << 30, "attention tiles: too many column tiles");
  const dim3 grid((unsigned)tiles, nkv, num_seqs);
#if defined(SL_F32)
  // (head sizes of the shapes served; from 32 columns on they win at every length measured)
  if ((D == 64 || D == 128) && cols >= 32 && row_stride % 4 == 0 && (uintptr_t)qkv % 16 == 0 && (uintptr_t)kc % 16 == 0 &&
      (uintptr_t)vc % 16 == 0 && (uintptr_t)out % 16 == 0) {
    // Two teams shorten a workgroup, one lets the chip hold twice as many columns: by the number of one team's workgroups beside the
    // keys, of which a team of two has none in a context of one block.  Of 438 prompts and batches of seven head shapes the form chosen takes 1.002 of the
    // faster one's time on average, 1.13 at worst (us, one / two: 14 heads on 2 of 64, 64 prompts of 70 tokens 25 / 36, 16 of 70 11.4 / 12.8, 16 of 150 30 / 25;
    // 32 on 8 of 128, 32 of 20 15 / 22, 64 of 100 115 / 156, 4 of 700 232 / 240; 12 on 2, three of 512, 100 and 30 64 / 39).
    const int g = nh / nkv;
    const long long least = nkv * (((long long)tokens * g + 63) / 64), workgroups = least > (long long)nkv * num_seqs ? least : (long long)nkv * num_seqs;
    const long long line = device_cus() / 4 + 2ll * longest;
    const bool few = longest > 32 && workgroups <= (D == 64 ? line + line / 2 : line);
    const long long columns = few ? 32 : 64;
    // (among sequences of very different lengths an odd number of places each: workgroups go to the eight dies in turn, and by a multiple of
    // eight the first tiles of all sequences would be one die's; a prompt of 1,000 tokens beside 15 steps of two at 500 keys, 16 heads of 128, 586 us, 123 so)
    const bool unequal = 4ll * tokens < 3ll * num_seqs * max_q_len;
    const dim3 wide((unsigned)((cols + columns - 1) / columns) | (unsigned)unequal, nkv, num_seqs);
    const size_t room = (few ? 2 : 1) * sizeof(float) * ((size_t)32 * (D + 4) + (size_t)D * 36);
    const char* failed = nullptr;
    auto run = [&](auto kernel) {
      const hipError_t e = room <= 48 * 1024 ? hipSuccess : hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)room);
      if (e != hipSuccess) {
        failed = hipGetErrorString(e);
        return;
      }
      kernel<<<wide, 256, room, stream>>>((const float*)qkv, row_stride, (const float*)kc, (const float*)vc, block_tables,
                                          max_pages, cu_q, positions, nh, nkv, page, scale, window, (float*)out);
    };
    if (few && D == 64) run(attention_f32_mfma_kernel<64, 2>);
    else if (few) run(attention_f32_mfma_kernel<128, 2>);
    else if (D == 64) run(attention_f32_mfma_kernel<64, 1>);
    else run(attention_f32_mfma_kernel<128, 1>);
    return failed != nullptr ? failed : sl_launch_status();
  }
#endif
  const int KB = D <= 128 ? 32 : 16;
  const size_t bytes = sizeof(float) * ((size_t)TILE_COLS * D + (size_t)KB * (D + 4) + (size_t)KB * (D + 1) +
                                        (size_t)TILE_COLS * KB);
  SL_CHECK(bytes <= 65536, "attention tiles: LDS need exceeds 64 KB");
  if (KB == 32)
    attention_general_tile_kernel<32><<<grid, TILE_THREADS, bytes, stream>>>(
        (const act_t*)qkv, row_stride, (const act_t*)kc, (const act_t*)vc, block_tables, max_pages,
        cu_q, positions, nh, nkv, D, page, scale, window, (act_t*)out);
  else
    attention_general_tile_kernel<16><<<grid, TILE_THREADS, bytes, stream>>>(
        (const act_t*)qkv, row_stride, (const act_t*)kc, (const act_t*)vc, block_tables, max_pages,
        cu_q, positions, nh, nkv, D, page, scale, window, (act_t*)out);
  return sl_launch_status();
}

// nsplit > 1: part_o holds T * nh * nsplit * D floats, part_ml T * nh * nsplit * 2.
extern "C" const char* sl_attention_general(
    const void* qkv, int row_stride, const void* kc, const void* vc, const int* block_tables,
    int max_pages, const int* tok_seq, const int* positions, int T, int nh, int nkv, int D,
    int page, float scale, int window, void* out, int nsplit, float* part_o, float* part_ml,
    hipStream_t stream) {
  SL_CHECK(T >= 0 && nh > 0 && nkv > 0 && nh % nkv == 0,
           "attention: heads must be a positive multiple of kv heads");
  SL_CHECK(D > 0 && D <= MAX_D, "attention: head_dim must be in 1..256");
  SL_CHECK(page == 16 || page == 32 || page == 64, "attention: page size must be 16, 32 or 64");
  SL_CHECK(nh <= 65535, "attention: more than 65535 heads");
  SL_CHECK(window >= 0, "attention: window must be >= 0 (0 = none)");
  SL_CHECK(nsplit >= 1 && nsplit <= 64, "attention: 1..64 shares of the keys");
  SL_CHECK(nsplit == 1 || (part_o != nullptr && part_ml != nullptr),
           "attention: shares of the keys need the partial buffers");
  if (T == 0) return nullptr;
  const int g = nh / nkv;
  if (g > 1) {                                       // the heads of a group together
    const int chunks = (g + GROUP_HEADS - 1) / GROUP_HEADS;
    const bool aligned = (((uintptr_t)kc | (uintptr_t)vc) % 16) == 0;
    auto few = [&](auto kernel) {
      kernel<<<dim3(T, nkv * chunks, nsplit), 64, 0, stream>>>((const act_t*)qkv, row_stride, (const act_t*)kc, (const act_t*)vc,
          block_tables, max_pages, tok_seq, positions, nh, nkv, page, scale, window, nsplit, part_o, part_ml);
    };
    // (by the numbers of tokens and shares only, so that a captured step and an eager one add up in the same order)
    const bool alone = nsplit > 1 && aligned && (long long)T * nkv * chunks * nsplit <= 4ll * device_cus();
    if (alone && D == 64) few(attention_few_keys_kernel<64>);
    else if (alone && D == 128) few(attention_few_keys_kernel<128>);
    else attention_general_group_kernel<<<dim3(T, nkv * chunks, nsplit), 64, 0, stream>>>(
        (const act_t*)qkv, row_stride, (const act_t*)kc, (const act_t*)vc, block_tables, max_pages,
        tok_seq, positions, nh, nkv, D, page, scale, window, (act_t*)out, nsplit, part_o, part_ml);
  } else {
    attention_general_kernel<<<dim3(T, nh, nsplit), 64, 0, stream>>>(
        (const act_t*)qkv, row_stride, (const act_t*)kc, (const act_t*)vc, block_tables, max_pages,
        tok_seq, positions, nh, nkv, D, page, scale, window, (act_t*)out, nsplit, part_o, part_ml);
  }
  const char* e = sl_launch_status();
  if (e || nsplit == 1) return e;
  const dim3 grid(T, nh, (D + 63) / 64);
  auto combine = [&](auto kernel) { kernel<<<grid, 64, 0, stream>>>(part_o, part_ml, nsplit, nh, D, (act_t*)out); };
  if (nsplit <= 8) combine(attention_general_combine_kernel<8>);
  else if (nsplit <= 16) combine(attention_general_combine_kernel<16>);
  else if (nsplit <= 32) combine(attention_general_combine_kernel<32>);
  else combine(attention_general_combine_kernel<64>);
  return sl_launch_status();
}
