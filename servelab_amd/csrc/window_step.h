// The matrix-core window attention of a step of one token a sequence; included by window_attention_mfma.hip, whose head says what is
// float and how a score and a weight are formed.
//
// What bounds a decode step is the chain of dependent trips to memory, so it is kept to three: the call's arguments; then the
// token's position, its q and all block table entries that the wavefront may need, side by side; then keys and values.  That is
// possible because the blocks of 32 keys go to the wavefronts in turn by their number in the sequence (block b to wavefront b modulo
// their number), not by the place of the window: a lane asks for the entries of one candidate before the position is known.
#pragma once

// Blocks of a class (b = r, r + R, r + 2 R, ..), nearest keys first, the kept first tokens last; which entries of the block table
// they need.
struct StepBlocks {
  const int* table;
  int max_pages, page_shift, r, R, nA, firstB, have, entries;

  __device__ __forceinline__ int ask(int j0) const {                  // entries of blocks j0 .. j0 + 31 of the class, two a block
    const int lane = threadIdx.x & 63;
    const int at = ((r + R * (j0 + (lane >> 1))) * 32 + ((lane & 1) << 4)) >> page_shift;
    return table[at < max_pages ? at : max_pages - 1];
  }
  __device__ __forceinline__ int settle(int j) const {
    const int b = r + R * j;
    return j >= 0 && b < firstB && b >= nA ? (nA > r ? (nA - 1 - r) / R : -1) : j;
  }
  __device__ __forceinline__ int first(int pos) const { return settle(pos / 32 >= r ? (pos / 32 - r) / R : -1); }
  __device__ __forceinline__ void pages(int j, int& a, int& b) {      // of keys 0 .. 15 and 16 .. 31 of block j
    if (j < have || j >= have + 32) {
      have = j >= 31 ? j - 31 : 0;                                    // (the walk goes down)
      entries = ask(have);
    }
    a = __builtin_amdgcn_readlane(entries, 2 * (j - have));
    b = __builtin_amdgcn_readlane(entries, 2 * (j - have) + 1);
  }
};

// One column's softmax over the blocks it has seen: this lane's 8 keys of a block, from the raw scores s0 (keys 8 gq .. + 3) and s1.
struct StepColumn {
  float scale2, cap2, uncap, slope2, m, l;
  bool capped;
  int pos, lo, keep_first;

  __device__ __forceinline__ StepColumn(const WindowAttention& a, int head, int pos_, int lo_)
      : scale2(a.scale * LOG2E), cap2(a.softcap * LOG2E), uncap(a.softcap > 0.f ? a.scale / a.softcap : 0.f),
        slope2(a.slopes != nullptr ? a.slopes[head] * LOG2E : 0.f), m(-INFINITY), l(0.f), capped(a.softcap > 0.f), pos(pos_), lo(lo_),
        keep_first(a.keep_first) {}

  __device__ __forceinline__ bool sees(int key) const { return (key <= pos) & ((key >= lo) | (key < keep_first)); }
  // weights of the lane's keys; returns what the sums before have to be multiplied by
  __device__ __forceinline__ float weights(f32x4 s0, f32x4 s1, int kbase, int gq, float (&p)[8]) {
    const float bias0 = -slope2 * (float)(pos - kbase - 8 * gq);
    float s[8], top = -INFINITY, factor = scale2;
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = j < 4 ? s0[j] : s1[j - 4];
    if (capped) {
      factor = cap2;
#pragma unroll
      for (int j = 0; j < 8; ++j) s[j] = tanhf(s[j] * uncap);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      s[j] = fmaf(s[j], factor, fmaf(slope2, (float)j, bias0));
      s[j] = sees(kbase + 8 * gq + j) ? s[j] : -INFINITY;
      top = fmaxf(top, s[j]);
    }
    const float mn = fmaxf(m, column_max4(top)), from = mn == -INFINITY ? 0.f : mn;
    float psum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = __builtin_amdgcn_exp2f(s[j] - from);
      psum += p[j];
    }
    const float alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mn);
    l = l * alpha + column_sum4(psum);
    m = mn;
    return alpha;
  }
};

// What a sequence's token sees: keys [0, keep) and [lo, pos].
struct StepKeys {
  int pos, lo, keep;
  __device__ __forceinline__ bool seen(int key) const { return (key <= pos) & ((key >= lo) | (key < keep)); }
  __device__ __forceinline__ int instead(int key, int kbase) const {  // the key, or one of the block that is seen
    key = min(key, pos);
    return key >= lo || key < keep ? key : (lo <= kbase + 31 ? lo : keep - 1);
  }
  __device__ __forceinline__ bool whole(int kbase) const { return kbase + 31 <= pos && (kbase >= lo || kbase + 31 < keep); }
};

// A column's output over all its keys: channels d .. d + 3, from their sums o, the maximum m (units of log 2) and the sum l
__device__ __forceinline__ void finish_column(const WindowAttention& a, int t, int head, int d, f32x4 o, float m, float l) {
  float top = m, extra = 0.f;                                          // (the token sees itself: m is finite)
  if (a.sinks != nullptr) {
    const float sink2 = a.sinks[head] * LOG2E;
    top = fmaxf(m, sink2);
    extra = __builtin_amdgcn_exp2f(sink2 - top);
  }
  const float w = __builtin_amdgcn_exp2f(m - top);
  float f = w / (l * w + extra);
  if (a.gate != nullptr) f *= sigmoidf_(to_f(a.gate[(size_t)t * a.gate_stride + head]));
  if (a.channel_gate != nullptr) {
    struct __attribute__((aligned(4))) gates4 { float v[4]; };
    const gates4 z = *(const gates4*)(a.channel_gate + (size_t)t * a.channel_stride + (size_t)head * DV + d);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] *= sigmoidf_(z.v[e]);
  }
  bf16x4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = (__bf16)(o[e] * f);
  *(bf16x4*)(a.out + ((size_t)t * a.nh + head) * DV + d) = r;
}

// columns are the heads of a kv head, 16 a workgroup; grid (shares, kv heads * tiles of columns, sequences)
constexpr int STEP_WAVES = VK || DV <= 256 ? 4 : 2;
constexpr int STEP_BLOCKS = VK ? 1 : NARROW ? STEP_WAVES : 0;          // classes of blocks a workgroup

#if !SL_VK && SL_NARROW
// Keys and values go from the pages to the operands' registers; a wavefront takes blocks of its own and the four of a workgroup add up
// what they have in LDS, so that a call has a quarter of the shares to merge.
__global__ __launch_bounds__(64 * STEP_WAVES) void window_step_kernel(const WindowAttention a) {
  __shared__ __attribute__((aligned(16))) float os[STEP_WAVES][16][DV + 4];
  __shared__ float2 ml[STEP_WAVES][16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, gq = lane >> 4;
  const int g = a.nh / a.nkv, tiles = (g + 15) / 16, seq = blockIdx.z, share = blockIdx.x;
  const int kvh = __builtin_amdgcn_readfirstlane(blockIdx.y / tiles), c0 = 16 * (blockIdx.y - kvh * tiles);
  const int head = kvh * g + min(c0 + n, g - 1), page = a.page;
  StepBlocks blocks{a.tables + (size_t)seq * a.max_pages, a.max_pages, __builtin_ctz(page), share * STEP_WAVES + wave, a.nsplit * STEP_WAVES,
                    0, 0, 0, 0};
  blocks.entries = blocks.ask(0);
  bf16x8 qf[KK];
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) qf[kk] = *(const bf16x8*)(a.q + (size_t)seq * a.q_stride + (size_t)head * DK + 8 * gq + 32 * kk);
  const int pos = __builtin_amdgcn_readfirstlane(a.positions[seq]), lo = first_key(a, pos);
  const StepKeys keys{pos, lo, min(a.keep_first, lo)};
  blocks.nA = (keys.keep + 31) / 32;
  blocks.firstB = max(lo / 32, blocks.nA);
  StepColumn col(a, head, pos, lo);
  f32x4 o[DD];
#pragma unroll
  for (int dd = 0; dd < DD; ++dd) o[dd] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 k0[KK], k1[KK], v[DD];
  int pgA = 0, pgB = 0;
  auto load_keys = [&](int kbase) {                                    // row i of score tile m: key 8 (i / 4) + 4 m + i % 4
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int key = keys.instead(kbase + 8 * (n / 4) + 4 * m + n % 4, kbase), pg = key < kbase + 16 ? pgA : pgB;
      const __bf16* row = a.kc + (((size_t)pg * a.nkv + kvh) * page + (key & (page - 1))) * DK + 8 * gq;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) (m ? k1 : k0)[kk] = *(const bf16x8*)(row + 32 * kk);
    }
  };
  auto load_values = [&](int kbase) {                                  // a chunk of 8 keys with one that is seen, or of one that is
    const int key0 = kbase + 8 * gq;
    const int key = key0 <= pos && (key0 + 7 >= lo || key0 < keys.keep) ? key0 : keys.instead(key0, kbase) & ~7;
    const int pg = key < kbase + 16 ? pgA : pgB;
    const __bf16* at = a.vc + (((size_t)pg * a.nkv + kvh) * DV + n) * page + (key & (page - 1));
#pragma unroll
    for (int dd = 0; dd < DD; ++dd) v[dd] = *(const bf16x8*)(at + (size_t)(16 * dd) * page);
  };
  int j = blocks.first(pos);
  if (j >= 0) {
    blocks.pages(j, pgA, pgB);
    load_keys((blocks.r + blocks.R * j) * 32);
    load_values((blocks.r + blocks.R * j) * 32);
  }
  while (j >= 0) {
    const int kbase = (blocks.r + blocks.R * j) * 32, after = blocks.settle(j - 1), next = (blocks.r + blocks.R * after) * 32;
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0[kk], qf[kk], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1[kk], qf[kk], s1, 0, 0, 0);
    }
    if (after >= 0) {
      blocks.pages(after, pgA, pgB);
      load_keys(next);
    }
    float p[8];
    const float alpha = col.weights(s0, s1, kbase, gq, p);
    bf16x8 p1, p2, p3;
    three_terms(p, p1, p2, p3);
    if (!keys.whole(kbase)) {                                          // a slot that holds no key the token sees may hold anything
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (!keys.seen(kbase + 8 * gq + e))
#pragma unroll
          for (int dd = 0; dd < DD; ++dd) v[dd][e] = (__bf16)0.f;
    }
#pragma unroll
    for (int dd = 0; dd < DD; ++dd) o[dd] *= alpha;
#pragma unroll
    for (int dd = 0; dd < DD; ++dd) o[dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[dd], p3, o[dd], 0, 0, 0);
#pragma unroll
    for (int dd = 0; dd < DD; ++dd) o[dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[dd], p2, o[dd], 0, 0, 0);
#pragma unroll
    for (int dd = 0; dd < DD; ++dd) o[dd] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[dd], p1, o[dd], 0, 0, 0);
    if (after >= 0) load_values(next);
    j = after;
  }
  // this lane holds channels 16 dd + 4 gq .. + 3 of its column
#pragma unroll
  for (int dd = 0; dd < DD; ++dd) *(f32x4*)&os[wave][n][16 * dd + 4 * gq] = o[dd];
  if (gq == 0) ml[wave][n] = make_float2(col.m, col.l);
  __syncthreads();
  const int columns = min(16, g - c0);
  for (int i = threadIdx.x; i < columns * (DV / 4); i += 64 * STEP_WAVES) {
    const int c = i / (DV / 4), d = 4 * (i % (DV / 4));
    float2 x[STEP_WAVES];
    float top = -INFINITY, sum = 0.f;
#pragma unroll
    for (int w = 0; w < STEP_WAVES; ++w) {
      x[w] = ml[w][c];
      top = fmaxf(top, x[w].x);
    }
    f32x4 all = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < STEP_WAVES; ++w) {
      const float wgt = x[w].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(x[w].x - top);
      all += wgt * *(const f32x4*)&os[w][c][d];
      sum += wgt * x[w].y;
    }
    const int h = kvh * g + c0 + c;
    if (a.nsplit == 1) {
      finish_column(a, seq, h, d, all, top, sum);
    } else {
      const size_t at = ((size_t)seq * a.nh + h) * a.nsplit + share;
      *(f32x4*)(a.part_o + at * DV + d) = all;
      if (d == 0) *(float2*)(a.part_ml + 2 * at) = make_float2(top == -INFINITY ? top : top * (1.f / LOG2E), sum);
    }
  }
}
#elif SL_VK
// Values are channels of the key rows: a block is staged in LDS, as rows and turned, by the whole workgroup, whose wavefronts divide the
// key channels of the scores among them (parts that meet in LDS) and the value channels of the weighted sum.
constexpr int STEP_NT = cdiv((DV / 8) * 4, 256), STEP_NR = RCH ? cdiv(32 * RCH, 256) : 1;      // as NT, NR: for four wavefronts
constexpr int STEP_DD = (DD + 3) / 4, STEP_KK = (KK + 3) / 4;          // channel tiles and key-channel steps a wavefront
__global__ __launch_bounds__(256) void window_step_kernel(const WindowAttention a) {
  extern __shared__ __attribute__((aligned(16))) __bf16 lds16[];
  __bf16* ks = lds16;                                                  // [32][KROW]
  __bf16* vt = ks + 32 * KROW;                                         // channel_row(d) of channel d
  __shared__ f32x4 scores[4][2][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = lane & 15, gq = lane >> 4;
  const int g = a.nh / a.nkv, tiles = (g + 15) / 16, seq = blockIdx.z, share = blockIdx.x;
  const int kvh = __builtin_amdgcn_readfirstlane(blockIdx.y / tiles), c0 = 16 * (blockIdx.y - kvh * tiles);
  const int head = kvh * g + min(c0 + n, g - 1), page = a.page;
  StepBlocks blocks{a.tables + (size_t)seq * a.max_pages, a.max_pages, __builtin_ctz(page), share, a.nsplit, 0, 0, 0, 0};
  blocks.entries = blocks.ask(0);
  bf16x8 qf[STEP_KK];
#pragma unroll
  for (int i = 0; i < STEP_KK; ++i) {
    const int kk = min(wave + 4 * i, KK - 1);
    qf[i] = *(const bf16x8*)(a.q + (size_t)seq * a.q_stride + (size_t)head * DK + 8 * gq + 32 * kk);
  }
  const int pos = __builtin_amdgcn_readfirstlane(a.positions[seq]), lo = first_key(a, pos);
  const StepKeys keys{pos, lo, min(a.keep_first, lo)};
  blocks.nA = (keys.keep + 31) / 32;
  blocks.firstB = max(lo / 32, blocks.nA);
  StepColumn col(a, head, pos, lo);
  f32x4 o[STEP_DD];
#pragma unroll
  for (int i = 0; i < STEP_DD; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 treg[STEP_NT][8], rreg[STEP_NR];
  auto fetch = [&](int j) {
    const int kbase = (blocks.r + blocks.R * j) * 32;
    int pgA, pgB;
    blocks.pages(j, pgA, pgB);
    auto key_row = [&](int kl) {
      const int key = keys.instead(kbase + kl, kbase), pg = key < kbase + 16 ? pgA : pgB;
      return a.kc + (((size_t)pg * a.nkv + kvh) * page + (key & (page - 1))) * DK;
    };
#pragma unroll
    for (int i = 0; i < STEP_NT; ++i) {
      const int idx = min(tid + 256 * i, (DV / 8) * 4 - 1), cb = idx / 4, kg = idx % 4;
#pragma unroll
      for (int e = 0; e < 8; ++e) treg[i][e] = *(const bf16x8*)(key_row(8 * kg + e) + 8 * cb);
    }
    if constexpr (RCH > 0) {
#pragma unroll
      for (int i = 0; i < STEP_NR; ++i) {
        const int idx = min(tid + 256 * i, 32 * RCH - 1);
        rreg[i] = *(const bf16x8*)(key_row(idx / RCH) + 8 * (DV / 8 + idx % RCH));
      }
    }
  };
  int j = blocks.first(pos);
  if (j >= 0) fetch(j);
  while (j >= 0) {
    const int kbase = (blocks.r + blocks.R * j) * 32, after = blocks.settle(j - 1);
    __syncthreads();                                                   // the last block's readers are done
#pragma unroll
    for (int i = 0; i < STEP_NT; ++i) {
      const int idx = tid + 256 * i, cb = idx / 4, kg = idx % 4;
      if (idx < (DV / 8) * 4) {
#pragma unroll
        for (int e = 0; e < 8; ++e) *(bf16x8*)(ks + staged_row(8 * kg + e) * KROW + 8 * cb) = treg[i][e];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          bf16x8 t;
#pragma unroll
          for (int u = 0; u < 8; ++u) t[u] = treg[i][u][e];
          *(bf16x8*)(vt + channel_row(8 * cb + e) + 8 * kg) = t;
        }
      }
    }
    if constexpr (RCH > 0) {
#pragma unroll
      for (int i = 0; i < STEP_NR; ++i) {
        const int idx = tid + 256 * i;
        if (idx < 32 * RCH) *(bf16x8*)(ks + staged_row(idx / RCH) * KROW + 8 * (DV / 8 + idx % RCH)) = rreg[i];
      }
    }
    __syncthreads();
    if (after >= 0) fetch(after);
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
    const __bf16* kp = ks + n * KROW + 8 * gq;
#pragma unroll
    for (int i = 0; i < STEP_KK; ++i) {
      const int kk = wave + 4 * i;
      if (kk >= KK) break;
      s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(kp + 32 * kk), qf[i], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8*)(kp + 16 * KROW + 32 * kk), qf[i], s1, 0, 0, 0);
    }
    scores[wave][0][lane] = s0;
    scores[wave][1][lane] = s1;
    __syncthreads();
    s0 = (scores[0][0][lane] + scores[1][0][lane]) + (scores[2][0][lane] + scores[3][0][lane]);
    s1 = (scores[0][1][lane] + scores[1][1][lane]) + (scores[2][1][lane] + scores[3][1][lane]);
    float p[8];
    const float alpha = col.weights(s0, s1, kbase, gq, p);
    bf16x8 p1, p2, p3, v[STEP_DD];
    three_terms(p, p1, p2, p3);
#pragma unroll
    for (int i = 0; i < STEP_DD; ++i) {
      v[i] = *(const bf16x8*)(vt + channel_row(16 * min(wave * STEP_DD + i, DD - 1) + n) + 8 * gq);
      o[i] *= alpha;
    }
#pragma unroll
    for (int i = 0; i < STEP_DD; ++i) o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[i], p3, o[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < STEP_DD; ++i) o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[i], p2, o[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < STEP_DD; ++i) o[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[i], p1, o[i], 0, 0, 0);
    j = after;
  }
  if (c0 + n >= g) return;
  const size_t at = ((size_t)seq * a.nh + head) * a.nsplit + share;
#pragma unroll
  for (int i = 0; i < STEP_DD; ++i) {
    const int dd = wave * STEP_DD + i;
    if (dd >= DD) break;
    if (a.nsplit == 1) finish_column(a, seq, head, 16 * dd + 4 * gq, o[i], col.m, col.l);
    else *(f32x4*)(a.part_o + at * DV + 16 * dd + 4 * gq) = o[i];
  }
  if (a.nsplit > 1 && wave == 0 && gq == 0)
    *(float2*)(a.part_ml + 2 * at) = make_float2(col.m == -INFINITY ? col.m : col.m * (1.f / LOG2E), col.l);
}
#endif
