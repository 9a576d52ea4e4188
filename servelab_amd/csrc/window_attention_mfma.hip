// The window attention of window_attention.hip on the matrix cores, bfloat16 only, for key widths
// SL_DK (a multiple of 32) and value widths SL_DV (a multiple of 16) fixed at compile time;
// SL_VK = 1: values are the first SL_DV channels of the key rows.  Same call, same meaning.
//
// What is float stays float.  The scores are products of bfloat16 numbers added up in float by
// the matrix instruction (every product is exact in float); scale, cap, distance bias, mask, the
// running maximum and sum and the exponentials are float vector code.  A weight p is not rounded
// to bfloat16 for the second product: it is cut into three bfloat16 terms p = p1 + p2 + p3 (each
// the upper 16 bits of what the terms before left over, 8 bits of significand a term), which
// together are the float exactly, and the weighted sum of the values is three matrix
// instructions, one per term, on float accumulators.
//
// Work layout of prompts (steps of single tokens: window_step.h).  A column is a (token, query head) pair of one sequence and one kv
// head; a wavefront owns 16 columns, a workgroup 64 consecutive ones, and walks the blocks of 32 keys any of them sees.  A block is
// staged in LDS once for the wavefronts that compute on it: the key rows [32][SL_DK], and the values channel-major [SL_DV][32] (copied
// from the value pages, which are channel-major already, or turned in registers, 8 keys x 8 channels a thread, on their way
// from the key rows); the next block is on its way from the pages to registers while a block is
// computed.  Per block and wavefront:
//   S^T[key, column] = K[key, :] . Q[column, :]          mfma 16x16x32, A = K rows, B = Q (registers)
//   O^T[d, column] += V^T[d, key] P^T[key, column]       mfma 16x16x32, A = V^T rows, B = the terms of P
// Row i of score tile m is key 8 (i / 4) + 4 m + i % 4 of the block, so that a lane ends up with
// the weights of 8 consecutive keys of its column: the B operand of the second product as it is.
//
// What bounds it: a block is a chain (stage, scores, maximum, exponentials, terms, sums) of a few thousand cycles, of which the matrix
// instructions are 500 to 2,100, and the longest tile walks all of its keys; so where the chip has few workgroups one is eight wavefronts: two teams that take every
// other block and meet at the end, or, of a wide latent (132 matrix instructions a block, more registers than two
// wavefronts a SIMD have), pairs that share columns, each with half the channels; the longest tiles start first; a
// block has 150 vector instructions and no branches inside (addresses looked up key by key and a cap chosen score by score were 270 and
// eight).  us, before / now: 128 / 128, 16 heads on 2, one prompt of 2,048 tokens 104 / 68 (255 TFLOP/s counted once a weight), 1,000 and 889 56 /
// 38, 1,500 with a window of 1,024 64 / 40; 576 / 512, 16 heads, 1,000 and 889 150 / 137, 2,048 282 / 248.  Tried: blocks of 64
// keys (a tenth slower at 128, half as slow again at 576), two blocks on their way (registers spill; no gain at 576).
#include "window_attention.h"

#if defined(SL_F32)
#error "window_attention_mfma is a bfloat16 kernel; the float32 path uses window_attention.hip"
#endif
#if !defined(SL_DK) || !defined(SL_DV) || !defined(SL_VK)
#error "SL_DK, SL_DV and SL_VK must be defined"
#endif
#if SL_DK % 32 != 0 || SL_DV % 16 != 0 || SL_DK < 32 || SL_DV < 16 || SL_DV > 512 || SL_DK > 1024
#error "SL_DK must be a multiple of 32 up to 1024, SL_DV a multiple of 16 up to 512"
#endif
#if SL_VK && SL_DV > SL_DK
#error "values read from key rows cannot be wider than a key"
#endif

// Values with pages of their own: two teams, and the kernel of window_step.h for steps, hold keys, values and sums of up to this
// width in registers.  Wider ones spill there (512 / 512: 158 and 126 registers), and some do not fit two staged blocks in a CU: they take
// one team, whose wavefronts have twice the registers, and their steps the same kernel with the keys cut into shares.  us, two teams and step
// kernel / one team and shares, 16 heads on 2: a prompt of 1,024, and steps of 8 requests at 1,500: 128 / 128 33 / 48 and 7.6 / 10.1, 512 / 256 64 / 85
// and 13.3 / 16.5, 704 / 256 88 / 101 and 14.8 / 20.0; beyond the line 512 / 512 197 / 119 and 35.6 / 22.4, 384 / 512 123 / 111 and 29.8 /
// 21.1, 1024 / 112 105 / 102 and 15.7 / 20.6.
#define SL_NARROW (SL_DK + 2 * SL_DV <= 1216)

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int DK = SL_DK, DV = SL_DV;
constexpr bool VK = SL_VK != 0, NARROW = SL_NARROW;
constexpr int KK = DK / 32, DD = DV / 16;
constexpr int KROW = DK + 8;          // elements of a staged key row (the pad spreads rows over the banks)
constexpr int VROW = 40;              // elements of a staged channel row: 32 keys and a pad
constexpr int VPAD = VK ? 32 : 0;     // and more behind every eight of them, where a thread turns eight: neighbouring threads' rows in other banks
constexpr int VT = DV * VROW + DV / 8 * VPAD;
__device__ __forceinline__ int channel_row(int d) { return d * VROW + (d >> 3) * VPAD; }
// Key 8 a + 4 m + b of a block is staged as row 16 m + 4 a + b: the rows of a score tile side by side, which take every bank once.
__device__ __forceinline__ int staged_row(int key) { return 16 * ((key >> 2) & 1) + 4 * (key >> 3) + (key & 3); }
constexpr float LOG2E = 1.4426950408889634f;

// Maximum / sum over the four lanes n, n + 16, n + 32, n + 48 that share a column, by the row-swap
// instructions of gfx950 (register to register): after a swap of x with itself one result holds
// the lower partner and the other the upper one, in every lane.
__device__ __forceinline__ float column_max4(float x) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float column_sum4(float x) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// p = p1 + p2 + p3 exactly: each term is the upper 16 bits (a bfloat16) of what the terms before left over, 8 bits of significand a
// term; two terms of neighbouring keys share a register.
__device__ __forceinline__ void three_terms(const float (&p)[8], bf16x8& p1, bf16x8& p2, bf16x8& p3) {
  u32x4 w1, w2, w3;
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    unsigned t1[2], t2[2], t3[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float x = p[j + e];
      t1[e] = __float_as_uint(x) & 0xffff0000u;
      const float r1 = x - __uint_as_float(t1[e]);
      t2[e] = __float_as_uint(r1) & 0xffff0000u;
      t3[e] = __float_as_uint(r1 - __uint_as_float(t2[e]));
    }
    w1[j / 2] = __builtin_amdgcn_perm(t1[1], t1[0], 0x07060302u);
    w2[j / 2] = __builtin_amdgcn_perm(t2[1], t2[0], 0x07060302u);
    w3[j / 2] = __builtin_amdgcn_perm(t3[1], t3[0], 0x07060302u);
  }
  p1 = __builtin_bit_cast(bf16x8, w1);
  p2 = __builtin_bit_cast(bf16x8, w2);
  p3 = __builtin_bit_cast(bf16x8, w3);
}

constexpr int cdiv(int a, int b) { return (a + b - 1) / b; }
constexpr int COLS = 64;                               // of a workgroup
constexpr int STAGE = 32 * KROW + VT;                  // values of a staged block
constexpr int KCH = DK / 8, RCH = VK ? (DK - DV) / 8 : 0;      // chunks of 8 values (16 bytes) of a key row, and of one behind the values

// A prompt's workgroup owns 64 columns, sixteen for each of four wavefronts; TEAMS 2: twice as many, in two teams that take every other block
// and meet at the end; PARTS 2: twice as many, two of them for sixteen columns, each with half of the channels (of a latent).
template <int TEAMS, int PARTS> struct Form {
  static constexpr int THREADS = 256 * PARTS;          // of a team
  static constexpr int KKP = cdiv(KK, PARTS), DDP = cdiv(DD, PARTS);      // steps of key channels and tiles of value channels a wavefront
  static constexpr int MEETS = PARTS == 2 ? 8 * 2 * 64 * 16 : 0;          // bytes in which the parts of the scores meet
  static constexpr int MEET = TEAMS == 2 ? 256 * DV + 512 : 0;            // bytes in which the second team hands over what it has
  static constexpr int STAGED = 2 * TEAMS * STAGE + MEETS, LDS_BYTES = STAGED > MEET ? STAGED : MEET;
  static_assert(LDS_BYTES <= 160 * 1024, "a prompt's workgroup fits a CU");
  // what a thread stages of a block
  static constexpr int NKC = VK ? 1 : cdiv(32 * KCH, THREADS);            // chunks of keys
  static constexpr int NVC = VK ? 1 : cdiv(DV * 4, THREADS);              // chunks of values (a channel's 8 keys)
  static constexpr int NT = VK ? cdiv((DV / 8) * 4, THREADS) : 1;         // 8 keys x 8 channels tiles (turned on their way into LDS)
  static constexpr int NR = RCH ? cdiv(32 * RCH, THREADS) : 1;
  // A thread's places in a block are the same for all blocks and stay in registers, except where these are short; us, kept / worked out
  // anew: 512 / 256 64 / 69 (no register spilled either way), 896 / 64 145 (50 spilled) / 80; one team: 512 / 512 119 / 135 (none), 640 / 512 146 (13) /
  // 145 and steps of 32 requests 41 / 37, 1024 / 512 241 (76) / 200.
  static constexpr bool PLACES_ANEW = !VK && (TEAMS == 2 ? 4 * DK + 5 * DV > 3328 : DK + 2 * DV > 1600);
  static constexpr int WAVES = TEAMS * PARTS == 1 ? (DK <= 128 && DV <= 128 ? (VK && DK + DV > 192 ? 3 : 4) : DK + DV <= 576 ? 2 : 1)
                                                  : (!VK && DK <= 128 && DV <= 128 ? 4 : 2);      // a SIMD holds, at least
};

// Prompts' forms that are built.  FEW: of few workgroups each wants to be short, and has eight wavefronts: two teams, or pairs where the latent is so
// wide that two teams spill or do not fit.  MANY: of many workgroups the chip wants as many as it can hold at once, four wavefronts each and no
// meeting; only where those leave room for two on a SIMD (576 / 512: pairs 12 % ahead at every number of workgroups, 256 / 256 64 / 85).
constexpr bool PAIRS = VK && DK + DV > 576;
constexpr int FEW_TEAMS = !PAIRS && (VK || NARROW) ? 2 : 1, FEW_PARTS = PAIRS ? 2 : 1;
constexpr bool MANY = FEW_TEAMS == 2 && DK + DV <= 576;

// Workgroups start in the order of their number, and numbers go to the eight dies in turn and there to the groups of CUs in
// turn.  Without a window or chunks a tile takes as long as its keys are many, so the late tiles come first:
// BY_LENGTH, for sequences of one length: of every sequence and head, so that the short ones fill what is left at the end;
// BY_LENGTH_MOVED, for nearly equal ones: the same, and a sequence and head moves on by one place from tile to tile;
// LATE_FIRST, for unequal ones: sequence by sequence.  (Among short sequences every 32nd workgroup, say, is one of the long
// prompt's, and with BY_LENGTH all of these are one die's: a prompt of 500 tokens among 31 decoding, 16 heads on 1, 576 / 512:
// 720 us, 127 in this order; prompts of 1,200, 300, 100 and 20 tokens 413 us, 467 moved, 195; of 1,200 and three of
// 1,000 410 moved, 463 with early tiles first.)
enum { LATE_FIRST, BY_LENGTH, BY_LENGTH_MOVED };

template <int TEAMS, int PARTS>
__global__ __launch_bounds__(256 * TEAMS * PARTS, (Form<TEAMS, PARTS>::WAVES)) void window_attention_mfma_kernel(const WindowAttention a, int order) {
  using F = Form<TEAMS, PARTS>;
  constexpr int THREADS = F::THREADS, KKP = F::KKP, DDP = F::DDP, NKC = F::NKC, NVC = F::NVC, NT = F::NT, NR = F::NR;
  extern __shared__ __attribute__((aligned(16))) __bf16 lds16[];
  const int team = TEAMS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / THREADS);
  __bf16* ks = lds16 + team * STAGE;                   // [32][KROW]
  __bf16* vt = ks + 32 * KROW;                         // channel_row(d) of channel d
  f32x4 (*meets)[64] = (f32x4(*)[64])(lds16 + STAGE);  // [2 parts][4 wavefronts][2 tiles of keys]
  const int tid = threadIdx.x % THREADS, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3, n = lane & 15, gq = lane >> 4;
  const int part = PARTS == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 8);
  const int page = a.page, nkv = a.nkv;
  int seq = blockIdx.z, kvh = blockIdx.y, item = gridDim.x - 1 - blockIdx.x;
  if (order == BY_LENGTH) {                     // (launched with the heads along x and the tiles along z)
    seq = blockIdx.y;
    kvh = blockIdx.x;
    item = gridDim.z - 1 - blockIdx.z;
  } else if (order == BY_LENGTH_MOVED) {
    // (read back from a lane: a division is done in vector registers, and so would be all that follows from it)
    const int number = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), pairs = gridDim.y * gridDim.z;
    const int rank = __builtin_amdgcn_readfirstlane(number / pairs), moved = pairs < 8 ? rank * pairs / 8 : rank;
    const int pair = __builtin_amdgcn_readfirstlane((number % pairs + moved) % pairs);
    seq = __builtin_amdgcn_readfirstlane(pair / gridDim.y);
    kvh = pair - seq * gridDim.y;
    item = gridDim.x - 1 - rank;
  }
  const int g = a.nh / nkv;
  const int q0 = a.cu_q[seq], qlen = a.cu_q[seq + 1] - q0;
  const int ncols = qlen * g;
  const int tile = __builtin_amdgcn_readfirstlane(item / a.nsplit), share = item - tile * a.nsplit;
  const int c0 = tile * COLS;
  if (c0 >= ncols) return;
  const int pos0 = a.positions[q0];
  const int* table = a.tables + (size_t)seq * a.max_pages;

  // the keys any column of the workgroup sees: [0, keep) and [kmin, kmax], as blocks of 32
  const int tok_first = c0 / g;
  const int c_last = c0 + COLS - 1 < ncols - 1 ? c0 + COLS - 1 : ncols - 1;
  const int kmax = pos0 + c_last / g;
  const int kmin = first_key(a, pos0 + tok_first);
  const int keep = a.keep_first < kmin ? a.keep_first : kmin;
  const int nA = keep > 0 ? (keep - 1) / 32 + 1 : 0;
  int firstB = kmin / 32;
  if (firstB < nA) firstB = nA;
  const int nB = kmax / 32 - firstB + 1 > 0 ? kmax / 32 - firstB + 1 : 0;
  const int nblk = nA + nB;
  const int from_block = (int)((long long)nblk * share / a.nsplit), i0 = from_block + team;
  const int i1 = (int)((long long)nblk * (share + 1) / a.nsplit);
  // The blocks are walked from the nearest keys to the farthest (the kept first tokens last): a distance
  // bias makes nearer keys score higher, so the running maximum settles in the first block or two and
  // the sums are rarely rescaled; without a bias the order does not matter.
  auto block_base = [&](int i) {
    const int b = nblk - 1 - i;
    return (b < nA ? b : firstB + (b - nA)) * 32;
  };
  auto loadable = [&](int key) { return (key <= kmax) & ((key >= kmin) | (key < keep)); };

  // this wavefront's columns, and this lane's (a column past the last is computed like the last, never stored)
  const int cw0 = c0 + 16 * wave;
  const bool wave_live = cw0 < ncols;
  const int cw1 = cw0 + 15 < ncols - 1 ? cw0 + 15 : ncols - 1;
  int c = cw0 + n;
  const bool live = c < ncols;
  if (!live) c = ncols - 1;
  const int tok = c / g, head = kvh * g + c % g;
  const int pos_c = pos0 + tok;
  const int lo_c = first_key(a, pos_c);
  // every column of the wavefront sees all of a block [kb, kb + 31] when kb + 31 <= pos_lo and (kb >= lo_hi
  // or the block lies within the kept first tokens)
  const int pos_lo = pos0 + (wave_live ? cw0 : 0) / g, pos_hi = pos0 + (wave_live ? cw1 : 0) / g;
  const int lo_hi = first_key(a, pos_hi);
  const float scale2 = a.scale * LOG2E;
  const bool capped = a.softcap > 0.f;
  const float cap2 = a.softcap * LOG2E, uncap = capped ? a.scale / a.softcap : 0.f;
  const float slope2 = a.slopes != nullptr ? a.slopes[head] * LOG2E : 0.f;
  bf16x8 qf[KKP];
  {
    const __bf16* qp = a.q + (size_t)(q0 + tok) * a.q_stride + (size_t)head * DK + 8 * gq;
#pragma unroll
    for (int kk = 0; kk < KKP; ++kk) qf[kk] = *(const bf16x8*)(qp + 32 * min(part * KKP + kk, KK - 1));
  }
  f32x4 o[DDP];
#pragma unroll
  for (int dd = 0; dd < DDP; ++dd) o[dd] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;                        // the maximum in units of log 2
  const __bf16 zero = (__bf16)0.f;

  // A block travels pages -> registers -> LDS; the registers are filled for block i + 1 while block i
  // is computed from LDS.
  // The pages of a block (of its keys 0..15 and 16..31) are asked for one block earlier still, so
  // that a block costs one trip to memory and not two in a row; by a vector load (an even lane
  // asks for the first, an odd lane for the second) so that the wait for it is not the wait for LDS.
  const int page_shift = __builtin_ctz(page);
  auto ask_pages = [&](int kbase) {
    const int key = kbase + ((lane & 1) << 4);
    return table[(key <= kmax ? key : kbase) >> page_shift];
  };
  // A half of a block (16 keys, of one page) is read where it lies: a place for both halves, which is the same for all threads, and a
  // thread's own places beside it, which are the same for all blocks.  (Clamped and looked up key by key the addresses were 100 of
  // a block's 270 vector instructions.)  A half of which no column sees a key may have no page: the other half stands for it.  What
  // lies in slots no column sees gets no weight, and values there become zeros.  No load stands behind a condition: the
  // compiler waits for a load where the two ways meet.
  bf16x8 kreg[NKC], vreg[NVC], treg[NT][8], rreg[NR];
  auto this_thread = [&]() {
    int x = tid;
    if (F::PLACES_ANEW) asm volatile("" : "+v"(x));       // (nothing that follows from it is kept from block to block)
    return x;
  };
  auto fetch = [&](int kbase, int asked) {
    const int tid = this_thread();
    const int pgA = __builtin_amdgcn_readlane(asked, 0), pgB = __builtin_amdgcn_readlane(asked, 1);
    const bool seenA = kbase + 15 >= kmin || kbase < keep, seenB = kbase + 16 <= kmax && (kbase + 31 >= kmin || kbase + 16 < keep);
    const size_t headA = (size_t)(seenA ? pgA : pgB) * nkv + kvh, headB = (size_t)(seenB ? pgB : pgA) * nkv + kvh;
    const int inA = (seenA ? kbase : kbase + 16) & (page - 1), inB = (seenB ? kbase + 16 : kbase) & (page - 1);
    const __bf16 *keysA = a.kc + (headA * page + inA) * DK, *keysB = a.kc + (headB * page + inB) * DK;
    if constexpr (!VK) {
#pragma unroll
      for (int i = 0; i < NKC; ++i) {
        const int idx = min(tid + THREADS * i, 32 * KCH - 1), kl = idx / KCH;
        const bool second = 16 * KCH % THREADS == 0 ? THREADS * i >= 16 * KCH : kl >= 16;
        kreg[i] = *(const bf16x8*)((second ? keysB : keysA) + (kl & 15) * DK + 8 * (idx % KCH));
      }
      const __bf16 *valuesA = a.vc + headA * DV * page + inA, *valuesB = a.vc + headB * DV * page + inB;
#pragma unroll
      for (int i = 0; i < NVC; ++i) {
        const int idx = min(tid + THREADS * i, DV * 4 - 1);
        vreg[i] = *(const bf16x8*)((idx & 2 ? valuesB : valuesA) + (idx / 4) * page + 8 * (idx & 1));
      }
    } else {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int idx = min(tid + THREADS * i, (DV / 8) * 4 - 1), cb = idx / 4, kg = idx % 4;
        const __bf16* at = (kg & 2 ? keysB : keysA) + 8 * (kg & 1) * DK + 8 * cb;
#pragma unroll
        for (int j = 0; j < 8; ++j) treg[i][j] = *(const bf16x8*)(at + j * DK);
      }
      if constexpr (RCH > 0) {
#pragma unroll
        for (int i = 0; i < NR; ++i) {
          const int idx = min((PARTS == 2 ? tid ^ 256 : tid) + THREADS * i, 32 * RCH - 1), kl = idx / RCH, c8 = DV / 8 + idx % RCH;
          rreg[i] = *(const bf16x8*)((kl >= 16 ? keysB : keysA) + (kl & 15) * DK + 8 * c8);
        }
      }
    }
  };
  auto store = [&](int kbase) {
    const int tid = this_thread();
    const bool all_seen = kbase + 31 <= kmax && (kbase >= kmin || kbase + 31 < keep);
    if constexpr (!VK) {
#pragma unroll
      for (int i = 0; i < NKC; ++i) {
        const int idx = tid + THREADS * i, kl = idx / KCH, c8 = idx % KCH;
        if (32 * KCH % THREADS == 0 || idx < 32 * KCH) *(bf16x8*)(ks + staged_row(kl) * KROW + 8 * c8) = kreg[i];
      }
#pragma unroll
      for (int i = 0; i < NVC; ++i) {
        const int idx = tid + THREADS * i, d = idx / 4, k8 = idx % 4;
        bf16x8 v = vreg[i];
        if (!all_seen) {                               // a slot of the page that holds no visible key may hold anything
#pragma unroll
          for (int e = 0; e < 8; ++e)
            v[e] = loadable(kbase + 8 * k8 + e) ? v[e] : zero;
        }
        if (DV * 4 % THREADS == 0 || idx < DV * 4) *(bf16x8*)(vt + channel_row(d) + 8 * k8) = v;
      }
    } else {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int idx = tid + THREADS * i, cb = idx / 4, kg = idx % 4;
        if (DV / 2 % THREADS == 0 || idx < (DV / 8) * 4) {
          if (!all_seen) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (!loadable(kbase + 8 * kg + j)) treg[i][j] = bf16x8{zero, zero, zero, zero, zero, zero, zero, zero};
          }
#pragma unroll
          for (int j = 0; j < 8; ++j) *(bf16x8*)(ks + staged_row(8 * kg + j) * KROW + 8 * cb) = treg[i][j];
#pragma unroll
          for (int e = 0; e < 8; ++e) {                // channel 8 cb + e of the tile's 8 keys
            bf16x8 t;
#pragma unroll
            for (int j = 0; j < 8; ++j) t[j] = treg[i][j][e];
            *(bf16x8*)(vt + channel_row(8 * cb + e) + 8 * kg) = t;
          }
        }
      }
      if constexpr (RCH > 0) {
#pragma unroll
        for (int i = 0; i < NR; ++i) {
          const int idx = (PARTS == 2 ? tid ^ 256 : tid) + THREADS * i, kl = idx / RCH, c8 = DV / 8 + idx % RCH;
          if (32 * RCH % THREADS == 0 || idx < 32 * RCH) *(bf16x8*)(ks + staged_row(kl) * KROW + 8 * c8) = rreg[i];
        }
      }
    }
  };

  int asked = 0;
  if (i0 < i1) {
    fetch(block_base(i0), ask_pages(block_base(i0)));
    if (i0 + TEAMS < i1) asked = ask_pages(block_base(i0 + TEAMS));
  }
  // (q, asked for before the first keys, is waited for here: left to the loop, the wait for its first use would be one for the
  // next block's keys as well)
#pragma unroll
  for (int kk = 0; kk < KKP; ++kk) asm volatile("" : "+v"(qf[kk]));
  for (int i = i0; i - team < i1; i += TEAMS) {        // (as many rounds for both teams; the second may have no block in the last)
    const int kbase = block_base(i);
    __syncthreads();                                   // the last block's readers are done
    if (i < i1) store(kbase);
    __syncthreads();
    if (i + TEAMS < i1) {
      fetch(block_base(i + TEAMS), asked);
      if (i + 2 * TEAMS < i1) asked = ask_pages(block_base(i + 2 * TEAMS));
    }
    if (PARTS == 1 && (!wave_live || i >= i1)) continue;             // (a wavefront without columns only helps staging)

    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
    const __bf16* kp = ks + n * KROW + 8 * gq;
#pragma unroll
    for (int kk = 0; kk < KKP; ++kk) {
      if (KK % PARTS != 0 && part * KKP + kk >= KK) continue;
      const bf16x8 k0 = *(const bf16x8*)(kp + 32 * (part * KKP + kk));
      const bf16x8 k1 = *(const bf16x8*)(kp + 16 * KROW + 32 * (part * KKP + kk));
      s0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, qf[kk], s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, qf[kk], s1, 0, 0, 0);
    }
    if constexpr (PARTS == 2) {
      meets[(part * 4 + wave) * 2][lane] = s0;
      meets[(part * 4 + wave) * 2 + 1][lane] = s1;
      __syncthreads();
      if (!wave_live) continue;
      s0 = meets[2 * wave][lane] + meets[8 + 2 * wave][lane];
      s1 = meets[2 * wave + 1][lane] + meets[8 + 2 * wave + 1][lane];
    }
    // score of key kbase + 8 gq + j: raw * scale - slope * (pos_c - key), in units of log 2
    const float bias0 = -slope2 * (float)(pos_c - kbase - 8 * gq);
    // (a cap takes its own pass: chosen score by score it is eight branches a block, which nothing is scheduled across)
    float s[8], top = -INFINITY, factor = scale2;
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = j < 4 ? s0[j] : s1[j - 4];
    if (capped) {
      factor = cap2;
#pragma unroll 1
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float t = tanhf((h ? s[4 + j] : s[j]) * uncap);
          if (h) s[4 + j] = t;
          else s[j] = t;
        }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = fmaf(s[j], factor, fmaf(slope2, (float)j, bias0));
    const bool whole = kbase + 31 <= pos_lo && (kbase >= lo_hi || kbase + 31 < a.keep_first);
    if (!whole) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int key = kbase + 8 * gq + j;
        const bool seen = (key <= pos_c) & ((key >= lo_c) | (key < a.keep_first));      // (no branches)
        s[j] = seen ? s[j] : -INFINITY;
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) top = fmaxf(top, s[j]);
    const float mn = fmaxf(m, column_max4(top));
    const float from = mn == -INFINITY ? 0.f : mn;     // (only while no key was seen: exp2(-inf) = 0)
    float p[8], psum = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      p[j] = __builtin_amdgcn_exp2f(s[j] - from);
      psum += p[j];
    }
    if (__any(mn > m)) {                               // the maximum of some column moved: rescale
      const float alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mn);
      l *= alpha;
#pragma unroll
      for (int dd = 0; dd < DDP; ++dd) o[dd] *= alpha;
      m = mn;
    }
    l += column_sum4(psum);
    bf16x8 p1, p2, p3;
    three_terms(p, p1, p2, p3);
    // (four tiles of channels side by side: the three products of one depend on each other)
    constexpr int SIDE = DDP % 4 == 0 && DD % PARTS == 0 ? 4 : 1;
#pragma unroll
    for (int dd = 0; dd < DDP; dd += SIDE) {
      if (DD % PARTS != 0 && part * DDP + dd >= DD) continue;
      bf16x8 vf[SIDE];
#pragma unroll
      for (int u = 0; u < SIDE; ++u) vf[u] = *(const bf16x8*)(vt + channel_row(16 * (part * DDP + dd + u) + n) + 8 * gq);
#pragma unroll
      for (int u = 0; u < SIDE; ++u) o[dd + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[u], p3, o[dd + u], 0, 0, 0);
#pragma unroll
      for (int u = 0; u < SIDE; ++u) o[dd + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[u], p2, o[dd + u], 0, 0, 0);
#pragma unroll
      for (int u = 0; u < SIDE; ++u) o[dd + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[u], p1, o[dd + u], 0, 0, 0);
    }
  }
  if constexpr (TEAMS == 2) {                          // the first team takes what the second has of its columns
    f32x4* os = (f32x4*)lds16;
    float2* ml = (float2*)(os + THREADS * DD);
    __syncthreads();
    if (team == 1) {
#pragma unroll
      for (int dd = 0; dd < DD; ++dd) os[THREADS * dd + tid] = o[dd];
      if (gq == 0) ml[16 * wave + n] = make_float2(m, l);
    }
    __syncthreads();
    if (team == 1) return;
    const float2 other = ml[16 * wave + n];
    const float both = fmaxf(m, other.x), ours = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - both),
                theirs = other.x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(other.x - both);
#pragma unroll
    for (int dd = 0; dd < DD; ++dd) o[dd] = o[dd] * ours + os[THREADS * dd + tid] * theirs;
    l = l * ours + other.y * theirs;
    m = both;
  }
  if (!live) return;
  // this lane holds channels 16 dd + 4 gq .. + 3 of its column
  const size_t row = (size_t)(q0 + tok) * a.nh + head;
  if (a.nsplit > 1) {
    float* po = a.part_o + (row * a.nsplit + share) * DV + 16 * part * DDP + 4 * gq;
#pragma unroll
    for (int dd = 0; dd < DDP; ++dd)
      if (DD % PARTS == 0 || part * DDP + dd < DD) *(f32x4*)(po + 16 * dd) = o[dd];
    if (gq == 0 && part == 0) {
      a.part_ml[(row * a.nsplit + share) * 2] = m == -INFINITY ? m : m * (1.f / LOG2E);
      a.part_ml[(row * a.nsplit + share) * 2 + 1] = l;
    }
    return;
  }
  // every query sees itself, so m is finite here
  float top = m, extra = 0.f;
  if (a.sinks != nullptr) {
    const float sink2 = a.sinks[head] * LOG2E;
    top = fmaxf(m, sink2);
    extra = __builtin_amdgcn_exp2f(sink2 - top);
  }
  const float w = __builtin_amdgcn_exp2f(m - top);
  float f = w / (l * w + extra);
  if (a.gate != nullptr) f *= sigmoidf_(to_f(a.gate[(size_t)(q0 + tok) * a.gate_stride + head]));
  __bf16* op = a.out + row * DV + 16 * part * DDP + 4 * gq;
  const float* cg = a.channel_gate != nullptr
      ? a.channel_gate + (size_t)(q0 + tok) * a.channel_stride + (size_t)head * DV + 16 * part * DDP + 4 * gq : nullptr;
#pragma unroll
  for (int dd = 0; dd < DDP; ++dd) {
    if (DD % PARTS != 0 && part * DDP + dd >= DD) continue;
    bf16x4 r;
    if (cg != nullptr) {
      struct __attribute__((aligned(4))) gates4 { float v[4]; };      // (one load, whatever the rows' alignment)
      const gates4 z = *(const gates4*)(cg + 16 * dd);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[dd][e] *= sigmoidf_(z.v[e]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = (__bf16)(o[dd][e] * f);
    *(bf16x4*)(op + 16 * dd) = r;
  }
}

#include "window_step.h"

template <int TEAMS, int PARTS> static const char* launch_mfma(const WindowAttention& a, dim3 grid, int order, hipStream_t stream) {
  constexpr int bytes = Form<TEAMS, PARTS>::LDS_BYTES;
  if (bytes > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)window_attention_mfma_kernel<TEAMS, PARTS>, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return hipGetErrorString(e);
  }
  window_attention_mfma_kernel<TEAMS, PARTS><<<grid, 256 * TEAMS * PARTS, bytes, stream>>>(a, order);
  return sl_launch_status();
}
#if SL_VK || SL_NARROW
static const char* launch_step(const WindowAttention& a, int num_seqs, hipStream_t stream) {
  const size_t bytes = VK ? sizeof(__bf16) * ((size_t)32 * KROW + (size_t)VT) : 0;
  if (bytes > 48 * 1024) {
    hipError_t e = hipFuncSetAttribute((const void*)window_step_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if (e != hipSuccess) return hipGetErrorString(e);
  }
  window_step_kernel<<<dim3(a.nsplit, a.nkv * ((a.nh / a.nkv + 15) / 16), num_seqs), 64 * STEP_WAVES, bytes, stream>>>(a);
  return sl_launch_status();
}
#else
static const char* launch_step(const WindowAttention&, int, hipStream_t) { return "window attention: no kernel for steps of this width"; }
#endif

// Blocks of 32 keys that a workgroup of a step of single tokens takes side by side; 0: such steps take the kernel of prompts, cut into shares.
extern "C" int sl_window_attention_mfma_step_blocks() { return STEP_BLOCKS; }

// The call of sl_window_attention, for Dk == SL_DK, Dv == SL_DV and (vc == nullptr) == SL_VK.
// q rows, key rows and value rows must be 16-byte aligned.  few: the form of few workgroups; step: a step of one token a sequence by
// the kernel for it (either is a wish: what is not built, or does not fit the call, is the other).
extern "C" const char* sl_window_attention_mfma(
    const void* q, int q_stride, const void* kc, const void* vc, const int* tables, int max_pages,
    const int* cu_q, const int* positions, int num_seqs, int max_q_len, int num_tokens, int nh,
    int nkv, int Dk, int Dv, int page, float scale, float softcap, int window, int chunk, int keep_first, const float* slopes,
    const float* sinks, const void* gate, int gate_stride, const float* channel_gate, int channel_stride, void* out,
    int few, int step, int nsplit, float* part_o, float* part_ml, hipStream_t stream) {
  SL_CHECK(Dk == DK && Dv == DV && (vc == nullptr) == VK, "window attention (matrix cores): built for other widths");
  SL_CHECK(num_seqs >= 0 && max_q_len >= 1 && nh > 0 && nkv > 0 && nh % nkv == 0,
           "window attention: heads must be a positive multiple of kv heads");
  SL_CHECK(page == 16 || page == 32 || page == 64, "window attention: page size must be 16, 32 or 64");
  SL_CHECK(nkv <= 65535 && num_seqs <= 65535, "window attention: grid too large");
  SL_CHECK(window >= 0 && chunk >= 0 && keep_first >= 0 && softcap >= 0.f,
           "window attention: window, chunk, keep_first and the cap must be >= 0");
  SL_CHECK(nsplit >= 1 && nsplit <= 64, "window attention: 1..64 shares of the keys");
  SL_CHECK(nsplit == 1 || (part_o != nullptr && part_ml != nullptr),
           "window attention: shares of the keys need the partial buffers");
  SL_CHECK(gate == nullptr || gate_stride >= nh, "window attention: gate rows are shorter than the heads");
  SL_CHECK(channel_gate == nullptr || channel_stride >= nh * Dv, "window attention: gate rows are shorter than the output");
  SL_CHECK((uintptr_t)q % 16 == 0 && q_stride % 8 == 0 && (uintptr_t)kc % 16 == 0 && (uintptr_t)vc % 16 == 0 &&
           (uintptr_t)out % 8 == 0 && (uintptr_t)part_o % 16 == 0,
           "window attention (matrix cores): operands must be 16-byte aligned");
  if (num_seqs == 0 || num_tokens == 0) return nullptr;
  const WindowAttention a{(const act_t*)q, q_stride, (const act_t*)kc, (const act_t*)vc, tables, max_pages,
                          cu_q, positions, nh, nkv, Dk, Dv, page, scale, softcap, window, chunk, keep_first, slopes, sinks,
                          (const act_t*)gate, gate_stride, channel_gate, channel_stride, (act_t*)out, nsplit, part_o,
                          part_ml};
  if (step && STEP_BLOCKS > 0 && max_q_len == 1 && num_tokens == num_seqs && (nsplit == 1 || (uintptr_t)part_ml % 8 == 0) &&
      (long long)nkv * ((nh / nkv + 15) / 16) <= 65535) {              // (a token each)
    const char* e = launch_step(a, num_seqs, stream);
    if (e || nsplit == 1) return e;
    launch_combine(a, num_tokens, stream);
    return sl_launch_status();
  }
  const long long cols = (long long)max_q_len * (nh / nkv);
  const long long tiles = (cols + COLS - 1) / COLS;
  SL_CHECK(tiles * nsplit <= 1 << 30, "window attention: too many column tiles");
  const long long full = (long long)num_seqs * max_q_len;         // tokens if every sequence had as many as the longest
  const int order = num_tokens == full && tiles * nsplit <= 65535 ? BY_LENGTH :
                    4ll * num_tokens >= 3 * full ? BY_LENGTH_MOVED : LATE_FIRST;
  // (sequence by sequence: an odd number of tiles for each, so that the first tiles, which is all that single tokens among prompts have, lie on
  // all dies; with a multiple of eight they are one die's: a prompt of 1,000 tokens beside 31 single ones, 8 heads on 8, 128 / 128, 190 us and 41 so)
  const unsigned items = (unsigned)(tiles * nsplit) | (order == LATE_FIRST ? 1u : 0u);
  const dim3 grid = order == BY_LENGTH ? dim3(nkv, num_seqs, items) : dim3(items, nkv, num_seqs);
  const char* e = few || !MANY ? launch_mfma<FEW_TEAMS, FEW_PARTS>(a, grid, order, stream)
                               : launch_mfma<MANY ? 1 : FEW_TEAMS, MANY ? 1 : FEW_PARTS>(a, grid, order, stream);
  if (e || nsplit == 1) return e;
  launch_combine(a, num_tokens, stream);
  return sl_launch_status();
}
