// Routed-expert (MoE) block for 1..max_tokens tokens.
//
// The reference offloads expert projections given expert ids (GGML
// MUL_MAT_ID, ollama-xdna/backend/ggml-xdna.cpp:1301-1441; Colibri expert
// group, colibri-xdna/backend/backend_xdna.cpp:316-348: gate, up, silu(g)*u,
// down).  This file adds the router and the combine around them:
//   router        r = W_router @ x (float32), 16 experts of one token per
//                 workgroup (router_logits); then p = softmax(r), top-k by p
//                 with ties to the lower expert id (one wave per token, lane =
//                 expert)
//   plan          groups the (token, expert) pairs by expert, in one workgroup
//                 (with the top-k for small batches): the shared experts
//                 (every token, weight 1) and the routed experts in id order,
//                 in groups of at most 64 rows
//   expert GEMMs  gate/up + SwiGLU, then down, each expert's weights streamed
//                 once per group (expert_slab: one workgroup per 16 or 32
//                 outputs of a group, K split over its waves, the weights
//                 read from MFMA-native copies)
//   combine       y = bf16(sum_k p_k * e_k + sum_s e_s) in float32, rank order,
//                 one thread per output element
// Rounding points follow the dense layer: bf16 after gate/up, after SwiGLU and
// after down.
#include <algorithm>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/hk.h"
#include "hk_common.h"
#include "hk_internal.h"

namespace hk {
namespace {

#define MOE_CHECK(expr)                                   \
  do {                                                    \
    const hipError_t err_ = (expr);                       \
    if (err_ != hipSuccess) return hip_fail(err_, #expr); \
  } while (0)
#define MOE_TRY(expr)         \
  do {                        \
    const int rc_ = (expr);   \
    if (rc_ != 0) return rc_; \
  } while (0)

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kMaxRouted = 64;   // one lane per routed expert
constexpr int kMaxShared = 8;
constexpr int kMaxTopK = 16;
constexpr int kMaxWidth = 1 << 25;  // 64 rows of activations are one buffer resource (expert_slab)

constexpr int kRouterRows = 16;  // routed experts per router_logits workgroup
constexpr int kPlanThreads = 1024;
constexpr int kPlanTokens = kPlanThreads / 64;  // topk_plan: one wave per token
constexpr int kMaxTokens = 256;
constexpr int kMaxPairWords = kMaxTokens * kMaxTopK / 64;

// r[t][e] = W_router[e] . x[t] in float32 for the kRouterRows experts e0.. of
// token t = blockIdx.x: wave w takes experts e0 + 4 w .. + 3 and requests
// every lane's chunks of the four rows at once.  Per expert row the lane sums
// its chunks c = lane + 64 j in order into two accumulators (even and odd
// elements), and the 64 lanes are added by group_sum.
__global__ __launch_bounds__(kThreads) void router_logits_kernel(const uint16_t* x, const uint16_t* router,
                                                                 int H, int E, float* logits) {
  constexpr int R = kRouterRows / (kThreads / 64);  // rows per wave
  constexpr int J = 4;                               // chunks per lane per round
  const int t = blockIdx.x;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int e0 = blockIdx.y * kRouterRows + wave * R;
  const int CH = H / 8;
  const uint16_t* xt = x + (size_t)t * H;
  float a0[R], a1[R];
#pragma unroll
  for (int r = 0; r < R; ++r) a0[r] = a1[r] = 0.0f;
  const u32x4 zero = {0u, 0u, 0u, 0u};
  for (int c0 = 0; c0 < CH; c0 += 64 * J) {
    u32x4 xv[J], wv[R][J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int c = c0 + lane + 64 * j;
      xv[j] = c < CH ? load16(xt + c * 8) : zero;
#pragma unroll
      for (int r = 0; r < R; ++r) wv[r][j] = c < CH && e0 + r < E ? load16(router + (size_t)(e0 + r) * H + c * 8) : zero;
    }
#pragma unroll
    for (int j = 0; j < J; ++j)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const u32x4 v = wv[r][j], xx = xv[j];
        a0[r] = fmaf(bf_lo(v.x), bf_lo(xx.x), a0[r]);
        a1[r] = fmaf(bf_hi(v.x), bf_hi(xx.x), a1[r]);
        a0[r] = fmaf(bf_lo(v.y), bf_lo(xx.y), a0[r]);
        a1[r] = fmaf(bf_hi(v.y), bf_hi(xx.y), a1[r]);
        a0[r] = fmaf(bf_lo(v.z), bf_lo(xx.z), a0[r]);
        a1[r] = fmaf(bf_hi(v.z), bf_hi(xx.z), a1[r]);
        a0[r] = fmaf(bf_lo(v.w), bf_lo(xx.w), a0[r]);
        a1[r] = fmaf(bf_hi(v.w), bf_hi(xx.w), a1[r]);
      }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float v = group_sum<64>(a0[r] + a1[r]);
    if (lane == 0 && e0 + r < E) logits[t * E + e0 + r] = v;
  }
}

// The largest of the wave's 64 values in every lane (DPP row moves, then the
// last lane's value: a few cycles per step, where a shuffle goes through LDS).
__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
  auto step = [&](uint32_t w) { v = max(v, w); };
  step(__builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, false));   // quad_perm 1,0,3,2
  step(__builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, false));   // quad_perm 2,3,0,1
  step(__builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, false));  // row_half_mirror
  step(__builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, false));  // row_mirror
  step(__builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));  // row_bcast15 into rows 1 and 3
  step(__builtin_amdgcn_update_dpp(0, v, 0x143, 0x8, 0xf, false));  // row_bcast31 into row 3
  return __builtin_amdgcn_readlane(v, 63);
}

// p = softmax(r) over the routed experts and the top K by p (ties to the
// lower expert id) of token t, on one wave (lane = expert).
__device__ __forceinline__ void topk_wave(const float* logits, int t, int E, int K, int lane, int32_t* ids,
                                          float* weights, int32_t* ids_lds) {
  const bool live = lane < E;
  const float r = live ? logits[t * E + lane] : -INFINITY;
  const float m = group_max<64>(r);
  const float ex = live ? expf(r - m) : 0.0f;
  const float s = group_sum<64>(ex);
  const float p = ex / s;
  // an order-preserving key per lane, never zero; the lowest lane that holds
  // the largest key is the expert that argmax over (p, -id) gives
  uint32_t key = live ? (uint32_t)(argmax_key(p, 0) >> 32) : 0u;
  int mine = 0;
  float pmine = 0.0f;
  for (int k = 0; k < K; ++k) {
    const int idx = __ffsll(__ballot(key == wave_umax(key))) - 1;
    const float pw = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p), idx));
    if (lane == k) mine = idx, pmine = pw;
    if (lane == idx) key = 0u;
  }
  if (lane < K) {
    ids[t * K + lane] = mine;
    weights[t * K + lane] = pmine;
    if (ids_lds) ids_lds[t * K + lane] = mine;
  }
}

// One launch entry of the expert GEMMs: at most kGroupRows rows of an expert,
// rows 0 for an entry past the last.
struct ExpertGroup {
  int expert, offset, rows, unused;
};
constexpr int kGroupRows = 64;

struct PlanLds {
  unsigned long long bits[kMaxRouted][kMaxPairWords];  // expert e's pairs, one bit each
  uint16_t before[kMaxRouted][kMaxPairWords];          // its pairs before word w
  int32_t ids[kMaxTokens * kMaxTopK];
  int counts[kMaxRouted];
  int offs[kMaxRouted + kMaxShared];
  int n_groups;
};

// The grouping of the T*(K+S) (token, expert) pairs by expert, from the ids
// in LDS, on the calling workgroup (every thread calls it): pair i = t K + k
// sets bit i of its expert's mask, and its slot is the expert's offset plus
// the number of the expert's pairs before it (the popcounts of the whole
// words before its own, from a prefix sum per expert, and of the word's lower
// bits), so the slots follow pair order whatever the timing and an expert may
// appear twice for a token.  A serial walk over the pairs by one thread per
// expert had taken 200 us of a 256-token call; the masks take about 4.  The
// groups list the shared experts first (every token: the longest), then the
// non-empty routed ones in id order, in runs of at most kGroupRows rows; the
// slots list the routed pairs by expert, then the shared experts' rows.
__device__ void plan_pairs(PlanLds& l, int T, int K, int E, int S, int max_groups, ExpertGroup* groups,
                           int32_t* a_rows, int32_t* pair_slot) {
  static_assert(kMaxRouted <= 64 && kMaxPairWords <= 64, "one lane per routed expert and per word of pairs");
  const int tid = threadIdx.x, nt = blockDim.x, wave = tid >> 6, lane = tid & 63;
  const int P = T * K, W = (P + 63) / 64, per = K + S;
  auto expert_of = [&](int i) { return min(max(l.ids[i], 0), E - 1); };
  for (int i = tid; i < E * W; i += nt) l.bits[i / W][i % W] = 0ull;
  __syncthreads();
  for (int i = tid; i < P; i += nt) atomicOr(&l.bits[expert_of(i)][i >> 6], 1ull << (i & 63));
  __syncthreads();
  auto inclusive = [&](int v) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(v, d, 64);
      if (lane >= d) v += up;
    }
    return v;
  };
  if (W <= 8) {  // (small batches: a thread per expert, no scan over lanes)
    for (int e = tid; e < E; e += nt) {
      int sum = 0;
      for (int w = 0; w < W; ++w) {
        l.before[e][w] = (uint16_t)sum;
        sum += __popcll(l.bits[e][w]);
      }
      l.counts[e] = sum;
    }
  } else {
    for (int e = wave; e < E; e += nt / 64) {
      const int c = lane < W ? __popcll(l.bits[e][lane]) : 0;
      const int incl = inclusive(c);
      if (lane < W) l.before[e][lane] = (uint16_t)(incl - c);
      if (lane == 63) l.counts[e] = incl;
    }
  }
  __syncthreads();
  if (wave == 0) {
    const int shared_runs = (T + kGroupRows - 1) / kGroupRows;
    const int c = lane < E ? l.counts[lane] : 0, runs = (c + kGroupRows - 1) / kGroupRows;
    const int off = inclusive(c) - c, last_run = inclusive(runs), first = S * shared_runs + last_run - runs;
    if (lane < E) {
      l.offs[lane] = off;
      for (int j = 0; j < runs; ++j)
        groups[first + j] = {lane, off + j * kGroupRows, min(kGroupRows, c - j * kGroupRows), 0};
    }
    if (lane < S) {
      const int so = P + lane * T;
      l.offs[E + lane] = so;
      for (int j = 0; j < shared_runs; ++j)
        groups[lane * shared_runs + j] = {E + lane, so + j * kGroupRows, min(kGroupRows, T - j * kGroupRows), 0};
    }
    if (lane == 63) l.n_groups = S * shared_runs + last_run;
  }
  __syncthreads();
  for (int i = l.n_groups + tid; i < max_groups; i += nt) groups[i] = {0, 0, 0, 0};
  for (int i = tid; i < T * per; i += nt) {
    const int t = i / per, k = i % per;
    int slot;
    if (k < K) {
      const int pair = t * K + k, e = expert_of(pair), w = pair >> 6;
      slot = l.offs[e] + l.before[e][w] + __popcll(l.bits[e][w] & ((1ull << (pair & 63)) - 1ull));
    } else {
      slot = l.offs[E + k - K] + t;
    }
    a_rows[slot] = t;
    pair_slot[t * per + k] = slot;
  }
}

// Top-k of every token (one wave each) and the plan, one workgroup: batches
// of up to kPlanTokens tokens, one token per wave.
__global__ __launch_bounds__(kPlanThreads) void topk_plan_kernel(const float* logits, int T, int E, int K, int S,
                                                                 int max_groups, int32_t* ids, float* weights,
                                                                 ExpertGroup* groups, int32_t* a_rows,
                                                                 int32_t* pair_slot) {
  __shared__ PlanLds l;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (wave < T) topk_wave(logits, wave, E, K, lane, ids, weights, l.ids);
  __syncthreads();
  plan_pairs(l, T, K, E, S, max_groups, groups, a_rows, pair_slot);
}

// Top-k alone, for larger batches: one wave per token over many workgroups
// (16 tokens after each other on each wave of one workgroup took 35 us of a
// 256-token call).
__global__ __launch_bounds__(kThreads) void topk_kernel(const float* logits, int T, int E, int K, int32_t* ids,
                                                        float* weights) {
  const int t = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
  if (t < T) topk_wave(logits, t, E, K, threadIdx.x & 63, ids, weights, nullptr);
}

// The plan alone: ids from topk_kernel or the caller.
__global__ __launch_bounds__(kPlanThreads) void route_plan_kernel(const int32_t* ids, int T, int K, int E, int S,
                                                                  int max_groups, ExpertGroup* groups,
                                                                  int32_t* a_rows, int32_t* pair_slot) {
  __shared__ PlanLds l;
  for (int i = threadIdx.x; i < T * K; i += kPlanThreads) l.ids[i] = ids[i];
  __syncthreads();
  plan_pairs(l, T, K, E, S, max_groups, groups, a_rows, pair_slot);
}

// y[t][d] = bf16(sum_k p_k e_k[d] + sum_s e_s[d]) in float32, ranks in order;
// one thread per (t, d): every expert output of the element requested at once.
__global__ __launch_bounds__(kThreads) void combine_kernel(const uint16_t* out, const int32_t* pair_slot,
                                                           const float* weights, int H, int K, int S,
                                                           uint16_t* y) {
  const int t = blockIdx.x;
  const int d = blockIdx.y * kThreads + threadIdx.x;
  if (d >= H) return;
  const int per = K + S;
  float v[kMaxTopK + kMaxShared];
#pragma unroll
  for (int k = 0; k < kMaxTopK + kMaxShared; ++k)
    v[k] = k < per ? bf16_to_f32(out[(size_t)pair_slot[t * per + k] * H + d]) : 0.0f;
  float acc = 0.0f;
  for (int k = 0; k < K; ++k) acc = acc + weights[t * K + k] * v[k];
  for (int s = 0; s < S; ++s) acc = acc + v[K + s];
  y[(size_t)t * H + d] = (uint16_t)f32_to_bf16(acc);
}

// SwiGLU of the bf16 gate and up sums, as in the dense layer's GEMMs.
__device__ __forceinline__ float silu_mul(float g, float u) {
  const float clipped = fminf(fmaxf(g, -80.0f), 80.0f);
  return (g / (1.0f + expf(-clipped))) * u;
}

struct ExpertGemmArgs {
  const uint16_t* A;          // row-major bf16 rows of K values
  const uint16_t* Wn;         // MFMA-native copies of the experts' weights, w_stride apart
  uint16_t* Y;                // [slots, N]
  const ExpertGroup* groups;  // gridDim.y entries
  const int32_t* a_rows;      // A row of each slot (PAIR; else the slot itself)
  long long w_stride;
  int N, K, a_bytes;          // bytes of A (PAIR)
};

// The outputs n0 .. of one group on RB blocks of 16 rows, NF weight fragments
// of 16 weight rows per K step (PAIR: NF / 2 gate and NF / 2 up ones); see
// expert_slab_kernel.
template <bool PAIR, int NF, int WAVES, int RB, int DEPTH>
__device__ __forceinline__ void expert_slab(const ExpertGemmArgs& a, const ExpertGroup& g, int n0, f32x4* red) {
  constexpr int NO = PAIR ? NF / 2 : NF;  // 16-output blocks
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fk = (lane >> 4) * 8;
  const int N = a.N, K = a.K;
  // Wn of an expert: [rows / 16][K / 8][16] pieces of 8 weights, so a
  // fragment's 16 rows are one 256-byte run, a wave's K step one 1 KiB run and
  // the 16 rows in all one run of 32 K bytes: a buffer resource each, so that
  // no 32-bit size or offset spans the whole matrix (2 GiB and more from 2^30
  // weights).  Where the rows of A follow each other, one resource over the
  // group's (a resource per 16 rows: 233.1 us per 256-token call, so 231.8).
  // Steps, outputs and rows past the ends read zero.
  const uint16_t* We = a.Wn + (size_t)g.expert * (size_t)a.w_stride;
  __amdgpu_buffer_rsrc_t wr[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int n = n0 + 16 * (f % NO), r = f < NO ? n : N + n;
    wr[f] = rsrc(We + (size_t)r * K, n < N ? 32 * K : 0);
  }
  constexpr unsigned kOutside = PAIR ? 0x7ffffff0u : 0xfffffff0u;  // past every resource of A
  const unsigned wofs = (unsigned)((fk >> 3) * 16 + fr) * 16u;  // this lane's piece of a fragment
  const __amdgpu_buffer_rsrc_t rr = rsrc(PAIR ? a.a_rows + g.offset : nullptr, PAIR ? g.rows * 4 : 0);
  const __amdgpu_buffer_rsrc_t ar =
      PAIR ? rsrc(a.A, a.a_bytes) : rsrc(a.A + (size_t)g.offset * K, (int)(2u * (unsigned)g.rows * (unsigned)K));
  unsigned row[RB];  // the numbers of this lane's A rows in it
#pragma unroll
  for (int b = 0; b < RB; ++b)
    row[b] = PAIR ? __builtin_amdgcn_raw_buffer_load_b32(rr, (16 * b + fr) * 4, 0, 0) : 16 * b + fr;
  const int steps = K / 32;
  const int mine = steps > wave ? (steps - wave + WAVES - 1) / WAVES : 0;
  f32x4 acc[RB][NF];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[b][f] = f32x4{0.f, 0.f, 0.f, 0.f};
  // a ring of DEPTH K steps per wave: a step's products free its slot for the
  // loads of the step DEPTH on, so about DEPTH steps stay in flight (the
  // barriers keep the scheduler from pairing each load with its use)
  u32x4 w[DEPTH][NF], x[DEPTH][RB];
  unsigned aofs[RB];
  auto load_w = [&](int slot, int j) {
    const unsigned k0w = (unsigned)(wave + WAVES * j) * 1024u;  // four k groups of 16 pieces
#pragma unroll
    for (int f = 0; f < NF; ++f)
      w[slot][f] = __builtin_amdgcn_raw_buffer_load_b128(wr[f], wofs + k0w, 0, 2);  // (past K: outside)
  };
  auto load_x = [&](int slot, int j) {
    const unsigned k0b = (unsigned)(wave + WAVES * j) * 64u;  // bytes along an A row
#pragma unroll
    for (int b = 0; b < RB; ++b)
      x[slot][b] = __builtin_amdgcn_raw_buffer_load_b128(ar, j < mine ? aofs[b] + k0b : kOutside, 0, 0);
  };
  auto multiply = [&](int slot) {
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int f = 0; f < NF; ++f)
        acc[b][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x[slot][b]),
                                                            __builtin_bit_cast(bf16x8, w[slot][f]), acc[b][f], 0, 0, 0);
  };
#pragma unroll
  for (int i = 0; i < DEPTH; ++i) load_w(i, i);
  __builtin_amdgcn_sched_barrier(0);
  // (after the weight loads: the rows' numbers are waited for here)
#pragma unroll
  for (int b = 0; b < RB; ++b)
    aofs[b] = !PAIR || 16 * b + fr < g.rows ? (row[b] * (unsigned)K + fk) * 2u : kOutside;
#pragma unroll
  for (int i = 0; i < DEPTH; ++i) load_x(i, i);
  __builtin_amdgcn_sched_barrier(0);
  for (int j0 = 0; j0 + DEPTH < mine; j0 += DEPTH) {
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
      multiply(i);
      load_w(i, j0 + DEPTH + i);
      load_x(i, j0 + DEPTH + i);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int i = 0; i < DEPTH; ++i) multiply(i);  // (slots past the last step hold zeros)
  auto part = [&](int wv, int b, int f) -> f32x4& { return red[((wv * RB + b) * NF + f) * 64 + lane]; };
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int f = 0; f < NF; ++f) part(wave, b, f) = acc[b][f];
  __syncthreads();
  // the waves add the (row block, output block) pairs over all waves, in wave
  // order.  D layout: lane holds rows 4 (lane / 16) + r, output lane % 16
  for (int it = wave; it < RB * NO; it += WAVES) {
    const int b = it / NO, o = it % NO, n = n0 + 16 * o + fr;
    f32x4 s0 = part(0, b, o), s1 = PAIR ? part(0, b, NO + o) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int wv = 1; wv < WAVES; ++wv) {
      s0 += part(wv, b, o);
      if constexpr (PAIR) s1 += part(wv, b, NO + o);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * b + 4 * (lane >> 4) + r;
      if (i >= g.rows || n >= N) continue;
      const float y = PAIR ? silu_mul(round_bf16(s0[r]), round_bf16(s1[r])) : s0[r];
      a.Y[(size_t)(g.offset + i) * N + n] = (uint16_t)f32_to_bf16(y);
    }
  }
}

// Expert GEMM over the plan's groups: workgroup (s, z) computes NF / 2 blocks
// of 16 gate and up outputs (PAIR: SwiGLU bf16(silu(bf16(g)) * bf16(u))) or
// NF blocks of plain ones of group z's expert, for the group's rows (at most
// kGroupRows).  Wave w takes the 32-column K steps w, w + WAVES, ... and
// multiplies on MFMA 16x16x32 (rows x outputs); the waves' partial sums meet
// in LDS and are added in wave order.  A group runs on as many 16-row blocks
// as it has rows for, with a shorter ring of steps in flight for more.
//
// HBM bounds it up to about 10 rows per expert: every expert's weights go by
// once per group (66 experts of 2048 x 1408 in 120 us for gate/up, 6.3 TB/s).
// With more rows the A fragments, re-read from L2 by every workgroup of the
// group, weigh as much as the weights; WIDE halves them with twice the
// outputs per workgroup, on half the waves with twice the registers (the same
// two workgroups per CU).  Whole calls of a 2048 / 64 + 2 x 1408 / top-6
// block, narrow and wide: 1 token 38.8 and 40.1 us, 24 169 and 170, 61 195
// and 188, 100 210 and 199, 256 302 and 238 (750 on 64 x 64 tiles of the
// row-major weights with the plan's slots by a serial walk).
template <bool PAIR, bool WIDE>
__global__ __launch_bounds__(WIDE ? 256 : 512, WIDE ? 2 : 4) void expert_slab_kernel(ExpertGemmArgs a) {
  constexpr int NF = WIDE ? 4 : 2, WAVES = WIDE ? 4 : 8;
  __shared__ f32x4 red[WAVES * (kGroupRows / 16) * NF * 64];
  const int4 e = reinterpret_cast<const int4*>(a.groups)[blockIdx.y];
  const ExpertGroup g = {e.x, e.y, e.z, 0};
  if (g.rows == 0) return;
  const int n0 = blockIdx.x * 16 * (PAIR ? NF / 2 : NF);
  if (g.rows <= 16)
    expert_slab<PAIR, NF, WAVES, 1, 8>(a, g, n0, red);
  else if (g.rows <= 32)
    expert_slab<PAIR, NF, WAVES, 2, 6>(a, g, n0, red);
  else
    expert_slab<PAIR, NF, WAVES, 4, WIDE ? 4 : 3>(a, g, n0, red);
}

template <bool PAIR>
int launch_expert_slab(const ExpertGemmArgs& a, int groups, bool wide, hipStream_t st) {
  const int outs = (PAIR ? 16 : 32) * (wide ? 2 : 1);  // per workgroup
  const dim3 grid((a.N + outs - 1) / outs, groups);
  if (wide)
    hipLaunchKernelGGL((expert_slab_kernel<PAIR, true>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((expert_slab_kernel<PAIR, false>), grid, dim3(512), 0, st, a);
  MOE_CHECK(hipGetLastError());
  return 0;
}

// Tokens from which the expert GEMMs run WIDE.  What decides is the rows per
// expert and how many workgroups an expert makes; the line is in tokens, where
// the 2048 / 64 + 2 x 1408 / top-6 block is even (24 to 32; 4% of a call at 61).
// Narrow and wide elsewhere, us per call: 8 experts of 2048 x 4096, top-2, 4
// tokens 64.7 and 61.4, 32 84.6 and 78.0; of 4096 x 7168, 8 tokens 142 and 154,
// 24 218 and 220, 32 226 and 221; 64 of 2048 x 1408, top-1, 64 tokens 118 and
// 124, 256 182 and 181.
constexpr int kWideTokens = 33;

}  // namespace
}  // namespace hk

using namespace hk;

struct hk_moe {
  std::mutex mu;
  hk_moe_desc d{};
  const uint16_t* router = nullptr;
  uint16_t* gate_up_n = nullptr;  // MFMA-native copies of every expert (expert_slab_kernel)
  uint16_t* down_n = nullptr;
  float* logits = nullptr;       // [max_tokens * experts] router outputs
  int32_t* ids = nullptr;        // [max_tokens * top_k]
  float* weights = nullptr;      // [max_tokens * top_k]
  ExpertGroup* groups = nullptr;
  int32_t* a_rows = nullptr;     // [pairs]
  int32_t* pair_slot = nullptr;  // [max_tokens * (top_k + shared)]
  uint16_t* act = nullptr;       // [pairs, I]
  uint16_t* out = nullptr;       // [pairs, H]
};

namespace {

void moe_free(hk_moe* m) {
  void* bufs[] = {m->gate_up_n, m->down_n, m->logits, m->ids, m->weights, m->groups, m->a_rows, m->pair_slot, m->act, m->out};
  for (void* p : bufs)
    if (p) (void)hipFree(p);
  delete m;
}

// Groups that T tokens can make: every run of kGroupRows rows of an expert.
int max_groups(const hk_moe_desc& d, int T) {
  const int pairs = T * d.top_k, runs = (T + kGroupRows - 1) / kGroupRows;
  return std::min(d.experts, pairs) + pairs / kGroupRows + d.shared * runs;
}

// Tokens whose rows one buffer resource spans (expert_slab's A rows are
// gathered from all of them): a call of more runs in as many passes.
int pass_tokens(const hk_moe_desc& d) { return std::max(1, 0x3ffffff0 / d.hidden); }

// The expert GEMMs and the combine, after the plan.
int moe_run(hk_moe* m, const uint16_t* x, int T, const float* weights, uint16_t* y, hipStream_t st) {
  const hk_moe_desc& d = m->d;
  const int groups = max_groups(d, T);
  ExpertGemmArgs gu = {};
  gu.A = x;
  gu.Wn = m->gate_up_n;
  gu.Y = m->act;
  gu.groups = m->groups;
  gu.a_rows = m->a_rows;
  gu.w_stride = (long long)2 * d.intermediate * d.hidden;
  gu.N = d.intermediate;
  gu.K = d.hidden;
  gu.a_bytes = T * d.hidden * 2;
  MOE_TRY(launch_expert_slab<true>(gu, groups, T >= kWideTokens, st));
  ExpertGemmArgs dn = gu;
  dn.A = m->act;
  dn.Wn = m->down_n;
  dn.Y = m->out;
  dn.a_rows = nullptr;
  dn.w_stride = (long long)d.hidden * d.intermediate;
  dn.N = d.hidden;
  dn.K = d.intermediate;
  MOE_TRY(launch_expert_slab<false>(dn, groups, T >= kWideTokens, st));
  hipLaunchKernelGGL(combine_kernel, dim3(T, (d.hidden + kThreads - 1) / kThreads), dim3(kThreads), 0, st, m->out,
                     m->pair_slot, weights, d.hidden, d.top_k, d.shared, y);
  MOE_CHECK(hipGetLastError());
  return 0;
}

int plan_route(hk_moe* m, const int32_t* ids, int T, hipStream_t st) {
  const hk_moe_desc& d = m->d;
  hipLaunchKernelGGL(route_plan_kernel, dim3(1), dim3(kPlanThreads), 0, st, ids, T, d.top_k, d.experts, d.shared,
                     max_groups(d, T), m->groups, m->a_rows, m->pair_slot);
  MOE_CHECK(hipGetLastError());
  return 0;
}

// The router, the top-k and the plan of T tokens.
int route(hk_moe* m, const uint16_t* x, int T, int32_t* ids, float* weights, hipStream_t st) {
  const hk_moe_desc& d = m->d;
  hipLaunchKernelGGL(router_logits_kernel, dim3(T, (d.experts + kRouterRows - 1) / kRouterRows), dim3(kThreads), 0,
                     st, x, m->router, d.hidden, d.experts, m->logits);
  MOE_CHECK(hipGetLastError());
  // one token per wave of the plan's workgroup, or the top-k spread over the
  // GPU and the plan after it (one launch more)
  if (T <= kPlanTokens) {
    hipLaunchKernelGGL(topk_plan_kernel, dim3(1), dim3(kPlanThreads), 0, st, m->logits, T, d.experts, d.top_k,
                       d.shared, max_groups(d, T), ids, weights, m->groups, m->a_rows, m->pair_slot);
    MOE_CHECK(hipGetLastError());
    return 0;
  }
  hipLaunchKernelGGL(topk_kernel, dim3((T + kThreads / 64 - 1) / (kThreads / 64)), dim3(kThreads), 0, st, m->logits,
                     T, d.experts, d.top_k, ids, weights);
  MOE_CHECK(hipGetLastError());
  return plan_route(m, ids, T, st);
}

template <typename T>
int moe_alloc(T** p, size_t count) {
  MOE_CHECK(hipMalloc(reinterpret_cast<void**>(p), count * sizeof(T)));
  return 0;
}

}  // namespace

extern "C" {

int hk_moe_create(const hk_moe_desc* desc, const uint16_t* router, const uint16_t* gate_up,
                  const uint16_t* down, hk_moe** out) {
  if (!desc || !router || !gate_up || !down || !out) return fail("hk_moe_create: null argument");
  *out = nullptr;
  const hk_moe_desc& d = *desc;
  if (d.experts <= 0 || d.experts > kMaxRouted) return fail("hk_moe_create: 1..64 routed experts");
  if (d.shared < 0 || d.shared > kMaxShared) return fail("hk_moe_create: 0..8 shared experts");
  if (d.top_k <= 0 || d.top_k > d.experts || d.top_k > kMaxTopK) return fail("hk_moe_create: bad top_k");
  if (d.hidden <= 0 || d.hidden % 32 || d.intermediate <= 0 || d.intermediate % 32)
    return fail("hk_moe_create: hidden and intermediate must be positive multiples of 32");
  if (d.hidden >= kMaxWidth || d.intermediate >= kMaxWidth)
    return fail("hk_moe_create: hidden and intermediate must be below 2^25");
  if (d.max_tokens <= 0 || d.max_tokens > 256) return fail("hk_moe_create: max_tokens must be 1..256");
  hk_moe* m = new hk_moe();
  m->d = d;
  m->router = router;
  const size_t pairs = (size_t)d.max_tokens * (d.top_k + d.shared);
  const size_t groups = (size_t)d.experts + d.shared;
  auto body = [&]() -> int {
    // the MFMA-native copies, one repack per expert matrix
    const size_t gu_n = (size_t)2 * d.intermediate * d.hidden, dn_n = (size_t)d.hidden * d.intermediate;
    MOE_TRY(moe_alloc(&m->gate_up_n, groups * gu_n));
    MOE_TRY(moe_alloc(&m->down_n, groups * dn_n));
    for (size_t e = 0; e < groups; ++e) {
      MOE_TRY(launch_repack_mfma(gate_up + e * gu_n, m->gate_up_n + e * gu_n, 2 * d.intermediate, d.hidden, 2, 0,
                                 nullptr));
      MOE_TRY(launch_repack_mfma(down + e * dn_n, m->down_n + e * dn_n, d.hidden, d.intermediate, 2, 0, nullptr));
    }
    MOE_CHECK(hipStreamSynchronize(nullptr));
    MOE_TRY(moe_alloc(&m->logits, (size_t)d.max_tokens * d.experts));
    MOE_TRY(moe_alloc(&m->ids, (size_t)d.max_tokens * d.top_k));
    MOE_TRY(moe_alloc(&m->weights, (size_t)d.max_tokens * d.top_k));
    MOE_TRY(moe_alloc(&m->groups, max_groups(d, d.max_tokens)));
    MOE_TRY(moe_alloc(&m->a_rows, pairs));
    MOE_TRY(moe_alloc(&m->pair_slot, pairs));
    MOE_TRY(moe_alloc(&m->act, pairs * d.intermediate));
    MOE_TRY(moe_alloc(&m->out, pairs * d.hidden));
    return 0;
  };
  const int rc = body();
  if (rc != 0) {
    moe_free(m);
    return rc;
  }
  *out = m;
  return 0;
}

int hk_moe_forward(hk_moe* m, const uint16_t* x, int32_t tokens, uint16_t* y, int32_t* ids_out,
                   float* weights_out, void* stream) {
  if (!m || !x || !y) return fail("hk_moe_forward: null argument");
  std::lock_guard<std::mutex> lock(m->mu);
  if (tokens <= 0 || tokens > m->d.max_tokens) return fail("hk_moe_forward: token count out of range");
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const hk_moe_desc& d = m->d;
  for (int t0 = 0, T; t0 < tokens; t0 += T) {
    T = std::min(tokens - t0, pass_tokens(d));
    const size_t row = (size_t)t0 * d.hidden, pick = (size_t)t0 * d.top_k;
    MOE_TRY(route(m, x + row, T, m->ids + pick, m->weights + pick, st));
    MOE_TRY(moe_run(m, x + row, T, m->weights + pick, y + row, st));
  }
  const size_t nk = (size_t)tokens * d.top_k;
  if (ids_out)
    MOE_CHECK(hipMemcpyAsync(ids_out, m->ids, nk * sizeof(int32_t), hipMemcpyDeviceToDevice, st));
  if (weights_out)
    MOE_CHECK(hipMemcpyAsync(weights_out, m->weights, nk * sizeof(float), hipMemcpyDeviceToDevice, st));
  return 0;
}

int hk_moe_experts(hk_moe* m, const uint16_t* x, int32_t tokens, const int32_t* ids,
                   const float* weights, uint16_t* y, void* stream) {
  if (!m || !x || !ids || !weights || !y) return fail("hk_moe_experts: null argument");
  std::lock_guard<std::mutex> lock(m->mu);
  if (tokens <= 0 || tokens > m->d.max_tokens) return fail("hk_moe_experts: token count out of range");
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const size_t nk = (size_t)tokens * m->d.top_k;
  std::vector<int32_t> host(nk);
  MOE_CHECK(hipMemcpyAsync(host.data(), ids, nk * sizeof(int32_t), hipMemcpyDeviceToHost, st));
  MOE_CHECK(hipStreamSynchronize(st));
  for (int32_t e : host)
    if (e < 0 || e >= m->d.experts) return fail("hk_moe_experts: expert id out of range");
  for (int t0 = 0, T; t0 < tokens; t0 += T) {
    T = std::min(tokens - t0, pass_tokens(m->d));
    const size_t row = (size_t)t0 * m->d.hidden, pick = (size_t)t0 * m->d.top_k;
    MOE_TRY(plan_route(m, ids + pick, T, st));
    MOE_TRY(moe_run(m, x + row, T, weights + pick, y + row, st));
  }
  return 0;
}

void hk_moe_destroy(hk_moe* m) {
  if (m) moe_free(m);
}

}  // extern "C"
