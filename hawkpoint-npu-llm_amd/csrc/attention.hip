// Decode-step attention: RoPE on the new q/k heads, in-place KV append at slot
// `position`, and grouped-query softmax attention over slots 0..position.
//
// Follows npu_llm/runtime/cpu_backend.py:78-129:
//   rotate   [x1*c - x2*s, x2*c + x1*s] on the two 32-wide halves, then bf16
//            (cos/sin come from host tables built with the reference's own
//            NumPy expression, so they match bit for bit)
//   append   K[:, p] = bf16(rot k), V[:, p] = v                    :105-108
//   scores   (q . k) * head_dim**-0.5, minus the row max, exp, / sum   :110-125
//   output   bf16(P @ V)                                          :126-129
//
// Work split: one workgroup per (query head, chunk of 256 slots), four waves
// of 64 slots each, so positions below 256 use one workgroup per query head
// and no merge.  Eight lanes hold a slot's 64 dimensions, 16 bytes each: a
// wave's load is a run of eight slots (1 KiB), the scores are sums over eight
// lanes, and each lane keeps the probabilities of its own eight slots for
// P @ V, so nothing goes through LDS until the four waves' (max, sum, P @ V)
// meet.  With several chunks each workgroup publishes that triple for its
// chunk with device-coherent stores, and the last one of a head to finish (a
// per-head ticket) merges them with log-sum-exp rescaling: thread j fetches
// chunk j's (max, sum), and the four waves share the chunks' P @ V rows.
// What bounds it is latency: a launch, one round trip for the rows, the
// publication and the merge.  14 / 2 heads at position 9001: 12.1 us against 47.2
// with one thread per K row and one wave merging the 36 chunks after each
// other; 32 / 8 heads at 32000 34.7 against 352 (67 MB of K and V: 13 us).
// The KV cache layout is [kv head][slot][64] BF16 per layer, so one slot of
// one head is a contiguous 128-byte row.
#include <algorithm>

#include "hk_common.h"
#include "hk_internal.h"

namespace hk {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kPartStride = kHeadDim + 2;  // acc[64], max, sum
constexpr int kRowsPerLane = 8;            // slots of a wave per lane
constexpr int kSc1 = 16;                   // buffer access cache policy: device scope
static_assert(kAttnChunk == kWaves * 64, "64 slots per wave");
static_assert(kHeadDim == 64, "eight lanes of eight dimensions per slot");
static_assert(kMaxContext / kAttnChunk <= kThreads, "one thread per chunk in the merge");

// The callers' vectors are used at the alignment of their elements.
typedef u32x4 __attribute__((aligned(2))) row16_t;
typedef u32x4 __attribute__((aligned(4))) tab16_t;
__device__ __forceinline__ u32x4 load_row(const uint16_t* p) {
  return *(const __attribute__((address_space(1))) row16_t*)p;
}
__device__ __forceinline__ void store_row(uint16_t* p, const u32x4& v) {
  *(__attribute__((address_space(1))) row16_t*)p = v;
}

__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, a), __builtin_bit_cast(bf16x2_t, b), c, false);
}

// Maximum and sum over the eight lanes 8 apart (the wave's eight slot
// groups), the same value in each: lanes L ^ 8 by a row rotation, L ^ 16 and
// L ^ 32 by lane swaps.
__device__ __forceinline__ float groups_max(float v) {
  v = fmaxf(v, lane_dpp<0x128>(v));
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float groups_sum(float v) {
  v += lane_dpp<0x128>(v);
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Dimensions 8 c .. + 7 of a head row after RoPE, as bf16 pairs: x1 cos - x2
// sin in the first half, x2 cos + x1 sin in the second (own: the row's chunk
// c, other: chunk c ^ 4).
__device__ __forceinline__ u32x4 rotate8(const u32x4& own, const u32x4& other, const float (&cs)[8],
                                         const float (&sn)[8], bool second) {
  u32x4 o;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    float r[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float x = e ? bf_hi(own[w]) : bf_lo(own[w]), y = e ? bf_hi(other[w]) : bf_lo(other[w]);
      const float xc = x * cs[2 * w + e], ys = y * sn[2 * w + e];
      r[e] = second ? xc + ys : xc - ys;
    }
    o[w] = f32x2_to_bf16x2(r[0], r[1]);
  }
  return o;
}

// 2^(score - max) with the maximum of a set of slots.  Where all of them score
// -inf (a key with an infinite component) the maximum is no number to subtract:
// they weigh 0 in the larger set they belong to, and only a row of nothing else
// ends as 0 / 0, as the reference's softmax of it does.
__device__ __forceinline__ float finite_max(float m) { return m == -INFINITY ? 0.0f : m; }

__global__ __launch_bounds__(kThreads) void attention_decode_kernel(AttnArgs a) {
  const int p = a.position ? *a.position : a.pos;
  // workgroup b: chunk and head so that the heads of one chunk, which share
  // its K and V rows, fall on one XCD (workgroups 8 apart) and its L2
  const int width = min(8, a.splits);
  const int r = (int)blockIdx.x / width;
  const int h = r % a.q_heads, s = (r / a.q_heads) * width + (int)blockIdx.x % width;
  const int t0 = s * kAttnChunk;
  if (t0 > p || s >= a.splits) return;
  const int nsplit = p / kAttnChunk + 1;
  const int qpk = a.q_heads / a.kv_heads, g = h / qpk;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c8 = lane & 7, rg = lane >> 3;  // this lane's dimensions 8 c8 .. + 7; its slot of each eight

  __shared__ float wm[kWaves], wl[kWaves];
  __shared__ float wo[kWaves][kHeadDim];
  __shared__ float weight[kThreads];
  __shared__ int last;

  // every load goes out before the first result is used; a slot past the
  // cached ones reads row p of the cache (dropped below)
  const size_t head_base = (size_t)g * a.max_ctx;
  const int w0 = t0 + wave * 64;
  const bool live = w0 <= p;  // (uniform) the wave has slots
  u32x4 kr[kRowsPerLane], vr[kRowsPerLane];
  if (live) {
#pragma unroll
    for (int i = 0; i < kRowsPerLane; ++i) {
      const size_t row = (head_base + min(w0 + 8 * i + rg, p)) * kHeadDim + 8 * c8;
      kr[i] = load_row(a.kcache + row);
      vr[i] = load_row(a.vcache + row);
    }
    const uint16_t* qrow = a.qkv + (size_t)h * kHeadDim;
    const uint16_t* krow = a.qkv + (size_t)(a.q_heads + g) * kHeadDim;
    const uint16_t* vrow = a.qkv + (size_t)(a.q_heads + a.kv_heads + g) * kHeadDim;
    const u32x4 q0 = load_row(qrow + 8 * c8), q1 = load_row(qrow + 8 * (c8 ^ 4));
    const u32x4 k0 = load_row(krow + 8 * c8), k1 = load_row(krow + 8 * (c8 ^ 4));
    const u32x4 vnew = load_row(vrow + 8 * c8);
    float cs[8], sn[8];
    const size_t at = (size_t)p * (kHeadDim / 2) + 8 * (c8 & 3);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const u32x4 cw = *(const __attribute__((address_space(1))) tab16_t*)(a.cos_tab + at + 4 * q);
      const u32x4 sw = *(const __attribute__((address_space(1))) tab16_t*)(a.sin_tab + at + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        cs[4 * q + e] = __uint_as_float(cw[e]);
        sn[4 * q + e] = __uint_as_float(sw[e]);
      }
    }
    // the rotated query and new key (bf16-rounded as the reference does); the
    // first query head of the group appends k and v at slot p
    const u32x4 qr = rotate8(q0, q1, cs, sn, c8 >= 4), knew = rotate8(k0, k1, cs, sn, c8 >= 4);
    if (w0 + 63 >= p && h % qpk == 0 && rg == 0) {  // (the wave that holds slot p)
      store_row(a.kcache + (head_base + p) * kHeadDim + 8 * c8, knew);
      store_row(a.vcache + (head_base + p) * kHeadDim + 8 * c8, vnew);
    }
    float sc[kRowsPerLane], m = -INFINITY;
#pragma unroll
    for (int i = 0; i < kRowsPerLane; ++i) {
      const int slot = w0 + 8 * i + rg;
      if (slot == p) kr[i] = knew, vr[i] = vnew;
      float d = 0.0f;
#pragma unroll
      for (int w = 0; w < 4; ++w) d = dot2(qr[w], kr[i][w], d);
      // base-2 scores: (q . k) / 8 * log2(e)
      sc[i] = slot <= p ? lane_sum<8>(d) * (0.125f * 1.4426950408889634f) : -INFINITY;
      m = fmaxf(m, sc[i]);
    }
    m = groups_max(m);
    const float m_use = finite_max(m);
    float sum = 0.0f, o[8] = {};
#pragma unroll
    for (int i = 0; i < kRowsPerLane; ++i) {
      const float e = __builtin_amdgcn_exp2f(sc[i] - m_use);
      sum += e;
      const bool on = w0 + 8 * i + rg <= p;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        o[2 * w] = fmaf(e, on ? bf_lo(vr[i][w]) : 0.0f, o[2 * w]);
        o[2 * w + 1] = fmaf(e, on ? bf_hi(vr[i][w]) : 0.0f, o[2 * w + 1]);
      }
    }
    sum = groups_sum(sum);
#pragma unroll
    for (int d = 0; d < 8; ++d) o[d] = groups_sum(o[d]);
    if (lane == 0) wm[wave] = m, wl[wave] = sum;
    if (rg == 0) {
#pragma unroll
      for (int d = 0; d < 8; ++d) wo[wave][8 * c8 + d] = o[d];
    }
  } else if (lane == 0) {
    wm[wave] = -INFINITY;
  }
  __syncthreads();
  // the chunk's (max, sum, P @ V), every thread the same max and sum (wave 0
  // always has slots; a wave without any adds nothing)
  float m = wm[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) m = fmaxf(m, wm[w]);
  const float m_use = finite_max(m);
  float l = 0.0f, o = 0.0f;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (t0 + 64 * w > p) break;
    const float f = __builtin_amdgcn_exp2f(wm[w] - m_use);
    l = fmaf(wl[w], f, l);
    o = fmaf(wo[w][lane], f, o);
  }
  uint16_t* out = a.out + (size_t)h * kHeadDim;
  if (nsplit == 1) {
    if (wave == 0) out[lane] = (uint16_t)f32_to_bf16(o / l);
    return;
  }

  // Split-KV.  The triple goes out with device-coherent stores (no L2
  // write-back as a fence would do), all complete before the ticket is drawn.
  float* head_part = a.partial + (size_t)h * a.max_splits * kPartStride;
  const __amdgpu_buffer_rsrc_t pr = rsrc(head_part, nsplit * kPartStride * 4);
  if (wave == 0) {
    const int at = s * kPartStride * 4;
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o), pr, at + 4 * lane, 0, kSc1);
    if (lane < 2) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(lane ? l : m), pr, at + 4 * (kHeadDim + lane), 0, kSc1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (lane == 0)
      last = __hip_atomic_fetch_add(&a.counters[h], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(nsplit - 1);
  }
  __syncthreads();
  if (!last) return;
  // thread j: chunk j's (max, sum); reads past nsplit are past the resource
  const int mine = tid * kPartStride * 4;
  const bool has = tid < nsplit;
  const float cm = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(pr, mine + 4 * kHeadDim, 0, kSc1));
  const float cl = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(pr, mine + 4 * kHeadDim + 4, 0, kSc1));
  // this wave's chunks wave, wave + 4, ...: eight rows in flight
  const int rows = (nsplit - wave + kWaves - 1) / kWaves;  // (nsplit >= 2, may be 0 or less)
  constexpr int kBatch = 8;
  float row[kBatch];
  auto fetch = [&](int j0) {
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
      row[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
          pr, (wave + kWaves * (j0 + j)) * (kPartStride * 4) + 4 * lane, 0, kSc1));
  };
  fetch(0);
  float gm = group_max<64>(has ? cm : -INFINITY);
  if (lane == 0) wm[wave] = gm;
  __syncthreads();
  gm = wm[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) gm = fmaxf(gm, wm[w]);
  const float f = has ? __builtin_amdgcn_exp2f(cm - finite_max(gm)) : 0.0f;
  weight[tid] = f;
  const float ls = group_sum<64>(has ? cl * f : 0.0f);
  if (lane == 0) wl[wave] = ls;
  __syncthreads();
  float acc = 0.0f;
  for (int j0 = 0; j0 < rows; j0 += kBatch) {
    if (j0 > 0) fetch(j0);
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
      if (j0 + j < rows) acc = fmaf(row[j], weight[wave + kWaves * (j0 + j)], acc);
  }
  wo[wave][lane] = acc;
  __syncthreads();
  if (wave != 0) return;
  const float lt = (wl[0] + wl[1]) + (wl[2] + wl[3]);
  out[lane] = (uint16_t)f32_to_bf16(((wo[0][lane] + wo[1][lane]) + (wo[2][lane] + wo[3][lane])) / lt);
  if (lane == 0) __hip_atomic_store(&a.counters[h], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

int launch_attention_decode(const AttnArgs& args, hipStream_t stream) {
  AttnArgs a = args;
  if (a.kv_heads <= 0 || a.q_heads <= 0 || a.q_heads % a.kv_heads != 0)
    return fail("attention: q_heads must be a positive multiple of kv_heads");
  if (a.q_heads / a.kv_heads > kMaxQPerKV) return fail("attention: more than 16 q heads per kv head");
  if (a.max_ctx <= 0 || a.max_ctx > kMaxContext) return fail("attention: context out of range");
  if (a.max_splits < attention_splits(a.max_ctx)) return fail("attention: too few split-KV slots");
  // the position's own chunks where the host knows it, else the context's
  a.splits = a.position ? attention_splits(a.max_ctx) : a.pos / kAttnChunk + 1;
  const int width = std::min(8, a.splits);
  const dim3 grid(a.q_heads * width * ((a.splits + width - 1) / width));
  hipLaunchKernelGGL(attention_decode_kernel, grid, dim3(kThreads), 0, stream, a);
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? 0 : hip_fail(err, "attention launch");
}

}  // namespace hk
