// Routing of a MoE layer on the device: top-k of the router's softmax, and the expert-sorted
// order of the (token, slot) assignments with its segment offsets (train/model.py:158-163,
// kernels/moe_routing.py:116-130).
//
// As torch ops the routing of one layer was about 25 launches of 2 to 24 us each, with three
// copies to the host between them (bincount reads its minimum and maximum): 230 us in front of
// GEMMs of 180 to 550 us. Both steps here are bound by one launch's latency. A layer of 4096 ->
// 14336, top-2 of 8 experts, whole call: 16 tokens 492 -> 219 us, 512 tokens 821 -> 513.
#include "common.h"

namespace mls {

namespace {

constexpr int kMaxExperts = 256, kMaxTop = 8;

// One wavefront a token: lane l holds experts l, l + 64, ... The probabilities are softmax's in
// fp32 (exp of x - max over their sum); each of the k rounds takes the largest one left (the
// lowest expert of equal ones; a NaN counts as the largest, as in torch's topk), and the k
// values are divided by their sum.
template <typename T>
__global__ __launch_bounds__(256) void route_topk_kernel(const T* __restrict__ logits, int64_t ld, int64_t tokens,
                                                         int E, int k, float* __restrict__ weights,
                                                         int64_t* __restrict__ experts) {
  constexpr int C = kMaxExperts / 64;
  const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (t >= tokens) return;
  float v[C], m = -INFINITY;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int e = lane + 64 * c;
    v[c] = e < E ? to_f32(logits[t * ld + e]) : -INFINITY;
    m = fmaxf(m, v[c]);
  }
  m = wave_max(m);
  float s = 0.0f;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    v[c] = lane + 64 * c < E ? expf(v[c] - m) : 0.0f;
    s += v[c];
  }
  s = wave_sum(s);
  // keys that order as the probabilities do (>= 0, so their patterns are), 0 for none
  uint32_t key[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    v[c] = v[c] / s;
    key[c] = lane + 64 * c >= E ? 0u : __builtin_isnan(v[c]) ? 0xFFFFFFFFu : __float_as_uint(v[c]) + 1u;
  }
  float w[kMaxTop], total = 0.0f;
  int idx[kMaxTop];
#pragma unroll
  for (int r = 0; r < kMaxTop; ++r) {
    if (r >= k) break;
    // largest key, then lowest expert: packed as key << 32 | ~expert
    uint64_t best = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const uint64_t p = ((uint64_t)key[c] << 32) | (uint32_t)~(uint32_t)(lane + 64 * c);
      best = p > best && key[c] ? p : best;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      const uint64_t o = (uint64_t)__shfl_xor((unsigned long long)best, off, 64);
      best = o > best ? o : best;
    }
    const int e = (int)~(uint32_t)best;
    idx[r] = e;
    float mine = 0.0f;
#pragma unroll
    for (int c = 0; c < C; ++c)
      if (lane + 64 * c == e) {
        mine = v[c];
        key[c] = 0;
      }
    w[r] = __shfl(mine, e & 63, 64);
    total += w[r];
  }
  if (lane == 0) {
#pragma unroll
    for (int r = 0; r < kMaxTop; ++r) {
      if (r >= k) break;
      weights[t * k + r] = w[r] / total;
      experts[t * k + r] = idx[r];
    }
  }
}

// Stable counting sort of n expert ids by one workgroup: a histogram in LDS, its exclusive sum
// (the segment offsets), then tiles of 1024 entries in order; an entry's place is its expert's
// running base, plus the entries of the same expert in the tile's earlier wavefronts, plus those
// in earlier lanes of its own (a ballot a bit of the id). Ids outside [0, E) belong to no
// segment: their place is -1, the unused rows of the order read -1, and *bad tells (2 for a
// negative one, else 1).
__global__ __launch_bounds__(1024) void route_sort_kernel(const int64_t* __restrict__ experts, int n, int k, int E,
                                                          int bits, int32_t* __restrict__ token_of_slot,
                                                          int32_t* __restrict__ seg_off, int64_t* __restrict__ pos,
                                                          int32_t* __restrict__ bad) {
  __shared__ int base[kMaxExperts + 1], wcnt[16][kMaxExperts];
  __shared__ int wrong;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (tid <= E) base[tid] = 0;
  if (tid == 0) wrong = 0;
  __syncthreads();
  for (int i = tid; i < n; i += 1024) {
    const int64_t e = experts[i];
    if (e >= 0 && e < E) atomicAdd(&base[e], 1);
    else atomicMax(&wrong, e < 0 ? 2 : 1);
  }
  __syncthreads();
  if (tid == 0) {  // E is small: one thread's exclusive sum
    int sum = 0;
    for (int e = 0; e < E; ++e) {
      const int c = base[e];
      base[e] = sum;
      sum += c;
    }
    base[E] = sum;
    *bad = wrong;
  }
  __syncthreads();
  if (tid <= E) seg_off[tid] = base[tid];
  for (int i = base[E] + tid; i < n; i += 1024) token_of_slot[i] = -1;
  __syncthreads();
  for (int i0 = 0; i0 < n; i0 += 1024) {
    const int i = i0 + tid;
    int e = -1;
    if (i < n) {
      const int64_t v = experts[i];
      if (v >= 0 && v < E) e = (int)v;
    }
    for (int j = tid; j < 16 * E; j += 1024) wcnt[j / E][j % E] = 0;
    __syncthreads();
    uint64_t same = __ballot(e >= 0);
    for (int b = 0; b < bits; ++b) {
      const uint64_t ones = __ballot(e >= 0 && (e >> b & 1));
      same &= (e >> b & 1) ? ones : ~ones;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1));
    if (e >= 0 && rank == 0) wcnt[wave][e] = __popcll(same);
    __syncthreads();
    if (e >= 0) {
      int p = base[e] + rank;
      for (int w = 0; w < wave; ++w) p += wcnt[w][e];
      token_of_slot[p] = i / k;
      pos[i] = p;
    } else if (i < n) {
      pos[i] = -1;
    }
    __syncthreads();
    if (tid < E) {
      int c = 0;
      for (int w = 0; w < 16; ++w) c += wcnt[w][tid];
      base[tid] += c;
    }
    __syncthreads();
  }
}

}  // namespace

}  // namespace mls

using namespace mls;

extern "C" int mlsx_route_topk(const void* logits, int dt, int64_t ld, int64_t tokens, int E, int k, float* weights,
                               int64_t* experts, mls_stream_t stream) {
  const char* fn = "mlsx_route_topk";
  if (tokens < 0 || E < 1 || k < 1 || k > E || ld < E) return fail(MLS_ERR_ARG, "%s: bad sizes", fn);
  if (!is_float_dt(dt)) return fail(MLS_ERR_ARG, "%s: bad dtype %d", fn, dt);
  if (E > kMaxExperts || k > kMaxTop || tokens > 0x3FFFFFFF)
    return fail(MLS_ERR_UNSUPPORTED, "%s: at most %d experts and top-%d", fn, kMaxExperts, kMaxTop);
  if (tokens == 0) return MLS_OK;
  if (!logits || !weights || !experts) return fail(MLS_ERR_ARG, "%s: null pointer", fn);
  const dim3 grid((unsigned)cdiv(tokens, 4));
  hipStream_t st = (hipStream_t)stream;
  if (dt == MLS_F32)
    hipLaunchKernelGGL(route_topk_kernel<float>, grid, dim3(256), 0, st, (const float*)logits, ld, tokens, E, k, weights, experts);
  else if (dt == MLS_F16)
    hipLaunchKernelGGL(route_topk_kernel<_Float16>, grid, dim3(256), 0, st, (const _Float16*)logits, ld, tokens, E, k, weights, experts);
  else
    hipLaunchKernelGGL(route_topk_kernel<__bf16>, grid, dim3(256), 0, st, (const __bf16*)logits, ld, tokens, E, k, weights, experts);
  return check_launch(fn);
}

extern "C" int mlsx_route_sort(const int64_t* experts, int64_t n, int k, int E, int32_t* token_of_slot,
                               int32_t* seg_off, int64_t* pos, int32_t* bad, mls_stream_t stream) {
  const char* fn = "mlsx_route_sort";
  if (n < 1 || k < 1 || E < 1) return fail(MLS_ERR_ARG, "%s: bad sizes", fn);
  if (E > kMaxExperts || n > MLSX_ROUTE_MAX) return fail(MLS_ERR_UNSUPPORTED, "%s: too large", fn);
  if (!experts || !token_of_slot || !seg_off || !pos || !bad) return fail(MLS_ERR_ARG, "%s: null pointer", fn);
  int bits = 0;
  while ((1 << bits) < E) ++bits;
  hipLaunchKernelGGL(route_sort_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, experts, (int)n, k, E, bits,
                     token_of_slot, seg_off, pos, bad);
  return check_launch(fn);
}
