// Weighted combine of routed expert outputs (MoE), one launch: for token t, the down-projection
// rows of its top_k (token, slot) pairs times the routing weights, summed in ascending expert id
// (pairs of equal id in slot order) from a float zero, as the reference's loop over the sorted
// expert ids adds them with `index_add_` (app/architectures/moe_experts.py:81-88), with the
// module's casts: the projection output rounded to bfloat16 first when the layer computes in
// bfloat16 (`down.to(dtype)`), the product with the float32 weight rounded to float32, each sum
// rounded to float32. One thread per output element; the pair order is ranked once per workgroup.
#include "mxa_kernels.hpp"

#pragma clang fp contract(off)

namespace mxa {
namespace {

// float32 -> bfloat16 -> float32 with round-to-nearest-even, NaN to the quiet NaN 0x7FC0 (the
// conversion torch's `.to(torch.bfloat16)` performs)
__device__ __forceinline__ float round_bf16(float f) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7FFFFFFFu) > 0x7F800000u) return __uint_as_float(0x7FC00000u);
  return __uint_as_float((u + 0x7FFFu + ((u >> 16) & 1u)) & 0xFFFF0000u);
}

__global__ __launch_bounds__(256) void moe_combine_kernel(
    const float* __restrict__ down, const int32_t* __restrict__ rows,
    const int32_t* __restrict__ ids, const float* __restrict__ wts, int top_k, int n_embd,
    int bf16, float* __restrict__ out) {
  __shared__ int ord[kMoeMaxTopK];
  const int t = blockIdx.y, j = blockIdx.x * 256 + threadIdx.x;
  const int32_t* tid = ids + (size_t)t * top_k;
  if ((int)threadIdx.x < top_k) {  // slot k's place in the token's sorted order
    const int k = threadIdx.x, e = tid[k];
    int rank = 0;
    for (int k2 = 0; k2 < top_k; ++k2) rank += (tid[k2] < e) || (tid[k2] == e && k2 < k);
    ord[rank] = k;
  }
  __syncthreads();
  if (j >= n_embd) return;
  float acc = 0.0f;
  for (int i = 0; i < top_k; ++i) {
    const size_t p = (size_t)t * top_k + ord[i];
    const size_t r = rows != nullptr ? (size_t)rows[p] : p;
    float v = down[r * n_embd + j];
    if (bf16) v = round_bf16(v);
    acc = acc + v * wts[p];
  }
  out[(size_t)t * n_embd + j] = acc;
}

// Routing of the (token, slot) pairs by expert, one workgroup: a stable counting sort. Pair
// p = t * top_k + k has expert e = ids[p] clamped into [0, n_experts); its place in the sorted
// order is the pairs of smaller experts plus the earlier pairs of the same expert, which is where
// a stable argsort of the flattened ids puts it (the order the reference's per-expert loop visits
// tokens: moe_experts.py:81-88, tokens ascending within an expert). Every wave owns a contiguous run of
// pairs and its own counters, 64 pairs a step: the lanes of one expert find each other with a ballot
// per bit of the expert id, and the first of them updates the counter. One pass counts; the counts are
// prefixed over waves and experts; a second pass places.
//
// Bound: latency, of a step's ballots and counter and of the ids' loads (four steps requested at a time);
// the runs need no barrier. Measured on MI355X, kernel alone, 4096 pairs of 64 experts: 7.8 us; a ballot
// per distinct expert of a wave, in chunks of 1024 pairs between barriers, took 26.5.
constexpr int kRouteWaves = 16;
__global__ __launch_bounds__(64 * kRouteWaves) void moe_route_kernel(
    const void* __restrict__ ids, int ids64, int n_pairs, int top_k, int n_experts,
    int32_t* __restrict__ offsets, int32_t* __restrict__ pair_tok, int32_t* __restrict__ rows,
    int32_t* __restrict__ ids32) {
  __shared__ int cnt[kRouteWaves][kMoeRouteMaxExperts];
  __shared__ int part[kMoeRouteMaxExperts / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bits = n_experts > 1 ? 32 - __builtin_clz(n_experts - 1) : 0;
  const int run = (n_pairs + 64 * kRouteWaves - 1) / (64 * kRouteWaves) * 64;
  const int begin = wave * run, end = min(begin + run, n_pairs);
  const uint64_t below = (1ull << lane) - 1ull;
  // step(p, valid, v, e, m) for every 64 pairs of the run: m, the lanes of this lane's expert
  auto walk = [&](auto&& step) {
    for (int c0 = begin; c0 < end; c0 += 256) {
      long long v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int p = min(c0 + 64 * j + lane, n_pairs - 1);
        v[j] = ids64 ? ((const long long*)ids)[p] : (long long)((const int32_t*)ids)[p];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (c0 + 64 * j >= end) break;
        const int p = c0 + 64 * j + lane;
        const bool valid = p < end;
        const int e = v[j] < 0 ? 0 : v[j] >= n_experts ? n_experts - 1 : (int)v[j];
        uint64_t m = __ballot(valid);
        for (int b = 0; b < bits; ++b) {
          const bool one = (e >> b) & 1;
          const uint64_t ones = __ballot(one);
          m &= one ? ones : ~ones;
        }
        step(p, valid, v[j], e, m);
        wave_sync();  // the next step reads the counters that this one wrote
      }
    }
  };
#pragma unroll
  for (int i = 0; i < kMoeRouteMaxExperts / 64; ++i) cnt[wave][64 * i + lane] = 0;
  wave_sync();
  walk([&](int p, bool valid, long long v, int e, uint64_t m) {
    if (!valid) return;
    if ((m & below) == 0) cnt[wave][e] += __popcll(m);
    if (ids32 != nullptr) ids32[p] = (int32_t)v;  // torch's int64 -> int32 conversion
  });
  __syncthreads();
  // thread e: the waves' counts of expert e, prefixed; the experts' totals scanned over a wave, then waves
  int before[kRouteWaves], total = 0, incl = 0;
  if (tid < kMoeRouteMaxExperts) {
#pragma unroll
    for (int w = 0; w < kRouteWaves; ++w) before[w] = cnt[w][tid];
#pragma unroll
    for (int w = 0; w < kRouteWaves; ++w) {
      const int c = before[w];
      before[w] = total;
      total += c;
    }
    incl = total;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int x = __shfl_up(incl, off, 64);
      if (lane >= off) incl += x;
    }
    if (lane == 63) part[wave] = incl;
  }
  __syncthreads();
  if (tid < kMoeRouteMaxExperts) {
    int base = incl - total;
    for (int w = 0; w < wave; ++w) base += part[w];
    if (tid < n_experts) offsets[tid] = base;
#pragma unroll
    for (int w = 0; w < kRouteWaves; ++w) cnt[w][tid] = before[w] + base;
  }
  if (tid == 0) offsets[n_experts] = n_pairs;
  __syncthreads();
  walk([&](int p, bool valid, long long, int e, uint64_t m) {
    const int first = cnt[wave][e], place = first + __popcll(m & below);
    if (valid) {
      rows[p] = place;
      pair_tok[place] = p / top_k;
    }
    wave_sync();  // every lane has read its counter
    if (valid && (m & below) == 0) cnt[wave][e] = first + __popcll(m);
  });
}

}  // namespace

int launch_moe_route(const void* ids, bool ids64, int n_tokens, int top_k, int n_experts,
                     int32_t* offsets, int32_t* pair_tok, int32_t* rows, int32_t* ids32,
                     hipStream_t stream) {
  if (ids == nullptr || offsets == nullptr || pair_tok == nullptr || rows == nullptr ||
      n_tokens < 1 || top_k < 1 || n_experts < 1 || n_experts > kMoeRouteMaxExperts ||
      (long long)n_tokens * top_k > kMoeRouteMaxPairs)
    return -1;
  hipLaunchKernelGGL(moe_route_kernel, dim3(1), dim3(64 * kRouteWaves), 0, stream, ids,
                     ids64 ? 1 : 0, n_tokens * top_k, top_k, n_experts, offsets, pair_tok, rows,
                     ids32);
  return 0;
}

int launch_moe_combine(const float* down, const int32_t* rows, const int32_t* ids,
                       const float* weights, int n_tokens, int top_k, int n_embd, int bf16,
                       float* out, hipStream_t stream) {
  if (n_tokens < 1 || n_tokens > 65535 || top_k < 1 || top_k > kMoeMaxTopK || n_embd < 1)
    return -1;
  hipLaunchKernelGGL(moe_combine_kernel, dim3((n_embd + 255) / 256, n_tokens), dim3(256), 0,
                     stream, down, rows, ids, weights, top_k, n_embd, bf16, out);
  return 0;
}

}  // namespace mxa
