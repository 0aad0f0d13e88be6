// Matrix-core matmul on 16 x 16 tiles, Q4_K / Q6_K / Q8_0 (operands: mxa_tiles.hpp): the block-split batched
// decode for shapes that the streaming kernels do not take, its grouped MoE form, and the choice of kernel
// for up to 16 activation rows (more: mxa_ptile.hip). The blocks are folded in order 0..nb-1, so the outputs
// equal the oracle and the decode kernels bit for bit.
#include <math.h>

#include "mxa_kernels.hpp"
#include "mxa_tiles.hpp"

#pragma clang fp contract(off)

namespace mxa {
namespace {

// Batched decode (M <= 16): 32 weight rows per workgroup and the blocks of each chunk split over
// the 4 waves (wave w takes blocks w and w + 4 of an 8-block chunk, for both 16-row tiles), so that
// N = 4096..14336 still gives the GPU 128..448 workgroups. The block values go through LDS and are
// folded in block order by the thread that owns the output.
constexpr int kDecCh = 8;                     // blocks per chunk
constexpr int kDecQStride = kDecCh * QK + 16;
constexpr int kDecBStride = kDecCh * 16 + 8;

// kDecRT 16-row weight tiles per group: 2, or 1 for Q6_K (its per-lane block bytes need twice
// the registers; one tile keeps two waves per SIMD). The body of one workgroup: groups
// wg * kGroups .. + kGroups - 1 of n_wg * kGroups (16 kDecRT rows each) against M <= 16
// activation rows. A chunk's activations are staged once for all of the workgroup's groups (at
// 16 activation rows they weigh as much as 32 weight rows of the chunk), and each (chunk, group)
// step loads the next step's weights while it computes.
template <int TYPE, int kDecRT, int kGroups = 1>
__device__ __forceinline__ void mdec_rows(const uint8_t* w, long long row_bytes, const Act& act,
                                          YOut y, long long ldy, int M, int N, int wg,
                                          int n_wg) {
  using Tile = typename TileOf<TYPE>::T;
  using W = typename Tile::W;
  __shared__ __align__(16) int8_t Aq[16 * kDecQStride];
  __shared__ __align__(16) _Float16 Ab[16 * kDecBStride];
  __shared__ float Ad[kDecCh * 16];
  __shared__ float Tp[kDecRT][kDecCh][16][16];  // block values [tile][block][m][n]
  __shared__ float Dp[kDecRT][kDecCh][16];      // the block's weight scale where the fold uses one

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int ln = lane & 15, g = lane >> 4;
  const int n0 = xcd_tile(wg, n_wg) * 16 * kDecRT * kGroups;
  auto row_of = [&](int grp, int t) {
    return w + (size_t)min(n0 + 16 * (kDecRT * grp + t) + ln, N - 1) * row_bytes;
  };
  const int nb = act.nb;
  constexpr int kOut = kDecRT * 256 / 256;  // outputs per thread and group: kDecRT x 16 x 16 / 256
  float acc[kGroups][kOut];
#pragma unroll
  for (int grp = 0; grp < kGroups; ++grp)
#pragma unroll
    for (int k = 0; k < kOut; ++k) acc[grp][k] = 0.0f;

  // this wave's blocks wave and wave + 4 of chunk c0 for group grp (blocks past the chunk repeat
  // its last one: their values are never folded)
  auto load_step = [&](W (&dst)[2][kDecRT], int c0, int grp) {
    const int cn = min(kDecCh, nb - c0);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < kDecRT; ++t) dst[i][t] = Tile::load(row_of(grp, t), c0 + min(wave + 4 * i, cn - 1), g);
  };
  W cur[2][kDecRT], nxt[2][kDecRT];
  load_step(cur, 0, 0);
  for (int c0 = 0; c0 < nb; c0 += kDecCh) {
    const int cn = min(kDecCh, nb - c0);
    // 1. the chunk's activations into LDS (rows >= M repeat row M - 1, blocks >= cn repeat the
    //    chunk's last block: those values are never folded or stored)
    for (int p = tid; p < 16 * kDecCh * 16; p += 256) {
      const int r = p / (kDecCh * 16), o = p - r * (kDecCh * 16), bb = min(o >> 4, cn - 1), pc = o & 15;
      *(u32x4a4*)(Aq + r * kDecQStride + (o >> 4) * QK + 16 * pc) =
          ld16((const uint8_t*)(act.q + (size_t)min(r, M - 1) * act.k + (size_t)(c0 + bb) * QK) + 16 * pc);
    }
    {
      const int r = tid >> 4, o = tid & 15, bb = min(o >> 1, cn - 1), hf = o & 1;
      const u32x4a4 v = ld16((const uint8_t*)(act.bsums + ((size_t)min(r, M - 1) * nb + c0 + bb) * 16) + 16 * hf);
      const uint32_t wv[4] = {v.x, v.y, v.z, v.w};
      f16x8 hv;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        hv[2 * i] = (_Float16)(float)(int16_t)(wv[i] & 0xFFFFu);
        hv[2 * i + 1] = (_Float16)(float)(int16_t)(wv[i] >> 16);
      }
      *(f16x8*)(Ab + r * kDecBStride + (o >> 1) * 16 + 8 * hf) = hv;
    }
    if (tid < kDecCh * 16) {
      const int bb = tid >> 4, r = tid & 15;
      Ad[tid] = act.d[(size_t)min(r, M - 1) * nb + c0 + min(bb, cn - 1)];
    }
    const ActTile A{Aq, Ab, kDecQStride, kDecBStride};
#pragma unroll
    for (int grp = 0; grp < kGroups; ++grp) {
      // 2. the next step's weights: the next group of this chunk, or the first of the next chunk
      const bool more = grp + 1 < kGroups || c0 + kDecCh < nb;
      if (more) load_step(nxt, grp + 1 < kGroups ? c0 : c0 + kDecCh, grp + 1 < kGroups ? grp + 1 : 0);
      __syncthreads();  // the chunk is in LDS; the previous step's fold has read Tp
      // 3. this wave's blocks, every tile of the group: values into LDS
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int bb = wave + 4 * i;
        if (bb < cn) {
          const typename Tile::F f = Tile::frag(A, bb, 0, ln, g);
#pragma unroll
          for (int t = 0; t < kDecRT; ++t) {
            const typename Tile::P pp = Tile::prep(cur[i][t], g);
            Tile::value(pp, f, g, [&](int e, float v, float dd) {
              Tp[t][bb][4 * g + e][ln] = v;
              if (g == 0 && e == 0) Dp[t][bb][ln] = dd;
            });
          }
        }
      }
      __syncthreads();
      // 4. fold the chunk's blocks in order: thread -> outputs (tile, m, n) of the group
#pragma unroll
      for (int k = 0; k < kOut; ++k) {
        const int idx = tid + 256 * k, t = idx >> 8, m = (idx >> 4) & 15, n = idx & 15;
        for (int bb = 0; bb < cn; ++bb)
          acc[grp][k] = Tile::fold(acc[grp][k], Ad[bb * 16 + m], Tp[t][bb][m][n], Dp[t][bb][n]);
      }
      if (more) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int t = 0; t < kDecRT; ++t) cur[i][t] = nxt[i][t];
      }
    }
    __syncthreads();  // every fold has read Ad and Tp before the next chunk is staged
  }
#pragma unroll
  for (int grp = 0; grp < kGroups; ++grp)
#pragma unroll
    for (int k = 0; k < kOut; ++k) {
      const int idx = tid + 256 * k, t = idx >> 8, m = (idx >> 4) & 15;
      const int n = n0 + 16 * (kDecRT * grp + t) + (idx & 15);
      if (m < M && n < N) y.put((size_t)m * ldy + n, acc[grp][k]);
    }
}

template <int TYPE, int kDecRT>
__global__ __launch_bounds__(256) void mdec_kernel(const uint8_t* w, long long row_bytes, Act act,
                                                   YOut y, long long ldy, int M, int N) {
  mdec_rows<TYPE, kDecRT>(w, row_bytes, act, y, ldy, M, N, blockIdx.x, gridDim.x);
}

// Grouped MoE projection: expert e = blockIdx.y multiplies its rows [offsets[e], offsets[e + 1])
// of the Q8_K activations by its packed weight (w + e * expert_stride); the outputs go to the same
// rows of y. The expert's rows are taken 16 at a time, chunk z by the workgroups of blockIdx.z ==
// z mod gridDim.z, so every row is computed whatever the grid's depth (the host sizes it from a
// bound it knows without a sync; an expert with more rows loops). A workgroup whose expert has no
// row in its chunks exits. The offsets come from the device, so they are clamped to
// [0, total_rows): a bad table gives wrong rows, never an access outside the activations or y.
// Two waves per SIMD asked of the compiler: the chunk loop left to itself took Q6_K to 272 VGPRs
// (one workgroup per CU instead of two; the down projection ran 1.5x longer), with the bound it
// fits 206 VGPRs with no scratch (Q8_0 227, Q4_K 202).
template <int TYPE, int kDecRT, int kGroups>
__global__ __launch_bounds__(256, 2) void moe_dec_kernel(const uint8_t* w, long long row_bytes,
                                                      long long expert_stride, Act act,
                                                      const int32_t* __restrict__ offsets,
                                                      int total_rows, YOut y,
                                                      long long ldy, int N) {
  const int e = blockIdx.y;
  const int begin = min(max(offsets[e], 0), total_rows);
  const int end = min(max(offsets[e + 1], begin), total_rows);
  for (int p0 = begin + 16 * (int)blockIdx.z; p0 < end; p0 += 16 * (int)gridDim.z) {
    const int M = min(16, end - p0);  // uniform over the workgroup
    Act a = act;
    a.q = act.q + (size_t)p0 * act.k;
    a.d = act.d + (size_t)p0 * act.nb;
    a.bsums = act.bsums + (size_t)p0 * act.nb * 16;
    mdec_rows<TYPE, kDecRT, kGroups>(w + (size_t)e * expert_stride, row_bytes, a, y.at((size_t)p0 * ldy),
                                     ldy, M, N, blockIdx.x, gridDim.x);
    __syncthreads();  // the next chunk rewrites the LDS tiles this one read
  }
}

template <int TYPE>
int launch_mt_type(const uint8_t* w, long long row_bytes, const Act& act, YOut y, long long ldy,
                   int M, int N, hipStream_t stream) {
  // M <= 16: the per-wave streaming kernel where its slots fit LDS (measured on MI355X at M = 16,
  // the same bits: Q4_K 4096 x 4096 5.7 vs 7.1 us, 1024 x 4096 5.4 vs 6.3, Q8_0 4096 x 4096 7.1 vs
  // 8.4; Q4_K 14336 x 4096 12.1 vs 12.0-12.3), then the copy-wave kernels
  if (M <= 16 && launch_bwave(TYPE, w, row_bytes, act, y, ldy, M, N, stream) == 0) return 0;
  if (M <= 16 && launch_bflow(TYPE, w, row_bytes, act, y, ldy, M, N, stream) == 0) return 0;
  if (M <= 16 && launch_bres(TYPE, w, row_bytes, act, y, ldy, M, N, stream) == 0) return 0;
  if (M <= 16 && launch_bstream(TYPE, w, row_bytes, act, y, ldy, M, N, stream) == 0) return 0;
  if (M <= 16 && N < 512 * 64) {  // enough rows to fill the chip take the prefill tiles
    constexpr int RT = TYPE == T_Q6_K ? 1 : 2;
    const int tiles = (N + 16 * RT - 1) / (16 * RT);
    hipLaunchKernelGGL((mdec_kernel<TYPE, RT>), dim3(tiles), dim3(256), 0, stream, w, row_bytes, act, y, ldy, M, N);
    return 0;
  }
  return launch_ptile(TYPE, w, row_bytes, act, y, ldy, M, N, stream);
}

// Tile groups per workgroup of moe_dec_kernel (each group's chunk of activations staged once for all of
// them): the most of 4, 2, 1 that still gives two workgroups per CU (Q8_0 at most 2: four spill).
// Measured on MI355X, eager forward of 8 experts top 2 (4096 x 14336; Q4_K gate / up, Q6_K down), the same
// bits: 16 tokens 498 vs 523 us, 128 tokens 1146 vs 1364; with four groups forced, 40 small experts at 16
// tokens lost (214 vs 204 us) to the smaller grid.
int moe_dec_groups(int type, int tiles, int n_experts, int chunks) {
  for (int gs = type == T_Q8_0 ? 2 : 4; gs > 1; gs >>= 1)
    if ((long long)((tiles + gs - 1) / gs) * n_experts * chunks >= 2LL * cu_count()) return gs;
  return 1;
}
int moe_dec_tiles(int type, int n_rows) { return type == T_Q6_K ? (n_rows + 15) / 16 : (n_rows + 31) / 32; }

// Estimated times in us of the three forms of a grouped projection with a few rows an expert, kernel alone,
// weights from HBM:
// - body: the batched-decode bodies (16-row chunks). Every CU has its share of the weight rows that can be in
//   use, and walks it 16 rows at a time, parts of 8 blocks of long rows one after another; and there are the
//   workgroups of experts without rows;
// - ptile: the prefill tiles (32-row chunks). A workgroup of 128 weight rows walks the blocks;
// - tile: the decode tile below, 8 blocks a step.
// A start, the steps that a workgroup takes in a row, and for the last two what the other workgroups of its CU
// cost. The constants are fitted on MI355X to 2800 calls of two tokens or more (512 to 14336 rows, 2 to 56
// blocks, 4 to 128 experts, random routings of up to 20 rows an expert); half of the estimates are within 6%,
// the choice that they give is within 0.5% of the best of the three on average, where a rule on the number of
// prefill tiles and of rows an expert lost 4%. Some of it, us, prefill tiles / decode bodies: 8 experts
// top 2, Q4_K 14336 x 4096, 3 / 4 / 6 tokens 47 / 53, 53 / 62, 62 / 63, 36 / 40 / 48 tokens (9 / 10 / 12 rows
// an expert: from 9 on some expert has a second chunk of 16) 74 / 67, 73 / 75, 73 / 84; Q6_K 4096 x 14336, 4 /
// 36 / 48 tokens 139 / 135, 140 / 142, 141 / 230; 16 experts top 4, Q6_K 3072 x 2048, 3 / 4 / 5 / 7 / 40 tokens
// 27 / 31, 32 / 34, 38 / 34, 39 / 34, 39 / 34; Q8_0 2048 x 3072, 4 / 7 / 40 tokens 29 / 24, 31 / 24, 33 / 25; 64
// experts top 8, Q4_K 1024 x 2048, 4 / 5 / 16 tokens 16 / 16, 17 / 22, 23 / 32. Prefill tiles / decode tile: Q6_K
// 2048 x 1024, 64 experts top 8, 2 / 4 / 16 tokens 16 / 25, 23 / 42, 39 / 84; 2048 x 7168, 4 experts, 4 / 16 rows
// 71 / 33, 71 / 34; Q4_K 512 x 1536, 64 experts, 8 / 16 rows 12.2 / 11.9, 12.7 / 16.9.
struct MoeTimes {
  double body, ptile, tile;
};
MoeTimes moe_times(int type, int n_rows, int nb, int n_experts, int total_rows, int max_rows) {
  struct Fit {
    double b0, b1, b2, b3, b4, p0, p1, p2, p3, t0, t1, t2, t3, t4;
  };
  static constexpr Fit kQ4 = {3.77, 1.492, 0.044, 0.92, 0.003, 5.84, 1.169, 0.977, 0.218, 4.84, 2.163, 0.739, -0.14, 0.282};
  static constexpr Fit kQ6 = {5.31, 1.821, 0.065, 1.04, 0.004, 6.59, 2.219, 1.714, 0.169, 4.61, 3.439, 0.536, -0.36, 0.377};
  static constexpr Fit kQ8 = {4.02, 0.983, 0.133, 1.04, 0.004, 6.54, 1.744, 1.515, 0.209, 3.61, 7.086, 0.708, -0.21, 0.552};
  const Fit& f = type == T_Q4_K ? kQ4 : type == T_Q6_K ? kQ6 : kQ8;
  const double cus = cu_count(), most = min(n_experts, total_rows), rows = (double)total_rows / n_experts;
  // experts with rows: as many as max_rows tokens name that choose total_rows / max_rows experts each at random
  const double choices = (double)total_rows / max_rows;
  const double named = n_experts * (1 - pow(1 - fmin(1, choices / n_experts), max_rows));
  const double busy = fmin(most, fmax(named, fmax(1, choices)));
  const double second = fmin(1, fmax(0, (rows - 8.5) / 5));  // some expert's second chunk of 16 rows
  MoeTimes t;
  const double share = ceil(n_rows * most / cus);
  const int parts = nb <= 16 ? 1 : (nb + 7) / 8;
  t.body = f.b0 + ceil(share / 16) * parts * (f.b1 + f.b2 * min(nb, parts > 1 ? 8 : 16)) * (1 + f.b3 * second) +
           f.b4 * ceil(n_rows / share) * (n_experts + (total_rows + 15) / 16);
  const double xp = (n_rows + 127) / 128 * busy / cus;  // workgroups per CU
  t.ptile = f.p0 + nb * (f.p1 + f.p2 * fmax(0, ceil(xp - 0.02) - 1) + f.p3 * fmin(1, xp));
  const int tiles = moe_dec_tiles(type, n_rows);
  const int gs = moe_dec_groups(type, tiles, n_experts, (max_rows + 15) / 16);
  const double xt = (tiles + gs - 1) / gs * busy * (1 + 0.5 * second) / cus;
  t.tile = f.t0 + gs * ((nb + 7) / 8 * f.t1 + nb * f.t4) * (1 + f.t2 * fmax(0, ceil(xt - 0.02) - 1) + f.t3 * fmin(1, xt));
  return t;
}

}  // namespace

bool mtile_supported(int type) { return type == T_Q4_K || type == T_Q6_K || type == T_Q8_0; }

int launch_moe_dec(int type, const uint8_t* w, long long row_bytes, long long expert_stride,
                   int n_experts, const Act& act, const int32_t* offsets, int total_rows,
                   int max_rows, YOut y, long long ldy, int n_rows, hipStream_t stream) {
  if (act.q == nullptr || n_experts < 1 || n_experts > 65535 || max_rows < 1 || n_rows < 1 ||
      total_rows < 1)
    return -1;
  const int chunks = (max_rows + 15) / 16;
  if (chunks > 65535) return -1;
  // The form that should take least time while the experts have few rows (20 on average), the prefill tiles
  // past that.
  const MoeTimes est = moe_times(type, n_rows, act.nb, n_experts, total_rows, max_rows);
  const bool decode = total_rows <= 20LL * n_experts;
  constexpr int kMoeDecodeBodyMaxRows = 96, kMoeDecodeBodyMinN = 1024;
  if (decode && est.body <= fmin(est.ptile, est.tile) && max_rows <= kMoeDecodeBodyMaxRows &&
      n_rows >= kMoeDecodeBodyMinN &&
      launch_moe_bwave(type, w, row_bytes, expert_stride, n_experts, act, offsets, total_rows, y,
                       ldy, n_rows, stream) == 0)
    return 0;
  if ((!decode || est.ptile <= est.tile) &&
      launch_moe_ptile(type, w, row_bytes, expert_stride, n_experts, act, offsets, total_rows, y, ldy, n_rows,
                       stream) == 0)
    return 0;
  auto go = [&](auto k1, auto k2, auto k4, int rt) {
    const int t1 = (n_rows + 16 * rt - 1) / (16 * rt), gs = moe_dec_groups(type, t1, n_experts, chunks);
    const dim3 grid((t1 + gs - 1) / gs, n_experts, chunks);
    if (gs == 4)
      hipLaunchKernelGGL(k4, grid, dim3(256), 0, stream, w, row_bytes, expert_stride, act, offsets,
                         total_rows, y, ldy, n_rows);
    else if (gs == 2)
      hipLaunchKernelGGL(k2, grid, dim3(256), 0, stream, w, row_bytes, expert_stride, act, offsets,
                         total_rows, y, ldy, n_rows);
    else
      hipLaunchKernelGGL(k1, grid, dim3(256), 0, stream, w, row_bytes, expert_stride, act, offsets,
                         total_rows, y, ldy, n_rows);
    return 0;
  };
  switch (type) {
    case T_Q4_K:
      return go(moe_dec_kernel<T_Q4_K, 2, 1>, moe_dec_kernel<T_Q4_K, 2, 2>,
                moe_dec_kernel<T_Q4_K, 2, 4>, 2);
    case T_Q8_0:  // k4 is never taken (at most two groups): the two-group form stands in
      return go(moe_dec_kernel<T_Q8_0, 2, 1>, moe_dec_kernel<T_Q8_0, 2, 2>,
                moe_dec_kernel<T_Q8_0, 2, 2>, 2);
    case T_Q6_K:
      return go(moe_dec_kernel<T_Q6_K, 1, 1>, moe_dec_kernel<T_Q6_K, 1, 2>,
                moe_dec_kernel<T_Q6_K, 1, 4>, 1);
    default: return -1;
  }
}

int launch_mtile(int type, const uint8_t* w, long long row_bytes, const Act& act, YOut y,
                 long long ldy, int m_rows, int n_rows, hipStream_t stream) {
  if (act.q == nullptr || m_rows < 1) return -1;
  switch (type) {
    case T_Q4_K: return launch_mt_type<T_Q4_K>(w, row_bytes, act, y, ldy, m_rows, n_rows, stream);
    case T_Q6_K: return launch_mt_type<T_Q6_K>(w, row_bytes, act, y, ldy, m_rows, n_rows, stream);
    case T_Q8_0: return launch_mt_type<T_Q8_0>(w, row_bytes, act, y, ldy, m_rows, n_rows, stream);
    default: return -1;
  }
}

}  // namespace mxa
