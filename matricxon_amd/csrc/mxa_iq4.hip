// IQ4_XS prefill (M > 16) on the matrix cores.
//
// The reference multiplies fp32 activations by dl * K[q] (app/native/src/mx_dot_f32.c:32-58, K the
// IQ4_NL grid, dl = d * (ls - 32) per 32-value sub-block). Here x is first split into two bf16
// parts, x = hi + lo (hi = x rounded to bf16, lo = the rest rounded to bf16; relative error of the
// pair about 2^-17), written to the workspace by split_bf16_kernel. The grid values are small
// integers, exact in bf16, so bf16 MFMAs on (hi, K) and (lo, K) give sum(K * x) of one sub-block.
// The sub-block scale dl is applied in fp32 after them. The result
// meets the float tolerance against the reference (rel-L2 <= 1e-4); its summation order differs from the
// decode kernels', which is why batches of up to 16 rows stay on those.
#include "mxa_kernels.hpp"
#include "mxa_pcopy.hpp"

#pragma clang fp contract(off)

namespace mxa {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));  // 16-byte aligned

typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr f32x16 kZero16 = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

// bf16 bits of x rounded to nearest even (NaN stays NaN, overflow gives +-Inf).
__device__ __forceinline__ uint32_t bf16_rne(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

__global__ __launch_bounds__(256) void split_bf16_kernel(const float* __restrict__ x,
                                                         uint16_t* __restrict__ hi,
                                                         uint16_t* __restrict__ lo, long long n4) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n4) return;
  const float4 v = ((const float4*)x)[i];
  const float e[4] = {v.x, v.y, v.z, v.w};
  uint32_t h[4], l[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    h[k] = bf16_rne(e[k]);
    const float rest = e[k] - __builtin_bit_cast(float, h[k] << 16);  // exact in fp32
    l[k] = bf16_rne(rest);
  }
  ((uint2*)hi)[i] = uint2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
  ((uint2*)lo)[i] = uint2{l[0] | (l[1] << 16), l[2] | (l[3] << 16)};
}

// Eight bf16 grid values (as four dwords) for the eight 4-bit indices in the low nibbles of the
// bytes of (a, b).
__device__ __forceinline__ u32x4a4 grid_bf16x8(uint32_t a, uint32_t b) {
  const uint32_t ka = iq4_lookup4(a), kb = iq4_lookup4(b);
  uint32_t f[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[i] = __builtin_bit_cast(uint32_t, (float)(int8_t)(uint8_t)(ka >> (8 * i)));
    f[4 + i] = __builtin_bit_cast(uint32_t, (float)(int8_t)(uint8_t)(kb >> (8 * i)));
  }
  // bf16 = the top half of an fp32 holding a small integer (exact); two per dword
  return u32x4a4{__builtin_amdgcn_perm(f[1], f[0], 0x07060302u), __builtin_amdgcn_perm(f[3], f[2], 0x07060302u),
                 __builtin_amdgcn_perm(f[5], f[4], 0x07060302u), __builtin_amdgcn_perm(f[7], f[6], 0x07060302u)};
}

// Tiling (as mxa_ptile.hip): a wave owns 32 weight rows x 32 MTW activation rows, a workgroup WN waves
// along the weight rows. v_mfma_f32_32x32x16_bf16 takes 16 of a sub-block's 32 values: lane (row, h)
// holds bytes 8 h .. 8 h + 7 of the sub-block's 16, whose low nibbles are elements 8 h .. of the first
// step's 16 and whose high nibbles are those of the second's, so both operands come in natural order.
// A sub-block is four MFMAs (two steps of hi, two of lo) into a sum of its own, scaled by dl in fp32.
// The activations of half a block (128 values: 256 bytes of hi, 256 of lo per row) go straight into one of
// two LDS buffers, piece c of row r at place c ^ (r & 15); a wave's weights into a slot that only it reads.
//
// Bound: latency at few waves. A sub-block of 32 rows costs about 50 VALU instructions to look its 512 values
// up as bf16, and 16 to scale and four MFMAs of 32 cycles per activation tile; at 4096 x 4096 M = 512 one wave
// stands on a SIMD, whose VALU issues in 43% of the cycles and whose matrix core is busy in 24%, with nothing
// to run in its waits. At M = 2048 two waves do.
// Measured on MI355X against 16 x 16 tiles whose eight waves read every operand from LDS (us per call with
// the split, the same bits): 4096 x 4096 M = 64 41 vs 83, M = 512 58 vs 87, M = 2048 180 vs 282 (382 TFLOP/s),
// 14336 x 4096 M = 2048 610 vs 944, 4096 x 14336 M = 128 131 vs 248.
struct PIQ4 {
  static constexpr int kBytes = 136, kShift = 8;  // blocks start at 8-byte multiples of the row
};

template <int WN, int MTW>
__global__ __launch_bounds__(64 * WN, 2) void iq4_ptile_kernel(const uint8_t* w, long long row_bytes,
                                                               const uint16_t* __restrict__ xh,
                                                               const uint16_t* __restrict__ xl, int K, YOut y,
                                                               long long ldy, int M, int N, int pieces) {
  constexpr int kRows = 32 * MTW, kBuf = 2 * kRows * 256;
  extern __shared__ __align__(16) uint8_t smem[];  // two activation buffers (hi rows, lo rows), the slots
  const int lane = threadIdx.x & 63;
  const int wave = (int)uniform(threadIdx.x >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int n0 = (xcd_tile(blockIdx.x, gridDim.x) * WN + wave) * 32, n = n0 + r, m0 = kRows * blockIdx.y;
  const int nb = K / QK;
  const PWeights<PIQ4> pw(w, row_bytes, n0, N, pieces, lane);
  const int slot = 2 * kBuf + wave * pslot_bytes(pieces);
  const uint32_t lds0 = lds_addr(smem), slot0 = lds0 + slot;

  // this wave's copies of half a block: 4 rows of hi or lo each (rows >= M repeat row M - 1)
  constexpr int kCopies = 2 * kRows / 4 / WN;
  static_assert(kCopies * 4 * WN == 2 * kRows, "whole copies per wave");
  const uint16_t* src[kCopies];
#pragma unroll
  for (int c = 0; c < kCopies; ++c) {
    const int row = 4 * (wave * kCopies + c) + (lane >> 4), rr = row & (kRows - 1);
    src[c] = (row < kRows ? xh : xl) + (size_t)min(m0 + rr, M - 1) * K + 8 * ((lane & 15) ^ (rr & 15));
  }
  auto copy_x = [&](int half, int buf) {
#pragma unroll
    for (int c = 0; c < kCopies; ++c)
      copy16_to_lds(src[c] + (size_t)half * 128, uniform(lds0 + buf * kBuf + (wave * kCopies + c) * 1024));
  };

  f32x16 acc[MTW];
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) acc[mt] = kZero16;
  copy_x(0, 0);
  pw.copy(0, slot0);
  wait_vmcnt(0);
  __syncthreads();
  for (int b = 0; b < nb; ++b) {
    u32x2a4 hdr, qs[8];
    {
      const uint8_t* p = smem + slot + pw.at(b, r);
      hdr = ld8(p);
#pragma unroll
      for (int t = 0; t < 8; ++t) qs[t] = ld8(p + 8 + 16 * t + 8 * h);
    }
    const float d = half_to_float(hdr.x);
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const bool more = half == 0 || b + 1 < nb;
      if (more) copy_x(2 * b + half + 1, half ^ 1);
      if (half == 0 && b + 1 < nb) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the weights are in registers
        __builtin_amdgcn_sched_barrier(0);
        pw.copy(b + 1, slot0);
      }
      const uint8_t* X = smem + half * kBuf;
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const int t = 4 * half + tt;
        const int ls = (int)(((hdr.y >> (4 * t)) & 15u) | (((hdr.x >> (16 + 2 * t)) & 3u) << 4));
        const float dl = d * (float)(ls - 32);
        const uint32_t q0 = qs[t].x, q1 = qs[t].y;
        const bf16x8 b0 = __builtin_bit_cast(bf16x8, grid_bf16x8(q0 & 0x0F0F0F0Fu, q1 & 0x0F0F0F0Fu));
        const bf16x8 b1 = __builtin_bit_cast(bf16x8, grid_bf16x8((q0 >> 4) & 0x0F0F0F0Fu, (q1 >> 4) & 0x0F0F0F0Fu));
#pragma unroll
        for (int mt = 0; mt < MTW; ++mt) {
          const uint8_t* xr = X + (32 * mt + r) * 256;
          auto a = [&](int part, int step) {
            return __builtin_bit_cast(bf16x8, *(const u32x4*)(xr + part * kRows * 256 +
                                                              16 * ((4 * tt + 2 * step + h) ^ (r & 15))));
          };
          f32x16 D = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a(0, 0), b0, kZero16, 0, 0, 0);
          D = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a(0, 1), b1, D, 0, 0, 0);
          D = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a(1, 0), b0, D, 0, 0, 0);
          D = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a(1, 1), b1, D, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 16; ++i) acc[mt][i] = fmaf(dl, D[i], acc[mt][i]);
        }
      }
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt) asm volatile("" : "+v"(acc[mt]));
      wait_vmcnt(0);    // this wave's pieces of the next half block are in LDS
      __syncthreads();  // everyone's are, and everyone is done with this one
    }
  }
  if (n < N) {
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int m = m0 + 32 * mt + 8 * (i >> 2) + 4 * h + (i & 3);
        if (m < M) y.put((size_t)m * ldy + n, acc[mt][i]);
      }
  }
}

}  // namespace

size_t iq4_prefill_workspace(int m_rows, int k) { return (size_t)m_rows * k * 2 * 2; }

int launch_iq4_prefill(const uint8_t* w, long long row_bytes, const float* x, void* workspace,
                       YOut y, long long ldy, int m_rows, int k, int n_rows, hipStream_t stream) {
  uint16_t* hi = (uint16_t*)workspace;
  uint16_t* lo = hi + (size_t)m_rows * k;
  const long long n4 = (long long)m_rows * k / 4;
  hipLaunchKernelGGL(split_bf16_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, stream, x, hi,
                     lo, n4);
  auto launch = [&](const uint8_t* w, YOut y, int n_rows) {
    const int pieces = ppieces<PIQ4>(((uintptr_t)w & 7) == 0);
    auto go = [&](auto kern, int wn, int mtw) {
      const int lds = 2 * 2 * 32 * mtw * 256 + wn * pslot_bytes(pieces);
      allow_lds((const void*)kern, lds);
      const dim3 grid((n_rows + 32 * wn - 1) / (32 * wn), (m_rows + 32 * mtw - 1) / (32 * mtw));
      hipLaunchKernelGGL(kern, grid, dim3(64 * wn), lds, stream, w, row_bytes, hi, lo, k, y, ldy, m_rows,
                         n_rows, pieces);
    };
    // Two activation tiles share a wave's looked-up weights, and eight waves an activation block in LDS,
    // while the grid fills the chip. Measured on MI355X, us per call with the split, eight waves of two
    // tiles / four of two / two of one: 4096 x 4096 M = 2048 (512 workgroups of the first form) 183 / 216 /
    // 317, M = 512 (128) 83 / 58 / 92, M = 64 (16) 80 / 53 / 41; 14336 x 4096 M = 512 (448) 166 / 200 / 269.
    const long long m_tiles = (m_rows + 63) / 64, cus = cu_count();
    if ((n_rows + 255) / 256 * m_tiles >= cus) go(iq4_ptile_kernel<8, 2>, 8, 2);
    else if ((n_rows + 127) / 128 * m_tiles >= cus * 3 / 4) go(iq4_ptile_kernel<4, 2>, 4, 2);
    else go(iq4_ptile_kernel<2, 1>, 2, 1);
  };
  const int step = prow_limit(row_bytes);
  for (long long n0 = 0; n0 < n_rows; n0 += step)
    launch(w + n0 * row_bytes, y.at(n0), (int)min((long long)step, n_rows - n0));
  return 0;
}

}  // namespace mxa
