// Prefill matmul (more than 16 activation rows) on the 32 x 32 matrix instructions: Q4_K, Q6_K and
// Q8_0 weights on Q8_K activations in the workspace.
//
// Tiling. A wave owns 32 weight rows x 32 MTW activation rows, a workgroup WN waves along the
// weight rows: every wave decodes its own weights (once, into registers) and all of them read the
// workgroup's activation rows from LDS. One v_mfma_i32_32x32x32_i8 covers one 32-value sub-block
// of Q4_K / Q8_0 (two 16-value sub-blocks of Q6_K): lane l supplies row l % 32 and elements
// 16 h .. 16 h + 15 of the chunk, h = l / 32, of both operands, and holds weight row n = l % 32 of
// the results for activation rows m = 8 (i / 4) + 4 h + i % 4, i < 16.
//
// Against 16 x 16 tiles each activation byte read from LDS meets twice the weights, and the
// weights of a chunk are decoded right before the MFMAs that use them, so that only one chunk's
// operands are live and the decode of one chunk overlaps the MFMAs of another.
//
// Copies. A block's 256 bytes of every activation row go straight into LDS (global_load_lds_dwordx4, no
// registers) in one of two buffers; 16-byte piece c of row r sits at place c ^ (r & 15), so the 32
// rows of an operand read are spread over all banks without padding. A wave's own weights go into a
// slot that only it reads: it takes the block into registers and refills the slot at once. Loading
// the weights per lane into registers instead cost a fifth (Q4_K) to a half (Q6_K) of the time.
//
// Bound: no unit of its own. A 32 x 64 x 256 step of a Q4_K wave issues about 430 VALU instructions (decode,
// fold, addresses) and 34 MFMAs of 32 cycles. Over Q4_K 14336 x 4096 M = 2048 VALU instructions issue in 56%
// of a SIMD's cycles and the matrix cores are busy in 33%, of which 59% beside VALU instructions; the waves
// spend 31% of their time in waits. Q6_K 4096 x 14336 M = 1024: 52%, 19%, 56%, and 25%; 29% goes to waiting to
// issue LDS reads (12% for Q4_K), which start at 2-byte places and lose 12 cycles each to bank conflicts (3.5).
// Two waves share a SIMD and meet at every block's barrier, so decode, MFMAs and folds overlap in part only;
// more stages of copies ahead or another order of the instructions change nothing.
//
// Measured on MI355X against the 16 x 16 tiles before (us, kernel alone, weights from HBM): Q4_K 14336 x 4096
// M = 2048 321 vs 351 (750 TFLOP/s equivalent), M = 512 88 vs 96, M = 64 24 vs 52; Q6_K 4096 x 14336 M = 1024 246
// vs 488 (its sub-block scales went into two planes: 16 quarter-filled MFMAs and 64 integer products per
// output quad before), 128256 x 4096 M = 32 159 vs 414; Q8_0 4096 x 4096 M = 2048 113 vs 258, M = 333 37 vs 58.
// Q4_K weights that start off a 16-byte boundary lose 5 to 17% to them: their blocks are read from LDS at
// dword places.
//
// Numerics: integer sums are exact and the fp32 steps are the oracle's, in block order, so the
// outputs equal the decode kernels' bit for bit.
#include "mxa_kernels.hpp"
#include "mxa_pcopy.hpp"
#include "mxa_tiles.hpp"

#pragma clang fp contract(off)

namespace mxa {
namespace {

typedef int32_t i32x16 __attribute__((ext_vector_type(16)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int16_t i16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ i32x16 mfma_i8(i32x4 a, i32x4 b, i32x16 c) {
  return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0);
}

// s_waitcnt lgkmcnt(0): this wave's LDS reads have returned.
__device__ __forceinline__ void wait_lgkm0() {
  __builtin_amdgcn_s_waitcnt(0xC07F);
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

constexpr f32x16 kZeroF = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

// Integer sums become floats without a conversion. An MFMA chain that starts from kMagic, the bits
// of 1.5 x 2^23, ends in the bits of the float 1.5 x 2^23 + sum, exactly, while |sum| < 2^22. Two planes
// hi and lo of weight S (a power of two) then give float(S hi + lo), rounded once as the integer
// conversion rounds it, by fma(hi', S, -(S + 1) x 1.5 x 2^23) + lo': the first term is S hi -
// 1.5 x 2^23, a multiple of S below 2^24 S, hence exact. On gfx950 v_fma_f32, v_add_f32 and
// v_mul_f32 issue in two cycles per wave, v_cvt_f32_i32 and v_lshl_add_u32 in four.
constexpr int kMagic = 0x4B400000;
constexpr float kMagicF = 12582912.0f;

// A value that the compiler keeps in vector registers: an AND with a scalar mask takes four cycles
// and one with a vector mask two, and a float that it knows to come from a half becomes an operand
// of v_fma_mix_f32 (four cycles, v_fma_f32 two).
template <class V>
__device__ __forceinline__ V in_vgpr(V v) {
  asm("" : "+v"(v));
  return v;
}

__device__ __forceinline__ float as_f32(int v) { return __builtin_bit_cast(float, v); }

// One block of the activations in LDS as a wave's tile mt reads it; the bsums as int16 (kRaw) or as fp16,
// exactly (|bsum| <= 2032).
template <bool kRaw>
struct PAct {
  const uint8_t* q;    // swizzled rows of 256 bytes
  const uint8_t* bs;   // bsums, 32 bytes per row
  const float* d;
  int r, h;            // lane % 32, lane / 32
  __device__ __forceinline__ i32x4 a(int mt, int t) const {
    return __builtin_bit_cast(i32x4, *(const u32x4*)(q + (32 * mt + r) * QK + 16 * ((2 * t + h) ^ (r & 15))));
  }
  // bsums 8 h .. 8 h + 7 of row r
  __device__ __forceinline__ f16x8 b(int mt) const {
    const uint8_t* p = bs + (32 * mt + r) * 32 + 16 * h;
    if constexpr (kRaw)
      return __builtin_convertvector(*(const i16x8*)p, f16x8);
    else
      return *(const f16x8*)p;
  }
  // scales of activation rows 8 q4 + 4 h + 0..3 of tile mt
  __device__ __forceinline__ f32x4 xd(int mt, int q4) const { return *(const f32x4*)(d + 32 * mt + 8 * q4 + 4 * h); }
};

// The two-plane types' block, chunk by chunk.
template <class T, int MTW, class Act, class Sink>
__device__ __forceinline__ void two_planes(const typename T::W& w, const Act& A, const i32x16& magic, Sink&& sink) {
  const typename T::S s = T::scales(w);
  const uint32_t m4 = in_vgpr(0x0F0F0F0Fu);
  i32x16 hi[MTW], lo[MTW];
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) hi[mt] = lo[mt] = magic;
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    i32x4 bh, bl;
    T::planes(w, s, t, m4, A.h, bh, bl);
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt) {
      const i32x4 a = A.a(mt, t);
      hi[mt] = mfma_i8(a, bh, hi[mt]);
      lo[mt] = mfma_i8(a, bl, lo[mt]);
    }
  }
  const typename T::F f = T::folds(w, s, A.h);
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) sink(mt, T::value(f, A, mt, hi[mt], lo[mt]), f.d);
}

// Every type: W, a lane's bytes of one block of its weight row; load(lds, off, h), from the wave's
// slot; and block<MTW>, which calls sink(mt, v, d) with the block's 16 values of each tile and its
// weight scale. The oracle's fold is acc = fma(xd, v, acc), or fma(xd * d, v, acc) where kScaled.
struct PQ4 {
  static constexpr bool kBsums = true, kScaled = false;
  struct W {
    u32x4a4 hdr, q[4];
  };
  static constexpr int kBytes = 144, kShift = 0;
  __device__ __forceinline__ static W load(const uint8_t* lds, int off, int h) {
    const uint8_t* p = lds + off;
    W w;
    w.hdr = ld16(p);
#pragma unroll
    for (int c = 0; c < 4; ++c) w.q[c] = ld16(p + 16 + 32 * c + 16 * h);
    return w;
  }
  struct S {
    K4Scales s;
  };
  __device__ __forceinline__ static S scales(const W& w) { return S{k4_scales(w.hdr.y, w.hdr.z, w.hdr.w)}; }
  // chunk t's planes: u * sc = 8 (u * (sc >> 3)) + u * (sc & 7), each at most 105
  __device__ __forceinline__ static void planes(const W& w, const S& s, int t, uint32_t m4, int, i32x4& bh, i32x4& bl) {
    const uint32_t sc = k4_pick(s.s.sc_lo, s.s.sc_hi, t), sh = sc >> 3, sl = sc & 7;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t q = w.q[t >> 1][i], u = ((t & 1) ? q >> 4 : q) & m4;
      bh[i] = (int)mul_bytes(u, sh);
      bl[i] = (int)mul_bytes(u, sl);
    }
  }
  struct F {
    f16x8 bm;
    float d, dmin, k9;
  };
  __device__ __forceinline__ static F folds(const W& w, const S& s, int h) {
    // summ = sum of min_{j / 2} * bsum_j over the 16 bsums, exact in one fp16 MFMA
    const uint32_t mn = h ? s.s.mn_hi : s.s.mn_lo;
    F f;
#pragma unroll
    for (int j = 0; j < 4; ++j) f.bm[2 * j] = f.bm[2 * j + 1] = (_Float16)(float)((mn >> (8 * j)) & 0xFFu);
    f.d = in_vgpr(half_to_float(w.hdr.x)), f.dmin = in_vgpr(half_to_float(w.hdr.x >> 16));
    f.k9 = in_vgpr(-9.0f * kMagicF);
    return f;
  }
  template <class Act>
  __device__ __forceinline__ static f32x16 value(const F& f, const Act& A, int mt, const i32x16& hi,
                                                 const i32x16& lo) {
    const f32x16 summ = __builtin_amdgcn_mfma_f32_32x32x16_f16(A.b(mt), f.bm, kZeroF, 0, 0, 0);
    f32x16 v;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float sumi = fmaf(as_f32(hi[i]), 8.0f, f.k9) + as_f32(lo[i]);
      v[i] = fmaf(f.d, sumi, -(f.dmin * summ[i]));
    }
    return v;
  }
  template <int MTW, class Act, class Sink>
  __device__ __forceinline__ static void block(const W& w, const Act& A, const i32x16& magic, Sink&& sink) {
    two_planes<PQ4, MTW>(w, A, magic, sink);
  }
};

struct PQ6 {
  static constexpr bool kBsums = false, kScaled = true;
  struct W {
    u32x4a4 ql[4], qh[2], sc;  // ql[64 hh + 32 q + 16 h ..] at 2 hh + q, qh[32 hh + 16 h ..]
    uint32_t d;
  };
  static constexpr int kBytes = 210, kShift = 14;
  // 16 bytes from a 2-byte aligned place, by dwords and v_alignbyte (sh = 0 takes no byte of e)
  __device__ __forceinline__ static u32x4a4 ld16_a2(const uint8_t* base, uint32_t sh) {
    const u32x4a4 v = ld16(base);
    const uint32_t e = ld4(base + 16);
    return u32x4a4{__builtin_amdgcn_alignbyte(v.y, v.x, sh), __builtin_amdgcn_alignbyte(v.z, v.y, sh),
                   __builtin_amdgcn_alignbyte(v.w, v.z, sh), __builtin_amdgcn_alignbyte(e, v.w, sh)};
  }
  __device__ __forceinline__ static W load(const uint8_t* lds, int off, int h) {
    const uint32_t sh = (uint32_t)(off & 2);
    const uint8_t* p = lds + (off & ~3);
    W w;
#pragma unroll
    for (int c = 0; c < 4; ++c) w.ql[c] = ld16_a2(p + 32 * c + 16 * h, sh);
#pragma unroll
    for (int c = 0; c < 2; ++c) w.qh[c] = ld16_a2(p + 128 + 32 * c + 16 * h, sh);
    const u32x4a4 v = ld16(p + 192);
    const uint32_t e = ld4(p + 208);
    w.sc = u32x4a4{__builtin_amdgcn_alignbyte(v.y, v.x, sh), __builtin_amdgcn_alignbyte(v.z, v.y, sh),
                   __builtin_amdgcn_alignbyte(v.w, v.z, sh), __builtin_amdgcn_alignbyte(e, v.w, sh)};
    w.d = e >> (8 * sh);
    return w;
  }
  struct S {};
  __device__ __forceinline__ static S scales(const W&) { return S{}; }
  __device__ __forceinline__ static void planes(const W& w, const S&, int t, uint32_t m4, int h, i32x4& bh, i32x4& bl) {
    // chunk t = elements 32 t .. of half hh = t / 4, quarter r = t % 4; this lane's sixteen share
    // scale 2 t + h. p = (u - 32) * sc is 13 bits: p + 128 in 16 bits, its high byte the plane
    // of 256, its low byte less 128 the plane of 1
    const int hh = t >> 2, r = t & 3;
    const uint32_t sw = w.sc[t >> 1] >> (16 * (t & 1));
    const int sc = (int)(int8_t)(uint8_t)(h ? sw >> 8 : sw);
    const u16x2 s2 = {(uint16_t)sc, (uint16_t)sc};
    const uint16_t c0 = (uint16_t)(128 - 32 * sc);
    const u16x2 c2 = {c0, c0};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t l = w.ql[2 * hh + (r & 1)][i], g = w.qh[hh][i];
      const uint32_t u = r == 0 ? q6_codes<0>(l, g) : r == 1 ? q6_codes<1>(l, g)
                       : r == 2 ? q6_codes<2>(l, g) : q6_codes<3>(l, g);
      const u16x2 ue = __builtin_bit_cast(u16x2, u & 0x00FF00FFu);
      const u16x2 uo = __builtin_bit_cast(u16x2, __builtin_amdgcn_perm(0u, u, 0x0C030C01u));
      const uint32_t pe = __builtin_bit_cast(uint32_t, (u16x2)(ue * s2 + c2));
      const uint32_t po = __builtin_bit_cast(uint32_t, (u16x2)(uo * s2 + c2));
      bh[i] = (int)__builtin_amdgcn_perm(po, pe, 0x07030501u);
      bl[i] = (int)(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
    }
  }
  struct F {
    float d, k257;
  };
  __device__ __forceinline__ static F folds(const W& w, const S&, int) {
    return F{in_vgpr(half_to_float(w.d)), in_vgpr(-257.0f * kMagicF)};
  }
  template <class Act>
  __device__ __forceinline__ static f32x16 value(const F& f, const Act&, int, const i32x16& hi, const i32x16& lo) {
    f32x16 v;
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = fmaf(as_f32(hi[i]), 256.0f, f.k257) + as_f32(lo[i]);
    return v;
  }
  template <int MTW, class Act, class Sink>
  __device__ __forceinline__ static void block(const W& w, const Act& A, const i32x16& magic, Sink&& sink) {
    two_planes<PQ6, MTW>(w, A, magic, sink);
  }
};

struct PQ8 {
  static constexpr bool kBsums = false, kScaled = false;
  struct W {
    // blocks 2 j and 2 j + 1 are 68 bytes from 68 j: d, 32 quants, d, 32 quants; this lane's half
    // of the even one's quants starts in the upper half of dword 4 h, the odd one's at dword 9 + 4 h
    u32x4a4 e[4], o[4];
    uint32_t x[4];  // dword 4 h + 4: the end of the even quants (h = 1: and the odd block's d)
  };
  static constexpr int kBytes = 272, kShift = 0;
  __device__ __forceinline__ static W load(const uint8_t* lds, int off, int h) {
    const uint8_t* p = lds + off + 16 * h;
    W w;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      w.e[j] = ld16(p + 68 * j);
      w.x[j] = ld4(p + 68 * j + 16);
      w.o[j] = ld16(p + 68 * j + 36);
    }
    return w;
  }
  template <int MTW, class Act, class Sink>
  __device__ __forceinline__ static void block(const W& w, const Act& A, const i32x16& magic, Sink&& sink) {
    const float kb = in_vgpr(kMagicF);
    i32x4 bq[8];
    float dk[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // lanes of h = 0 hold the even block's d (dword 0), those of h = 1 the odd one's (dword 8)
      const uint32_t mine = A.h ? w.x[j] >> 16 : w.e[j].x & 0xFFFFu;
      const uint32_t other = (uint32_t)__shfl_xor((int)mine, 32, 64);
      dk[2 * j] = in_vgpr(half_to_float(A.h ? other : mine));
      dk[2 * j + 1] = in_vgpr(half_to_float(A.h ? mine : other));
      const uint32_t ev[5] = {w.e[j].x, w.e[j].y, w.e[j].z, w.e[j].w, w.x[j]};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bq[2 * j][i] = (int)__builtin_amdgcn_alignbyte(ev[i + 1], ev[i], 2);
        bq[2 * j + 1][i] = (int)w.o[j][i];
      }
    }
    // tile by tile, the sums of two blocks open at a time
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt) {
      f32x16 bs = kZeroF;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const i32x16 p = mfma_i8(A.a(mt, k), bq[k], magic);
#pragma unroll
        for (int i = 0; i < 16; ++i) bs[i] = fmaf(dk[k], as_f32(p[i]) - kb, bs[i]);
        asm("" : "+v"(bs));
      }
      sink(mt, bs, 1.0f);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
};

template <int TYPE>
struct PTileOf;
template <> struct PTileOf<T_Q4_K> { using T = PQ4; };
template <> struct PTileOf<T_Q6_K> { using T = PQ6; };
template <> struct PTileOf<T_Q8_0> { using T = PQ8; };

// LDS bytes of one block of `rows` activation rows: q8 | bsums (fp16) | d.
constexpr int pbuf_bytes(int rows) { return rows * (QK + 32 + 4); }

// The outputs of activation rows m0 .. m0 + 32 MTW - 1 of M.
template <int TYPE, int WN, int MTW>
__device__ __forceinline__ void ptile_rows(const uint8_t* w, long long row_bytes, const Act& act, YOut y,
                                           long long ldy, int M, int N, int pieces, int wg, int n_wg, int m0) {
  using T = typename PTileOf<TYPE>::T;
  constexpr int kRows = 32 * MTW, kThreads = 64 * WN, kBuf = pbuf_bytes(kRows);
  extern __shared__ __align__(16) uint8_t smem[];  // two buffers
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int n0 = (xcd_tile(wg, n_wg) * WN + wave) * 32, n = n0 + r;
  const int nb = act.nb;

  const PWeights<T> pw(w, row_bytes, n0, N, pieces, lane);
  const int slot = 2 * kBuf + wave * pslot_bytes(pieces);
  const uint32_t slot0 = lds_addr(smem) + slot;

  // this wave's copies of a block: 4 rows x 16 pieces each (rows >= M repeat row M - 1)
  constexpr int kCopies = kRows / 4 / WN;
  static_assert(kCopies * 4 * WN == kRows, "whole copies per wave");
  const int8_t* src[kCopies];
#pragma unroll
  for (int c = 0; c < kCopies; ++c) {
    const int rr = 4 * (wave * kCopies + c) + (lane >> 4);
    src[c] = act.q + (size_t)min(m0 + rr, M - 1) * act.k + 16 * ((lane & 15) ^ (rr & 15));
  }
  const uint32_t lds0 = lds_addr(smem);
  auto copy_q = [&](int b, int buf) {
#pragma unroll
    for (int c = 0; c < kCopies; ++c)
      copy16_to_lds(src[c] + (size_t)b * QK,
                    (uint32_t)__builtin_amdgcn_readfirstlane(
                        (int)(lds0 + buf * kBuf + (wave * kCopies + c) * 4 * QK)));
  };
  // bsums (16 bytes = half a block per thread) and scales through registers
  constexpr int kBPer = (2 * kRows + kThreads - 1) / kThreads;
  constexpr int kDPer = (kRows + kThreads - 1) / kThreads;
  u32x4a4 sb[kBPer];
  float sd[kDPer];
  auto load_s = [&](int b) {
    if constexpr (T::kBsums) {
#pragma unroll
      for (int j = 0; j < kBPer; ++j) {
        const int p = min(tid + kThreads * j, 2 * kRows - 1);
        sb[j] = ld16((const uint8_t*)(act.bsums + ((size_t)min(m0 + (p >> 1), M - 1) * nb + b) * 16) + 16 * (p & 1));
      }
    }
#pragma unroll
    for (int j = 0; j < kDPer; ++j)
      sd[j] = act.d[(size_t)min(m0 + min(tid + kThreads * j, kRows - 1), M - 1) * nb + b];
  };
  auto store_s = [&](int buf) {
    uint8_t* bs = smem + buf * kBuf + kRows * QK;
    float* dd = (float*)(bs + kRows * 32);
    if constexpr (T::kBsums) {
#pragma unroll
      for (int j = 0; j < kBPer; ++j) {
        const int p = tid + kThreads * j;
        if (p < 2 * kRows) {
          *(f16x8*)(bs + 16 * p) = __builtin_convertvector(__builtin_bit_cast(i16x8, sb[j]), f16x8);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < kDPer; ++j)
      if (tid + kThreads * j < kRows) dd[tid + kThreads * j] = sd[j];
  };

  f32x16 acc[MTW];
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) acc[mt] = kZeroF;

  i32x16 magic;
#pragma unroll
  for (int i = 0; i < 16; ++i) magic[i] = kMagic;
  magic = in_vgpr(magic);
  load_s(0);
  copy_q(0, 0);
  pw.copy(0, slot0);
  store_s(0);
  wait_vmcnt(0);
  __syncthreads();
  for (int b = 0; b < nb; ++b) {
    const int buf = b & 1;
    const bool more = b + 1 < nb;
    const typename T::W cur = T::load(smem, slot + pw.at(b, r), h);
    if (more) {
      load_s(b + 1);
      copy_q(b + 1, buf ^ 1);
      wait_lgkm0();  // the weights are in registers: their slot takes the next block's
      pw.copy(b + 1, slot0);
    }
    const uint8_t* base = smem + buf * kBuf;
    const PAct<false> A{base, base + kRows * QK, (const float*)(base + kRows * (QK + 32)), r, h};
    T::template block<MTW>(cur, A, magic, [&](int mt, const f32x16& v, float d) {
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const f32x4 xd = A.xd(mt, q4);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[mt][4 * q4 + e] = fmaf(T::kScaled ? xd[e] * d : xd[e], v[4 * q4 + e], acc[mt][4 * q4 + e]);
      }
    });
    // the folds stay with their MFMAs (left alone, the compiler moves them past the next branch)
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt) asm volatile("" : "+v"(acc[mt]));
    if (more) store_s(buf ^ 1);
    wait_vmcnt(0);    // this wave's pieces of the next block are in LDS
    __syncthreads();  // everyone's are, and everyone is done with this block
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

template <int TYPE, int WN, int MTW>
__global__ __launch_bounds__(64 * WN, 2) void ptile_kernel(const uint8_t* w, long long row_bytes, Act act,
                                                           YOut y, long long ldy, int M, int N,
                                                           int pieces) {
  ptile_rows<TYPE, WN, MTW>(w, row_bytes, act, y, ldy, M, N, pieces, blockIdx.x, gridDim.x,
                            32 * MTW * blockIdx.y);
}

// Grouped MoE projection: item blockIdx.z of the (expert, chunk of 32 MTW rows) list
// (moe_chunk_item), workgroups along the expert's weight rows in blockIdx.x.
template <int TYPE, int WN, int MTW>
__global__ __launch_bounds__(64 * WN, 2) void moe_ptile_kernel(const uint8_t* w, long long row_bytes,
                                                               long long expert_stride, Act act,
                                                               const int32_t* __restrict__ offsets,
                                                               int n_experts, int total_rows, YOut y,
                                                               long long ldy, int N, int pieces) {
  int e, p0, M;
  // past the list: uniform over the workgroup, before any barrier
  if (!moe_chunk_item(offsets, n_experts, total_rows, 32 * MTW, blockIdx.z, e, p0, M)) return;
  Act a = act;
  a.q = act.q + (size_t)p0 * act.k;
  a.d = act.d + (size_t)p0 * act.nb;
  a.bsums = act.bsums + (size_t)p0 * act.nb * 16;
  const uint8_t* we = w + (size_t)e * expert_stride;
  const YOut ye = y.at((size_t)p0 * ldy);
  // an expert's last rows often need one tile only (the choice stands outside the block loop: inside it,
  // the accumulators' moves cost a tenth of the time)
  if (MTW == 2 && M <= 32)
    ptile_rows<TYPE, WN, 1>(we, row_bytes, a, ye, ldy, M, N, pieces, blockIdx.x, gridDim.x, 0);
  else
    ptile_rows<TYPE, WN, MTW>(we, row_bytes, a, ye, ldy, M, N, pieces, blockIdx.x, gridDim.x, 0);
}

// Few tiles (short prompts, narrow matrices): the four waves of a workgroup share one tile of 32 weight
// rows x 32 activation rows and take its blocks in turn, wave k blocks 4 r + k of round r, each with
// its own copies of both operands. A round's block values meet in LDS, and wave j folds the outputs of
// activation rows 8 j .. 8 j + 7 of each half, blocks in order, so the bits are the same.
//
// Bound: latency. A workgroup alone on its CU takes 1.8 us a round of four blocks (Q4_K; Q6_K 2.8, Q8_0 2.3):
// the wait for its copies, a decode and MFMAs that no other wave of the SIMD covers, two barriers. So what
// counts is the number of rounds and the waves in flight: two workgroups fit a CU (74 KB of LDS for Q4_K, 78
// for Q6_K; Q8_0's 86 leave one).
constexpr int kKs = 4;
template <class T>
constexpr int ks_act_bytes() { return 32 * QK + (T::kBsums ? 1024 : 0) + 256; }
constexpr int kKsV = 4096 + 256;  // a wave's block values, then its activation and weight scales

template <int TYPE>
__global__ __launch_bounds__(64 * kKs, 2) void ktile_kernel(const uint8_t* w, long long row_bytes, Act act,
                                                            YOut y, long long ldy, int M, int N, int pieces) {
  using T = typename PTileOf<TYPE>::T;
  extern __shared__ __align__(16) uint8_t smem[];
  const int lane = threadIdx.x & 63;
  const int wave = (int)uniform(threadIdx.x >> 6);
  const int r = lane & 31, h = lane >> 5;
  const int n0 = xcd_tile(blockIdx.x, gridDim.x) * 32, n = n0 + r, m0 = 32 * blockIdx.y;
  const int nb = act.nb;
  const int slot = pslot_bytes(pieces);
  const int mine = wave * (ks_act_bytes<T>() + slot), values = kKs * (ks_act_bytes<T>() + slot);
  uint8_t* base = smem + mine;
  const uint32_t lds0 = lds_addr(smem) + mine;
  const PWeights<T> pw(w, row_bytes, n0, N, pieces, lane);

  const int8_t* src[8];  // 4 activation rows per copy (rows >= M repeat row M - 1)
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    const int rr = 4 * c + (lane >> 4);
    src[c] = act.q + (size_t)min(m0 + rr, M - 1) * act.k + 16 * ((lane & 15) ^ (rr & 15));
  }
  const float* dsrc = act.d + (size_t)min(m0 + r, M - 1) * nb;
  const int16_t* bsrc = act.bsums + (size_t)min(m0 + (lane >> 1), M - 1) * nb * 16 + 8 * (lane & 1);
  constexpr int kBs = 32 * QK, kD = kBs + (T::kBsums ? 1024 : 0), kW = kD + 256;
  auto issue = [&](int b) {
    pw.copy(b, lds0 + kW);
#pragma unroll
    for (int c = 0; c < 8; ++c) copy16_to_lds(src[c] + (size_t)b * QK, uniform(lds0 + 1024 * c));
    if constexpr (T::kBsums) copy16_to_lds(bsrc + (size_t)b * 16, uniform(lds0 + kBs));
    copy4_to_lds(dsrc + b, uniform(lds0 + kD));
  };

  i32x16 magic;
#pragma unroll
  for (int i = 0; i < 16; ++i) magic[i] = kMagic;
  magic = in_vgpr(magic);
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  if (wave < nb) issue(wave);
  for (int b0 = 0; b0 < nb; b0 += kKs) {
    const int b = b0 + wave;
    if (b < nb) {
      wait_vmcnt(0);
      const typename T::W cur = T::load(base, kW + pw.at(b, r), h);
      const PAct<true> A{base, base + kBs, (const float*)(base + kD), r, h};
      f32x4* V = (f32x4*)(smem + values + wave * kKsV);
      T::template block<1>(cur, A, magic, [&](int, const f32x16& v, float d) {
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) V[64 * q4 + lane] = f32x4{v[4 * q4], v[4 * q4 + 1], v[4 * q4 + 2], v[4 * q4 + 3]};
        // lanes of h = 0 keep the activation scales, those of h = 1 the weight scales
        ((float*)(V + 256))[lane] = h ? d : A.d[r];
      });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // this wave has read its operands
      if (b + kKs < nb) issue(b + kKs);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kKs; ++k)
      if (b0 + k < nb) {
        const f32x4* V = (const f32x4*)(smem + values + k * kKsV);
        const float* s = (const float*)(V + 256);
        const f32x4 v = V[64 * wave + lane], xd = *(const f32x4*)(s + 8 * wave + 4 * h);
        const float d = s[32 + r];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(T::kScaled ? xd[e] * d : xd[e], v[e], acc[e]);
      }
    __syncthreads();  // the values have been read
  }
  if (n < N) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = m0 + 8 * wave + 4 * h + e;
      if (m < M) y.put((size_t)m * ldy + n, acc[e]);
    }
  }
}

template <int TYPE>
int launch_k(const uint8_t* w, long long row_bytes, const Act& act, YOut y, long long ldy, int M, int N,
             hipStream_t stream) {
  using T = typename PTileOf<TYPE>::T;
  const int pieces = ppieces<T>(((uintptr_t)w & 15) == 0 && row_bytes % 16 == 0);
  const int lds = kKs * (ks_act_bytes<T>() + pslot_bytes(pieces) + kKsV);
  allow_lds((const void*)ktile_kernel<TYPE>, lds);
  hipLaunchKernelGGL((ktile_kernel<TYPE>), dim3((N + 31) / 32, (M + 31) / 32), dim3(64 * kKs), lds, stream, w,
                     row_bytes, act, y, ldy, M, N, pieces);
  return 0;
}

template <int TYPE, int WN, int MTW>
int launch_p(const uint8_t* w, long long row_bytes, const Act& act, YOut y, long long ldy, int M, int N,
             hipStream_t stream) {
  const bool aligned = ((uintptr_t)w & 15) == 0 && row_bytes % 16 == 0;
  const int pieces = ppieces<typename PTileOf<TYPE>::T>(aligned);
  const int lds = 2 * pbuf_bytes(32 * MTW) + WN * pslot_bytes(pieces);
  allow_lds((const void*)ptile_kernel<TYPE, WN, MTW>, lds);
  const dim3 grid((N + 32 * WN - 1) / (32 * WN), (M + 32 * MTW - 1) / (32 * MTW));
  hipLaunchKernelGGL((ptile_kernel<TYPE, WN, MTW>), grid, dim3(64 * WN), lds, stream, w, row_bytes, act, y,
                     ldy, M, N, pieces);
  return 0;
}

// Few 32 x 32 tiles take a workgroup each. Otherwise two activation tiles share a wave's decoded
// weights, and eight waves an activation block in LDS, as long as the grid still fills the chip.
// Measured on MI355X, us, kernel alone, weights from HBM; workgroup per tile / two waves of one tile / four of two:
//   Q4_K 4096 x 4096 M = 32 / 128 / 200 / 333 (128 / 512 / 896 / 1408 tiles) 11 / 21 / 29, 13 / 21 / 30,
//   23 / 30 / 30, 32 / 31 / 30; 14336 x 4096 M = 64 / 128 (896 / 1792) 24 / 29 / 30, 40 / 35 / 31; Q6_K
//   4096 x 14336 M = 256 (1024) 124 / 172 / 152; Q8_0 4096 x 4096 M = 128 / 333 (512 / 1408) 24 / 30 / 45,
//   62 / 37 / 46, 14336 x 4096 M = 48 (896; its workgroup per tile has a CU to itself) 49 / 34 / 46;
// eight waves of two tiles / four of two / two of one: Q4_K 14336 x 4096 M = 2048 321 / 303 / 427, 4096 x
//   4096 M = 1024 48 / 49 / 70, 128256 x 4096 M = 32 106 / 101 / 94 (half of every second tile's rows are
//   repeats); Q6_K 4096 x 14336 M = 1024 250 / 250 / 453, 128256 x 4096 M = 32 159 / 156 / 144; Q8_0 4096 x 4096
//   M = 2048 116 / 112 / 158.
template <int TYPE>
int launch_p_type(const uint8_t* w, long long row_bytes, const Act& act, YOut y, long long ldy, int M, int N,
                  hipStream_t stream) {
  const long long m_tiles = (M + 63) / 64, cus = cu_count();
  const long long tiles = (long long)((N + 31) / 32) * ((M + 31) / 32);
  if (tiles <= (TYPE == T_Q8_0 ? 2 : 4) * cus) return launch_k<TYPE>(w, row_bytes, act, y, ldy, M, N, stream);
  if (TYPE != T_Q8_0 && (N + 255) / 256 * m_tiles >= cus)
    return launch_p<TYPE, 8, 2>(w, row_bytes, act, y, ldy, M, N, stream);
  if ((N + 127) / 128 * m_tiles >= (TYPE == T_Q8_0 ? cus * 3 / 2 : cus * 3 / 4))
    return launch_p<TYPE, 4, 2>(w, row_bytes, act, y, ldy, M, N, stream);
  return launch_p<TYPE, 2, 1>(w, row_bytes, act, y, ldy, M, N, stream);
}

template <int TYPE, int WN, int MTW>
int launch_moe_p(const uint8_t* w, long long row_bytes, long long expert_stride, int n_experts, const Act& act,
                 const int32_t* offsets, int total_rows, YOut y, long long ldy, int N, hipStream_t stream) {
  const bool aligned = ((uintptr_t)w & 15) == 0 && row_bytes % 16 == 0 && expert_stride % 16 == 0;
  const int pieces = ppieces<typename PTileOf<TYPE>::T>(aligned);
  const int lds = 2 * pbuf_bytes(32 * MTW) + WN * pslot_bytes(pieces);
  const long long items = n_experts + (total_rows + 32 * MTW - 1) / (32 * MTW);
  if (n_experts > 256 || items > 65535) return -1;
  allow_lds((const void*)moe_ptile_kernel<TYPE, WN, MTW>, lds);
  hipLaunchKernelGGL((moe_ptile_kernel<TYPE, WN, MTW>), dim3((N + 32 * WN - 1) / (32 * WN), 1, (unsigned)items),
                     dim3(64 * WN), lds, stream, w, row_bytes, expert_stride, act, offsets, n_experts, total_rows,
                     y, ldy, N, pieces);
  return 0;
}

template <int TYPE>
int launch_moe_p_type(const uint8_t* w, long long row_bytes, long long expert_stride, int n_experts, const Act& act,
                      const int32_t* offsets, int total_rows, YOut y, long long ldy, int N, hipStream_t stream) {
  // 64-row chunks once an expert has more than 32 rows on average: fewer workgroups read its weights.
  // Measured on MI355X, us, 64- / 32-row chunks, random routings: 8 experts, Q4_K 14336 x 4096 28 / 33 / 48 / 96
  // rows an expert 81 / 82, 91 / 97, 104 / 119, 169 / 193, Q6_K 4096 x 14336 22 / 33 / 64 rows 142 / 142, 158 / 225,
  // 249 / 307; over ten expert sets past 32 rows 64-row chunks take 0.92 (Q4_K), 0.78 (Q6_K) and
  // 0.85 (Q8_0) of the time on average, but up to 1.3 where few rows of few experts leave half the chip idle
  // (8 experts, Q4_K 2048 x 8192 33 to 56 rows 57 / 47).
  if (total_rows > 32LL * n_experts)
    return launch_moe_p<TYPE, 4, 2>(w, row_bytes, expert_stride, n_experts, act, offsets, total_rows, y, ldy, N, stream);
  return launch_moe_p<TYPE, 4, 1>(w, row_bytes, expert_stride, n_experts, act, offsets, total_rows, y, ldy, N, stream);
}

}  // namespace

int launch_moe_ptile(int type, const uint8_t* w, long long row_bytes, long long expert_stride, int n_experts,
                     const Act& act, const int32_t* offsets, int total_rows, YOut y, long long ldy, int n_rows,
                     hipStream_t stream) {
  const int step = prow_limit(row_bytes);
  for (long long n0 = 0; n0 < n_rows; n0 += step) {
    auto go = [&](auto f) {
      return f(w + n0 * row_bytes, row_bytes, expert_stride, n_experts, act, offsets, total_rows, y.at(n0), ldy,
               (int)min((long long)step, n_rows - n0), stream);
    };
    const int st = type == T_Q4_K ? go(launch_moe_p_type<T_Q4_K>) : type == T_Q6_K ? go(launch_moe_p_type<T_Q6_K>)
                 : type == T_Q8_0 ? go(launch_moe_p_type<T_Q8_0>) : -1;
    if (st != 0) return st;
  }
  return 0;
}

int launch_ptile(int type, const uint8_t* w, long long row_bytes, const Act& act, YOut y, long long ldy,
                 int m_rows, int n_rows, hipStream_t stream) {
  const int step = prow_limit(row_bytes);
  for (long long m0 = 0; m0 < m_rows; m0 += kMaxPrefillRows)
    for (long long n0 = 0; n0 < n_rows; n0 += step) {
      Act a = act;
      a.q = act.q + m0 * act.k;
      a.d = act.d + m0 * act.nb;
      a.bsums = act.bsums + m0 * act.nb * 16;
      auto go = [&](auto f) {
        return f(w + n0 * row_bytes, row_bytes, a, y.at(m0 * ldy + n0), ldy,
                 (int)min((long long)kMaxPrefillRows, m_rows - m0), (int)min((long long)step, n_rows - n0), stream);
      };
      const int st = type == T_Q4_K ? go(launch_p_type<T_Q4_K>) : type == T_Q6_K ? go(launch_p_type<T_Q6_K>)
                   : type == T_Q8_0 ? go(launch_p_type<T_Q8_0>) : -1;
      if (st != 0) return st;
    }
  return 0;
}

}  // namespace mxa
