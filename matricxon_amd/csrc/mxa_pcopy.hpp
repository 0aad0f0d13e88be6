// Copies of the prefill tiles' operands into LDS: a wave's own weight rows block by block.
#pragma once

#include "mxa_device.hpp"

namespace mxa {

// 16-byte pieces that cover one block of a weight row wherever it starts in its first piece, and a
// wave's LDS bytes for the 32 rows it owns (whole copies of 64 pieces).
// T::kBytes is a block's size, T::kShift how far past a 16-byte boundary its blocks start at most while the
// weight and its rows are aligned, else 12 (weights are 4-byte aligned).
template <class T>
__host__ __device__ constexpr int ppieces(bool aligned) {
  return (T::kBytes + (aligned || T::kShift > 12 ? T::kShift : 12) + 15) / 16;
}
constexpr int pslot_bytes(int pieces) { return (32 * pieces + 63) / 64 * 1024; }

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// 4 bytes per lane from `g` to LDS byte address lds + 4 * lane.
__device__ __forceinline__ void copy4_to_lds(const void* g, uint32_t lds) {
  asm volatile("global_load_lds_dword %0, off" ::"v"(g), "{m0}"(lds) : "memory");
}

// Weight rows that one launch takes: a lane's offset from its wave's first row has 32 bits, which 32 rows of
// 128 MiB (K past 10^8) outgrow.
inline int prow_limit(long long row_bytes) {
  const long long rows = ((1LL << 32) - 512) / row_bytes;
  return rows >= 32 ? 0x7FFFFFFF : rows > 1 ? (int)rows : 1;
}
// Activation rows that one launch takes: 65535 groups of 64 in the grid's second dimension.
constexpr int kMaxPrefillRows = 65535 * 64;

// A wave's 32 weight rows, copied block by block into a slot that only it reads. Piece c of row q comes
// from the 16-byte boundary at or below the block's start. Every piece holds at least one byte of the
// block (`clamp`: a piece that could lie past a block that starts at the boundary repeats the last one
// that does), so none lies outside the 16-byte units that the matrix occupies. Rows >= N repeat row N - 1.
template <class T>
struct PWeights {
  static constexpr int kMax = (32 * ppieces<T>(false) + 63) / 64;
  const uint8_t* row0;  // the 16-byte boundary at or below the first row
  uint32_t off[kMax], pc[kMax];
  uint32_t mine;  // of lane % 32's row from row0
  int pieces, copies;
  bool clamp;
  __device__ __forceinline__ PWeights(const uint8_t* w, long long row_bytes, int n0, int N, int pieces_, int lane)
      : pieces(pieces_), copies(pslot_bytes(pieces_) >> 10), clamp(16 * (pieces_ - 1) >= T::kBytes) {
    const uint32_t mis = (uint32_t)((uintptr_t)w & 15);
    const long long first = (long long)min(n0, N - 1) * row_bytes;
    row0 = (const uint8_t*)((uintptr_t)w & ~(uintptr_t)15) + (first & ~15LL);
    auto row_off = [&](int q) {
      return mis + (uint32_t)(first & 15) + (uint32_t)((min(n0 + q, N - 1) - min(n0, N - 1)) * row_bytes);
    };
#pragma unroll
    for (int i = 0; i < kMax; ++i) {
      const int s = min(64 * i + lane, 32 * pieces - 1), q = s / pieces;
      pc[i] = 16 * (uint32_t)(s - q * pieces);
      off[i] = row_off(q);
    }
    mine = row_off(lane & 31);
  }
  __device__ __forceinline__ void copy(int b, uint32_t slot) const {
#pragma unroll
    for (int i = 0; i < kMax; ++i)
      if (i < copies) {
        const uint32_t start = off[i] + (uint32_t)(T::kBytes * b);
        uint32_t p = (start & ~15u) + pc[i];
        if (clamp) p = min(p, (start + T::kBytes - 1) & ~15u);
        copy16_to_lds_s(row0, p, uniform(slot + 1024 * i));
      }
  }
  // where in the slot row r's block b starts
  __device__ __forceinline__ int at(int b, int r) const {
    return r * pieces * 16 + (int)((mine + (uint32_t)(T::kBytes * b)) & 15u);
  }
};

}  // namespace mxa
