// Operand tiles of the plain products (linear.hip, wgrad.hip) in LDS: filled
// by direct global -> LDS copies, which cannot pad a row, so the 16-byte
// chunks of a row are XOR-swizzled by the row to spread the MFMA operand reads
// over all banks.
#pragma once

#include "attn_kernels.h"

namespace t2t {

namespace {

// Byte offset past any buffer: the copy writes zeros and reads no memory.
constexpr int kNowhere = 0x7ffffff0;

// Chunk position of logical chunk c of row r in an LDS tile whose rows are
// BK elements: rows that share banks get different positions.
template <int BK>
__device__ __forceinline__ int swizzle(int r, int c) {
  return c ^ ((r / (128 / BK)) & (BK / 8 - 1));
}

// Operand rows r (of `rows` in the tile) of BK columns from k0 on.
template <int BK, int ROWS>
struct RowTile {
  static constexpr int kChunks = BK / 8;
  static constexpr int kRowsPerCopy = 64 / kChunks;
  static constexpr int kCopies = ROWS / kRowsPerCopy;  // 1 KiB each
  static constexpr int kPerWave = kCopies / kWaves;
  static_assert(kCopies % kWaves == 0, "copies split evenly");
  int off[kPerWave];  // byte offset of the lane's chunk at k0 = 0
  int k[kPerWave];    // its first column
  __device__ __forceinline__ void init(int row0, int64_t stride, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
      const int r = (wave + kWaves * i) * kRowsPerCopy + lane / kChunks;
      const int c = swizzle<BK>(r, lane % kChunks);
      k[i] = 8 * c;
      off[i] = (int)(((int64_t)(row0 + r) * stride + 8 * c) * 2);
    }
  }
  __device__ __forceinline__ void copy(uint32_t lds, u32x4 rsrc, int k0, int K, int wave) const {
#pragma unroll
    for (int i = 0; i < kPerWave; ++i)
      lds_copy16_m0(lds + (wave + kWaves * i) * 1024, k0 + k[i] < K ? off[i] + 2 * k0 : kNowhere,
                    rsrc);
  }
};

// Operand [BK][COLS] with the contraction along the rows.  LDS row r holds
// contraction index kperm(r), the order in which ds_read_b64_tr_b16 pairs
// (lds_col8's addresses) hand lane group g the indices 8 g .. 8 g + 7.
__device__ __forceinline__ int kperm(int r) {
  return (r & ~15) + 8 * (r & 1) + 4 * ((r >> 1) & 1) + ((r >> 2) & 3);
}
template <int COLS>
__device__ __forceinline__ int col_swizzle(int r, int c) {
  return c ^ ((4 * ((r >> 2) & 3)) & (COLS / 8 - 1));
}
template <int BK, int COLS>
struct ColTile {
  static constexpr int kChunks = COLS / 8;
  static constexpr int kRowsPerCopy = 64 / kChunks;
  static constexpr int kCopies = BK / kRowsPerCopy;
  static constexpr int kPerWave = kCopies / kWaves;
  static_assert(kCopies % kWaves == 0, "copies split evenly");
  int off[kPerWave];
  int k[kPerWave];
  __device__ __forceinline__ void init(int col0, int N, int64_t stride, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < kPerWave; ++i) {
      const int r = (wave + kWaves * i) * kRowsPerCopy + lane / kChunks;
      const int c = col_swizzle<COLS>(r, lane % kChunks);
      k[i] = kperm(r);
      // columns past N (features that are not stored) read nothing
      off[i] = col0 + 8 * c < N ? (int)((k[i] * stride + col0 + 8 * c) * 2) : kNowhere;
    }
  }
  __device__ __forceinline__ void copy(uint32_t lds, u32x4 rsrc, int k0, int K, int64_t stride,
                                       int wave) const {
#pragma unroll
    for (int i = 0; i < kPerWave; ++i)
      lds_copy16_m0(lds + (wave + kWaves * i) * 1024,
                    off[i] != kNowhere && k0 + k[i] < K ? off[i] + (int)(2 * k0 * stride)
                                                        : kNowhere,
                    rsrc);
  }
};

// Column operand over the 16 contraction indices of LDS rows [base, base +
// 16): lds_col8 on swizzled rows (8 bytes of rows base + g + 4 (l / 4) and of
// the rows two further on, l the lane in its 16).
template <int COLS>
__device__ __forceinline__ bf16x8 read_col8(const uint8_t* tile, int base, int col0, int lane) {
  const int l = lane & 15;
  const int r = base + (lane >> 5) + 4 * (l >> 2);
  const int col = col0 + 16 * ((lane >> 4) & 1) + 4 * (l & 3);
  const int at = 16 * col_swizzle<COLS>(r, col >> 3) + 2 * (col & 7);
  const __bf16* p = reinterpret_cast<const __bf16*>(tile + r * COLS * 2 + at);
  const bf16x4_ld lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4_ptr)(p));
  const bf16x4_ld hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4_ptr)(p + 2 * COLS));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

}  // namespace

}  // namespace t2t
