// Shared device code of the float32 attention kernels (v_mfma_f32_32x32x2_f32).
//
// What bounds them: the SIMD's float32 unit.  A float32 MFMA takes it for 64
// cycles and, unlike a bf16 one, hides no VALU work, of its own wave or of
// another (measured: n FMAs behind each MFMA make it 64 + 13 + 4 n cycles, and
// a second wave's FMAs wait for the first wave's MFMAs).  So every SIMD should
// always have MFMAs to issue, with as few vector instructions as possible
// around them, and in as few places.
//
// Decomposition.  A work-group owns 32 rows (queries, or keys in dK/dV) and
// its four waves share the 32 x 32 blocks of the other side out among
// themselves: block number i of the walk over the row's (column's) tiles,
// blocks without an allowed pair not counted, belongs to wave i % 4.  Each
// wave accumulates on its own -- no barrier and no LDS traffic between waves
// until one merge at the end -- so
//   * a row of L tiles is a chain of about L block steps instead of 4 L, and
//     the grid has four times the work-groups: a few short rows fill the chip
//     and the longest row no longer sets the time of a launch;
//   * empty 32 x 32 blocks cost nothing.
// Against 128-row work-groups (K and V staged in LDS in the forward, loads
// without look-ahead in the backward): B1 H4 T1024 D64 forward 28.7 -> 10.5 us;
// B1 H16 T4096 D128 on a linked row (30 % of causal) forward 324 -> 224 us,
// dQ 608 -> 322 us, dK/dV 744 -> 428 us (91, 95 and 95 TFLOP/s of allowed
// pairs; the MFMAs alone take 141, 212 and 283 us at 2.4 GHz).  What is left
// is the vector work above and a work-group's start and merge, about 12 us of
// the 45 that it lives.
// Operands of the streamed side go from global memory to registers (a wave
// reads a block's rows once per contraction, 16 KiB against the contraction's
// 4096 cycles of matrix pipe at D = 128), loaded a contraction ahead; the
// owned rows sit in LDS.
//
// Contractions.  MFMA operand A lane (g = l / 32, n = l % 32) is A[n][k = g],
// B is B[k = g][n], the accumulator entry i is C[acc_row(i, g)][n].
//   over the head dim: k-step 4 i + e pairs dims 8 i + e and 8 i + 4 + e, so
//     that lane (g, n) needs the 16 bytes at dim 8 i + 4 g of its row, and one
//     load instruction covers 32 contiguous bytes of each of 32 rows.  (Loads
//     of 64 bytes of 16 rows run at three times the L1's rate, 31 against 9.6
//     TB/s, but need a transpose inside each quad of lanes, and these kernels
//     do not have the VALU time for it: 930 against 873 us for the three.)
//   over tokens: k-step ks takes the token of accumulator entry ks
//     (acc_row(ks, g)), so a P or dS entry is the B operand as it sits, and
//     output row m of tile dt is head dim DT m + dt, so that a lane's A
//     operands of all DT = D / 32 tiles are one contiguous piece of a row.
#pragma once

#include "attn_kernels.h"

namespace t2t {
namespace f32 {

constexpr int kRows = 32;  // rows of a work-group, and of a streamed block

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f32x16 mfma(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// LDS pitch (floats) of an owned row: 16 bytes of padding.
template <int D>
__device__ __forceinline__ constexpr int pitch() { return D + 4; }

// Buffer over one [T, D] slice: rows at or past T read zero (the range check
// applies to the per-lane offset; the host keeps offsets below 2^31).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t slice(const float* base, int64_t st, int T,
                                                         int D) {
  const int64_t bytes = T > 0 ? ((int64_t)(T - 1) * st + D) * 4 : 0;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0,
                                           (int)(bytes < 0x7fffffff ? bytes : 0x7fffffff),
                                           0x00020000);
}

// Buffer over one head's row statistics (T floats).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_stats(const float* base, int T) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, 4 * T, 0x00020000);
}

__device__ __forceinline__ float load1(__amdgpu_buffer_rsrc_t r, int off) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

__device__ __forceinline__ f32x4 load4(__amdgpu_buffer_rsrc_t r, int off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// Keeps a unit's loads in front of the unit that is contracted meanwhile.
__device__ __forceinline__ void fence() { __builtin_amdgcn_sched_barrier(0); }

// Operands are streamed in units of four loads (16 registers, 16 MFMAs over
// the head dim or 4 DT over tokens).
// Row unit u of a contraction over the head dim (D / 32 units): pieces
// [4 u, 4 u + 4) of the lane's row; off: byte offset of that row plus 16 g.
__device__ __forceinline__ void load_row(f32x4 (&x)[4], __amdgpu_buffer_rsrc_t r, int off, int u) {
#pragma unroll
  for (int j = 0; j < 4; ++j) x[j] = load4(r, off + 32 * (4 * u + j));
}

// Token unit u of a contraction over tokens (4 units): k-steps 4 u + i, i.e.
// floats [DT n, DT n + DT) of rows acc_row(4 u + i, g); off: byte offset of
// row 4 g of the block plus 4 DT n, st4: the row stride in bytes.
template <int D>
__device__ __forceinline__ void load_tok(f32x4 (&x)[4], __amdgpu_buffer_rsrc_t r, int off, int st4,
                                         int u) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (D == 128) {
      x[i] = load4(r, off + (8 * u + i) * st4);
    } else {
      const f32x2 v = __builtin_bit_cast(
          f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off + (8 * u + i) * st4, 0, 0));
      x[i][0] = v[0];
      x[i][1] = v[1];
    }
  }
}

// Owned-row operands come from LDS in pairs of pieces (8 MFMAs): pair p is
// the pieces at floats 16 p and 16 p + 8 past own = LDS row n of the owned
// side plus 4 g floats.
struct OwnPair { f32x4 b[2]; };
__device__ __forceinline__ void load_own(OwnPair& x, const float* own, int p) {
  x.b[0] = *reinterpret_cast<const f32x4*>(own + 16 * p);
  x.b[1] = *reinterpret_cast<const f32x4*>(own + 16 * p + 8);
}

// acc += (streamed rows) x (owned rows)^T over row unit u: pairs 2 u and
// 2 u + 1 of `own`.  The pair in use was read 8 MFMAs earlier: `cur` holds
// pair 2 u on entry and pair 0 of `next_own` (when not NULL, else pair 2 u + 2
// of `own`) on return.
__device__ __forceinline__ void dot_unit(f32x16& acc, const f32x4 (&x)[4], OwnPair& cur,
                                         const float* own, const float* next_own, int u) {
  OwnPair odd;
  load_own(odd, own, 2 * u + 1);
  fence();
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = mfma(x[i][e], cur.b[i][e], acc);
  fence();
  if (next_own) load_own(cur, next_own, 0);
  else load_own(cur, own, 2 * u + 2);
  fence();
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = mfma(x[2 + i][e], odd.b[i][e], acc);
}

// out[dt] += (streamed rows)^T x coef over token unit u.
template <int D>
__device__ __forceinline__ void acc_unit(f32x16 (&out)[D / 32], const f32x4 (&x)[4],
                                         const f32x16& coef, int u) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt) out[dt] = mfma(x[i][dt], coef[4 * u + i], out[dt]);
}

// Seed of a mixed block, tokens in natural order: 0 where the pair is
// allowed, -inf where it is masked; nw = ~w >> (4 g), entry i of lane group g
// is token acc_row(i, g) = 8 (i / 4) + 4 g + i % 4 of the block.
template <int I = 0>
__device__ __forceinline__ void seed_fill(f32x16& c, uint32_t nw) {
  if constexpr (I < 16) {
    c[I] = __int_as_float(sbfe1_c<8 * (I >> 2) + (I & 3)>(nw) & (int)0xff800000);
    seed_fill<I + 1>(c, nw);
  }
}

// A wave's walk over its share of the 32-row blocks of one row's (column's)
// tiles, partial tiles first, then full ones.  The list of the wave's blocks
// is made 64 tiles at a time, outside the contraction loop (a walk that looked
// at a tile's words between two blocks waited, each time, for every operand
// load in flight): lane t of every wave reads its eight of the 32 owned rows'
// mask words of tile t, the waves put what they saw together through LDS, and
// each gathers its own blocks -- at most one per tile -- into one register,
// lane i holding block i.
struct BlockWalk {
  const int32_t* pidx;    // partial tiles
  const int32_t* fidx;    // full tiles
  const int32_t* pslot;   // bitmap slot per partial tile (NULL: the tile index)
  const uint32_t* words;  // slot 0 of the bitmaps
  uint32_t woff;          // word offset in a slot of the lane's owned row
  int npart, ntiles, lane, wave;
  int t0, cnt;            // tiles listed so far, blocks seen so far modulo 4
  int m;                  // blocks of this wave in the listed chunk
  int ent, slot;          // lane i: 4 * tile + block in tile, bit 31 = mixed; bitmap slot
  int tile, seen;         // lane t, between look() and gather(): tile, what its words hold

  // Lane t: tile t0 + t and, when it is partial, for this wave's eight owned
  // rows, bit j = block j has an allowed pair, bit 4 + j = it has a masked
  // one.  row0: word offset in a slot of the first owned row.
  __device__ __forceinline__ void look(uint32_t row0) {
    const int t = t0 + lane;
    tile = t < npart ? pidx[t] : (t < ntiles ? fidx[t - npart] : 0);
    slot = t < npart ? (pslot ? pslot[t] : tile) : 0;
    seen = t < ntiles ? 15 : 0;
    if (t < npart) {
      const uint4* q = reinterpret_cast<const uint4*>(
          words + (size_t)(uint32_t)slot * kTileBitsWords + row0 + 32 * wave);
      uint4 any = q[0], all = any;
#pragma unroll
      for (int r = 1; r < 8; ++r) {
        const uint4 x = q[r];
        any.x |= x.x; any.y |= x.y; any.z |= x.z; any.w |= x.w;
        all.x &= x.x; all.y &= x.y; all.z &= x.z; all.w &= x.w;
      }
      seen = (any.x ? 1 : 0) | (any.y ? 2 : 0) | (any.z ? 4 : 0) | (any.w ? 8 : 0) |
             (~all.x ? 16 : 0) | (~all.y ? 32 : 0) | (~all.z ? 64 : 0) | (~all.w ? 128 : 0);
    }
  }
  // Publishes look()'s result; a barrier separates it from gather().  Two
  // buffers in turn, so that one barrier per chunk is enough.
  __device__ __forceinline__ void publish(uint8_t (*flags)[4][64]) const {
    flags[(t0 >> 6) & 1][wave][lane] = (uint8_t)seen;
  }
  __device__ __forceinline__ void gather(const uint8_t (*flags)[4][64]) {
    const uint8_t(*f)[64] = flags[(t0 >> 6) & 1];
    const int all = f[0][lane] | f[1][lane] | f[2][lane] | f[3][lane];
    const int live = all & 15;
    // blocks before this tile (modulo 4), and the tile's block of this wave
    const int n = __builtin_popcount(live);
    const uint64_t b0 = __ballot(n & 1), b1 = __ballot(n & 2), below = (1ull << lane) - 1ull;
    const int before = cnt + __builtin_popcountll(b0 & below) + 2 * __builtin_popcountll(b1 & below);
    const int rank = (wave - before) & 3;
    const bool own = rank < n;
    int rest = live;
#pragma unroll
    for (int r = 0; r < 3; ++r) rest = rank > r ? rest & (rest - 1) : rest;
    const int j = own ? __builtin_ctz(rest) : 0;
    const int e = 4 * tile + j + (int)((uint32_t)(all >> (4 + j) & 1) << 31);
    // own lanes to the front, the others behind them
    const uint64_t mine = __ballot(own);
    const int dst = own ? __builtin_popcountll(mine & below)
                        : __builtin_popcountll(mine) + __builtin_popcountll(~mine & below);
    ent = __builtin_amdgcn_ds_permute(4 * dst, e);
    slot = __builtin_amdgcn_ds_permute(4 * dst, slot);
    m = uniform(__builtin_popcountll(mine));
    cnt = uniform((cnt + __builtin_popcountll(b0) + 2 * __builtin_popcountll(b1)) & 3);
    t0 += 64;
  }

  // Block i of the chunk: its first token, whether it has both allowed and
  // masked pairs (mixed), and this lane's mask word.  The load is issued for
  // every block (a conditional one would have to be waited for where its two
  // paths meet), but through a buffer of no size when the block is not mixed:
  // a full tile has no slot, and a row without partial tiles need not have a
  // valid kv_bits_off.
  __device__ __forceinline__ void block(int i, int& base, uint32_t& w, bool& mixed) const {
    const int e = __builtin_amdgcn_readlane(ent, i);
    const int s = __builtin_amdgcn_readlane(slot, i);
    base = 32 * (e & 0x7fffffff);
    mixed = e < 0;
    const auto bits = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(words + ((size_t)(uint32_t)s * kTileBitsWords + (e & 3))), 0,
        mixed ? 4 * (kTileBitsWords - 3) : 0, 0x00020000);
    w = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(bits, 4 * (int)woff, 0, 0);
  }
};

// Sums the four waves' accumulators through `red` (merge_floats<D>() floats of
// LDS) and stores this wave's share of the 32 owned rows, multiplied by `mul`:
// in pass h entries 8 h + 2 wave + {0, 1} of all tiles, 2 DT consecutive
// head dims of row n per lane.  Every wave calls it; the caller separates it
// from earlier use of `red` by a barrier.  Two passes rather than one halve
// the LDS, which else would hold the kernels at two work-groups per CU.
template <int D>
__device__ __forceinline__ constexpr int merge_floats() { return 4 * (D / 32) * 8 * 64; }

template <int D>
__device__ __forceinline__ void merge_store(float* red, const f32x16 (&acc)[D / 32], float mul,
                                            float* row, bool valid, int wave, int lane) {
  constexpr int DT = D / 32;
  f32x2* r2 = reinterpret_cast<f32x2*>(red) + lane;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    if (h) __syncthreads();
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        r2[((wave * DT + dt) * 4 + i) * 64] = f32x2{acc[dt][8 * h + 2 * i], acc[dt][8 * h + 2 * i + 1]};
    __syncthreads();
    f32x2 s[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      s[dt] = r2[(dt * 4 + wave) * 64];
#pragma unroll
      for (int u = 1; u < 4; ++u) s[dt] += r2[((u * DT + dt) * 4 + wave) * 64];
      s[dt] *= mul;
    }
    if (valid) {
      // acc_row(8 h + 2 wave + e, g)
      float* dst = row + DT * (16 * h + 8 * (wave >> 1) + 4 * (lane >> 5) + 2 * (wave & 1));
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        if constexpr (DT == 4)
          *reinterpret_cast<f32x4*>(dst + 4 * e) = f32x4{s[0][e], s[1][e], s[2][e], s[3][e]};
        else
          *reinterpret_cast<f32x2*>(dst + 2 * e) = f32x2{s[0][e], s[1][e]};
      }
    }
  }
}

}  // namespace f32
}  // namespace t2t
