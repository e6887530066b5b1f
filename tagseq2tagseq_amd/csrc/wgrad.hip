// Weight gradient of a linear map over many rows: C[m][n] = sum_k A[k][m] B[k][n]
// (dW = dY^T X for y = x W^T, with dY [K][M] and X [K][N] row-major bf16).
//
// At K = 16384 rows, M x N = 768 x 768 ... 4096 x 768, the output has only
// 36-192 tiles of 128 x 128, too few for 256 CUs, and the library products run
// at 0.2-0.7 PFLOP/s.  Here K is split: work-group (tile, s) contracts the
// s-th of S nearly equal ranges of 64-row steps into an fp32 partial, and a
// second launch sums the S partials of each element in a fixed order
// (deterministic, no atomics) and rounds once.
//
// Both operands are "column" operands of v_mfma_f32_32x32x16_bf16 (the
// contraction runs over the rows of both tiles), read from LDS tiles [64
// rows][128] by ds_read_b64_tr_b16 pairs.  4 waves, each a 64 x 64 quarter of
// the tile (2 x 2 MFMA blocks); two stages of both tiles (64 KiB: two
// work-groups per CU), refilled by direct global -> LDS copies a step ahead,
// one barrier a step of 64 rows.
//
// Bound by LDS: a wave's four MFMA of a 16-row slice (128 cycles) read 4 KiB,
// the four waves' reads alone all of the 128 bytes a cycle that LDS gives,
// beside 8 KiB of copies.  Against 32-row steps staged through registers into
// padded rows (us before / now, both launches):
//              K = 2048      K = 8192      K = 16384
//   768 x 768   21.2 / 15.0   29.7 / 24.6   43.7 / 34
//   2304 x 768  30.2 / 24.7   59.9 / 46    103.4 / 80
//   768 x 2048  27.7 / 21.6   49.4 / 42     83.2 / 72
//   4096 x 768  34.0 / 28.7   83.7 / 74    148.4 / 134
// 256 x 128 tiles (two thirds of the LDS reads) took 122 us for the last and
// 5 to 40 % longer everywhere else; three or four 32-row buffers the same.
#include "lds_tiles.h"

namespace t2t {

namespace {

constexpr int kWgTile = 128;     // output tile edge
constexpr int kWgRows = 64;      // rows (K) per step
constexpr int kWgThreads = 256;

struct WgradArgs {
  const __bf16* a;  // [K][lda]
  const __bf16* b;  // [K][ldb]
  float* part;      // [S][M][N]
  int64_t lda, ldb;
  int M, N, K, S;
};

__global__ __launch_bounds__(kWgThreads, 2) void wgrad_kernel(WgradArgs p) {
  constexpr int kTileBytes = kWgRows * kWgTile * 2;
  constexpr int kCopies = kTileBytes / 1024 / kWaves;  // a tile's, per wave
  __shared__ __attribute__((aligned(1024))) uint8_t lds[2][2][kTileBytes];
  const int tiles_n = p.N / kWgTile;
  const int tiles = (p.M / kWgTile) * tiles_n;
  // The hardware hands work-groups to the 8 XCDs round-robin; give each XCD
  // a contiguous range of (split, tile) ids instead, so that the work-groups
  // sharing a row range of A and B (one split, neighbouring tiles) share an
  // L2.
  const int G = tiles * p.S, q = G / 8, rem = G % 8, xcd = blockIdx.x % 8;
  const int id = xcd * q + (xcd < rem ? xcd : rem) + blockIdx.x / 8;
  const int tile = id % tiles, s = id / tiles;
  const int m0 = (tile / tiles_n) * kWgTile, n0 = (tile % tiles_n) * kWgTile;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;  // this wave's quarter
  const int units = p.K / kWgRows;
  const int u0 = (int)((int64_t)s * units / p.S), u1 = (int)((int64_t)(s + 1) * units / p.S);

  // This lane's 16 bytes of each copy (four tile rows a copy), a step further
  // each time; M, N and K are whole tiles, so every copy is in bounds.
  const __bf16 *pa[kCopies], *pb[kCopies];
#pragma unroll
  for (int i = 0; i < kCopies; ++i) {
    const int r = (wave + kWaves * i) * 4 + lane / 16;
    const int c = 8 * col_swizzle<kWgTile>(r, lane % 16);
    const int64_t k = (int64_t)u0 * kWgRows + kperm(r);
    pa[i] = p.a + k * p.lda + m0 + c;
    pb[i] = p.b + k * p.ldb + n0 + c;
  }
  const uint32_t base = lds_u32(lds);
  auto copy_step = [&](int buf) {
    const uint32_t to = base + buf * 2 * kTileBytes + wave * 1024;
#pragma unroll
    for (int i = 0; i < kCopies; ++i) {
      lds_copy16_at(to + kWaves * i * 1024, pa[i]);
      lds_copy16_at(to + kTileBytes + kWaves * i * 1024, pb[i]);
      pa[i] += kWgRows * p.lda;
      pb[i] += kWgRows * p.ldb;
    }
  };

  // Two sums, of the even and of the odd 16-row slices: half the rounding
  // steps in a row, at no cost (registers are free at two waves a SIMD).
  f32x16 acc[2][2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[h][i][j] = f32x16{};
  if (u0 < u1) copy_step(0);
  for (int u = u0; u < u1; ++u) {
    const int buf = (u - u0) & 1;
    vm_barrier<0>();  // step u has landed everywhere, the other buffer is read
    if (u + 1 < u1) copy_step(buf ^ 1);
#pragma unroll
    for (int kk = 0; kk < kWgRows / 16; ++kk) {
      bf16x8 av[2], bv[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        av[i] = read_col8<kWgTile>(lds[buf][0], 16 * kk, wm + 32 * i, lane);
        bv[i] = read_col8<kWgTile>(lds[buf][1], 16 * kk, wn + 32 * i, lane);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[kk & 1][i][j] = mfma32(av[i], bv[j], acc[kk & 1][i][j]);
    }
  }

  // C layout: lane l, entry i -> row acc_row(i, l / 32), column l % 32
  float* out = p.part + (int64_t)s * p.M * p.N;
  const int g = lane >> 5, c = lane & 31;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + wm + 32 * i + acc_row(e, g);
        const int n = n0 + wn + 32 * j + c;
        out[(int64_t)m * p.N + n] = acc[0][i][j][e] + acc[1][i][j][e];
      }
}

// out[m][n] = sum over s (in order) of part[s][m][n]; 4 elements per thread.
__global__ __launch_bounds__(kWgThreads) void wgrad_sum_kernel(const float* part, int S,
                                                               int64_t mn, void* out,
                                                               bool out_f32) {
  const int64_t i4 = ((int64_t)blockIdx.x * kWgThreads + threadIdx.x) * 4;
  if (i4 >= mn) return;
  float4 acc = *reinterpret_cast<const float4*>(part + i4);
#pragma unroll 4
  for (int s = 1; s < S; ++s) {
    const float4 v = *reinterpret_cast<const float4*>(part + (int64_t)s * mn + i4);
    acc.x += v.x;
    acc.y += v.y;
    acc.z += v.z;
    acc.w += v.w;
  }
  if (out_f32) {
    *reinterpret_cast<float4*>(static_cast<float*>(out) + i4) = acc;
  } else {
    bf16x4 o;
    o[0] = (__bf16)acc.x;
    o[1] = (__bf16)acc.y;
    o[2] = (__bf16)acc.z;
    o[3] = (__bf16)acc.w;
    *reinterpret_cast<bf16x4*>(static_cast<__bf16*>(out) + i4) = o;
  }
}

}  // namespace

// The split count of least time, in steps of 64 rows: the rounds of the 512
// work-groups that run at once (each its steps and about six of start and
// end), the partials' way to memory and back (128 KiB a work-group) and the
// second launch's walk over them.  768 x 768: K = 2048 S = 4 14.8 us (8: 18.9),
// K = 16384 S = 14 33 us (8: 39); 4096 x 768 K = 16384 S = 5 129 us (2: 129).
int wgrad_splits(int M, int N, int K) {
  const int64_t tiles = (int64_t)(M / kWgTile) * (N / kWgTile);
  const int64_t units = K / kWgRows;
  int best = 1;
  double least = 0;
  for (int64_t S = 1; S <= units && S <= 64; ++S) {
    const double t = (double)((tiles * S + 511) / 512) * (double)((units + S - 1) / S + 6) +
                     0.022 * (double)(tiles * S) + 0.4 * (double)S;
    if (S == 1 || t < least) {
      least = t;
      best = (int)S;
    }
  }
  return best;
}

hipError_t launch_wgrad(const __bf16* a, int64_t lda, const __bf16* b, int64_t ldb, float* part,
                        void* out, bool out_f32, int M, int N, int K, hipStream_t stream) {
  const int S = wgrad_splits(M, N, K);
  WgradArgs p{a, b, part, lda, ldb, M, N, K, S};
  const int64_t tiles = (int64_t)(M / kWgTile) * (N / kWgTile);
  hipLaunchKernelGGL(wgrad_kernel, dim3((unsigned)(tiles * S)), dim3(kWgThreads), 0, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t mn = (int64_t)M * N;
  const int64_t blocks = (mn / 4 + kWgThreads - 1) / kWgThreads;
  hipLaunchKernelGGL(wgrad_sum_kernel, dim3((unsigned)blocks), dim3(kWgThreads), 0, stream, part,
                     S, mn, out, out_f32);
  return hipGetLastError();
}

}  // namespace t2t
