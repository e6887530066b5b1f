// Linear maps of a short sequence: y = x W^T (x [M][K], W [N][K]) and the
// input gradient dx = dy W (dy [M][K], W [K][N]), bf16 rows, fp32 sums, one
// rounding.  These are the projections of the layers (tunalab
// FlexSelfAttention's qkv and out-projection, GLU's gate_up and down, called
// from model/modules/layer.py:33-35) at up to a few thousand tokens.
//
// What bounds them: at 2048 tokens a product is 2 to 13 GFLOP, 2 to 10 us of
// matrix pipe, over 100 to 500 tiles -- the copies' latency and, per call, the
// host: the library's product costs 23 us of host time (its algorithm lookup),
// more than its kernel takes at these sizes, this one 6.  A work-group
// computes one BM x BN tile (tokens x features), 4 waves of a quarter each,
// from kStages stages of BK columns of both operands in LDS: direct
// global -> LDS copies run a stage or more ahead of the contraction, one
// barrier a stage.  The copies cannot pad a row, so its 16-byte chunks are
// XOR-swizzled by the row instead, which spreads the 16 rows of a row read
// (and the 4 x 64 bytes of a column read) over all banks.  Features are the
// MFMA's M side, so that a lane's four consecutive accumulators are four
// features of one token; the tile leaves through LDS in whole 16-byte pieces.
//
// Kernel times in a graph of such calls, against the library's [us]; the
// tiles are chosen in launch():
//   tokens x features x width   forward       input gradient (width <- features)
//   512 x 1536 x 512            4.9 /  6.5     9.0 /  8.9
//   2048 x 768 x 768            7.1 /  8.8     7.7 / 11.4
//   2048 x 2304 x 768          15.0 / 16.3    18.0 / 24.3
//   2048 x 768 x 2048          12.7 / 14.3    13.2 / 13.1
//   2048 x 4096 x 768          21.1 / 18.3    27.2 / 39.0
//   4096 x 2304 x 768          24.1 / 19.5    24.8 / 28.0
//   16384 x 2304 x 768         70.9 / 69.8    66.5 / 57.0
// Up to about 2000 x 4096 x 768 a call here takes no longer than the library's
// host side; beyond, the library's kernel is ahead (short_product in linear.py).
#include "lds_tiles.h"

namespace t2t {

namespace {

struct LinearArgs {
  const __bf16* x;  // tokens [M][K], row stride xs
  const __bf16* w;  // NT: features [N][K]; NN: [K][N]; row stride ws
  __bf16* y;        // [M][N], row stride ys
  int64_t xs, ws, ys;
  int M, N, K;
};

}  // namespace

template <int BM, int BN, int BK, int kStages, bool NN>
__global__ __launch_bounds__(kThreads, 2) void linear_kernel(LinearArgs p) {
  constexpr int WM = BM / 2, WN = BN / 2;      // a wave's tokens x features
  constexpr int MI = WM / 32, NI = WN / 32;
  constexpr int kTokBytes = BM * BK * 2, kFeatBytes = BN * BK * 2;
  constexpr int kStage = kTokBytes + kFeatBytes;
  constexpr int kPitch = BN + 8;               // of the output tile in LDS
  constexpr int kLds = kStages * kStage > BM * kPitch * 2 ? kStages * kStage : BM * kPitch * 2;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kLds];

  // consecutive tiles (features fastest) to one XCD: they share token rows,
  // and its L2 keeps the weight
  const int tiles_n = (p.N + BN - 1) / BN;
  const int G = gridDim.x, b = blockIdx.x;
  const int q = G / 8, rem = G % 8, xcd = b % 8;
  const int id = xcd * q + (xcd < rem ? xcd : rem) + b / 8;
  const int m0 = (id / tiles_n) * BM, n0 = (id % tiles_n) * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int g = lane >> 5, n = lane & 31;
  const int wm = (wave >> 1) * WM, wn = (wave & 1) * WN;

  const u32x4 xr = rsrc_words(p.x, ((int64_t)(p.M - 1) * p.xs + p.K) * 2);
  const u32x4 wr = rsrc_words(p.w, ((int64_t)((NN ? p.K : p.N) - 1) * p.ws + (NN ? p.N : p.K)) * 2);
  RowTile<BK, BM> xt;
  xt.init(m0, p.xs, wave, lane);
  std::conditional_t<NN, ColTile<BK, BN>, RowTile<BK, BN>> wt;
  if constexpr (NN) wt.init(n0, p.N, p.ws, wave, lane);
  else wt.init(n0, p.ws, wave, lane);
  constexpr int kCopies = decltype(xt)::kPerWave + decltype(wt)::kPerWave;
  const uint32_t base = lds_u32(lds);
  // (stages past K copy nothing and write zeros, so that every stage counts
  // the same number of copies)
  auto copy_stage = [&](int s) {
    const uint32_t at = base + (s % kStages) * kStage;
    xt.copy(at, xr, s * BK, p.K, wave);
    if constexpr (NN) wt.copy(at + kTokBytes, wr, s * BK, p.K, p.ws, wave);
    else wt.copy(at + kTokBytes, wr, s * BK, p.K, wave);
  };

  f32x16 acc[NI][MI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j) acc[i][j] = f32x16{};

  const int steps = (p.K + BK - 1) / BK;
#pragma unroll
  for (int s = 0; s < kStages - 1; ++s) copy_stage(s);
  for (int s = 0; s < steps; ++s) {
    // stage s has landed everywhere, and its predecessor's buffer is free
    vm_barrier<(kStages - 2) * kCopies>();
    copy_stage(s + kStages - 1);
    const uint8_t* xs = lds + (s % kStages) * kStage;
    const uint8_t* ws = xs + kTokBytes;
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      bf16x8 bx[MI], aw[NI];
#pragma unroll
      for (int j = 0; j < MI; ++j) {
        const int r = wm + 32 * j + n;
        bx[j] = *reinterpret_cast<const bf16x8*>(xs + r * BK * 2 +
                                                 16 * swizzle<BK>(r, 2 * kk + g));
      }
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if constexpr (NN) {
          aw[i] = read_col8<BN>(ws, 16 * kk, wn + 32 * i, lane);
        } else {
          const int r = wn + 32 * i + n;
          aw[i] = *reinterpret_cast<const bf16x8*>(ws + r * BK * 2 +
                                                   16 * swizzle<BK>(r, 2 * kk + g));
        }
      }
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < MI; ++j) acc[i][j] = mfma32(aw[i], bx[j], acc[i][j]);
    }
  }

  // acc[i][j] entry e: feature wn + 32 i + acc_row(e, g) of token wm + 32 j + n
  vm_barrier<0>();  // the last copies have landed, the last stage is read
  __bf16* out = reinterpret_cast<__bf16*>(lds);
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bf16x4 v;
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = (__bf16)acc[i][j][4 * e + u];
        *reinterpret_cast<bf16x4*>(out + (wm + 32 * j + n) * kPitch + wn + 32 * i + 8 * e +
                                   4 * g) = v;
      }
  __syncthreads();
  const bool whole = (p.ys % 8) == 0 && (reinterpret_cast<uintptr_t>(p.y) & 15) == 0;
#pragma unroll 4
  for (int c = tid; c < BM * BN / 8; c += kThreads) {
    const int r = c / (BN / 8), col = 8 * (c % (BN / 8));
    if (m0 + r >= p.M || n0 + col >= p.N) continue;
    const bf16x8 v = *reinterpret_cast<const bf16x8*>(out + r * kPitch + col);
    __bf16* dst = p.y + (int64_t)(m0 + r) * p.ys + n0 + col;
    if (whole && n0 + col + 8 <= p.N) {
      *reinterpret_cast<bf16x8*>(dst) = v;
    } else {
      for (int u = 0; u < 8 && n0 + col + u < p.N; ++u) dst[u] = v[u];
    }
  }
}

namespace {

template <int BM, int BN, int BK, int kStages, bool NN>
void launch_tiles(const LinearArgs& p, hipStream_t stream) {
  const int64_t tiles = (int64_t)((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
  hipLaunchKernelGGL((linear_kernel<BM, BN, BK, kStages, NN>), dim3((unsigned)tiles),
                     dim3(kThreads), 0, stream, p);
}

// The largest tile that still gives every CU work: 128 x 128 from two tiles
// per CU (2048 x 4096 x 768: 21.1 us, 24.1 with 128 x 64; 2048 x 3072 x 1024,
// 1.5 tiles per CU: 20.5 and 19.8), else 128 x 64 from one per CU (4096 x 768
// x 768: 9.8 us, 12.3 with 64 x 64; 2048 x 768 x 2048, 0.75 per CU: 16.0 and
// 12.7), else 64 x 64.  Two deep stages beat four shallow ones wherever a
// second work-group shares the CU (16384 x 2304 x 768: 70.9 against 89.1 us);
// the gradient's 64 x 64 tiles, with their long contractions, want four
// (512 x 768 x 4096: 19.5 against 24.6).
template <bool NN>
hipError_t launch(const LinearArgs& p, hipStream_t stream) {
  const int64_t m128 = (p.M + 127) / 128;
  if (m128 * ((p.N + 127) / 128) >= 512) launch_tiles<128, 128, 64, 2, NN>(p, stream);
  else if (m128 * ((p.N + 63) / 64) >= 256) launch_tiles<128, 64, 64, 2, NN>(p, stream);
  else if (NN) launch_tiles<64, 64, 64, 4, NN>(p, stream);
  else launch_tiles<64, 64, 128, 2, NN>(p, stream);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_linear(bool nn, const __bf16* x, int64_t xs, const __bf16* w, int64_t ws,
                         __bf16* y, int64_t ys, int M, int N, int K, hipStream_t stream) {
  if (M == 0 || N == 0) return hipSuccess;
  const LinearArgs p{x, w, y, xs, ws, ys, M, N, K};
  return nn ? launch<true>(p, stream) : launch<false>(p, stream);
}

}  // namespace t2t
