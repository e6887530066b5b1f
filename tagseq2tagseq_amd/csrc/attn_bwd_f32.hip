// Masked flash-attention backward for float32 inputs, gfx950 fp32 MFMA.
//
// The float32 form of sdpa_dense_backward
// (torch/_higher_order_ops/flex_attention.py:825-994): P = exp(S - LSE),
// Delta = rowsum(O * dO), dS = P (dP - Delta) * scale, dQ = dS K,
// dK = dS^T Q (summed over each GQA group), dV = P^T dO; masked pairs and
// fully masked rows contribute nothing.  Every product and sum is float32; no
// atomics, and a fixed order of every sum, so the result is deterministic.
//
// Two launches: dQ (which also computes each of its rows' Delta and writes it
// out), then dK/dV, both with the decomposition of attn_f32.h: a work-group
// owns 32 queries (keys), whose rows sit in LDS, and deals the other side's
// 32-row blocks to its four waves.  A block is consumed as a run of units of
// 16 operand registers, each requested two units (2048 cycles of matrix pipe
// at D = 128) before it is contracted.
#include "attn_f32.h"

namespace t2t {

namespace {

struct BwdF32Params {
  const float* q; int64_t q_sb, q_sh, q_st;
  const float* k; int64_t k_sb, k_sh, k_st;
  const float* v; int64_t v_sb, v_sh, v_st;
  const float* o; int64_t o_sb, o_sh, o_st;
  const float* dout; int64_t do_sb, do_sh, do_st;
  float* dq; int64_t dq_sb, dq_sh, dq_st;
  float* dk; int64_t dk_sb, dk_sh, dk_st;
  float* dv; int64_t dv_sb, dv_sh, dv_st;
  const float* lse2;  // [B][Hq][T], log2 domain of scaled scores
  float* delta;       // [B][Hq][T]
  int B, Hq, Hkv, T;
  float scale, scale_log2;
  MaskTables m;
};

}  // namespace

// dQ (and Delta) of one (b, query head, 32 queries): S^T = K Q^T and
// dP^T = V dO^T with the queries in the lanes, dQ^T += K^T dS^T.
template <int D>
__global__ __launch_bounds__(kThreads, D == 64 ? 3 : 2) void bwd_dq_f32_kernel(BwdF32Params p) {
  constexpr int DT = D / 32;
  constexpr int P = f32::pitch<D>();
  constexpr int kOwn = f32::kRows * P;
  constexpr int kMerge = f32::merge_floats<D>();
  // Q and dO rows during the walk, the merge of the four dQ after it
  __shared__ __attribute__((aligned(16))) float lds[2 * kOwn > kMerge ? 2 * kOwn : kMerge];
  __shared__ float row_delta[32];
  __shared__ uint8_t flags[2][4][64];

  int h, y;
  head_and_slot(p.Hq, p.Hkv, 4 * p.m.nt, h, y);
  const int b = blockIdx.z;
  const int tid = threadIdx.x, wave = uniform(tid >> 6), lane = tid & 63;
  const int g = lane >> 5, n = lane & 31;
  const int hk = h / (p.Hq / p.Hkv);
  const int mb = p.m.Bm > 1 ? b : 0;
  const int T = p.T, nt = p.m.nt;
  const int qt = uniform(p.m.row_order[(size_t)mb * nt + (y >> 2)]);
  const int qloc = 32 * (3 - (y & 3)) + n;
  const int qrow = qt * kTile + qloc;
  if (qrow - n >= T) return;
  const bool qvalid = qrow < T;
  const size_t stat = ((size_t)b * p.Hq + h) * T;
  const float c = p.scale_log2;

  // Q, dO and O rows, requested before the tile list's chain of loads
  const int srow = tid >> 3, scol = 4 * (tid & 7);
  const int grow = qrow - n + srow;
  f32x4 q4[DT], d4[DT], o4[DT];
  {
    const float* qb = p.q + b * p.q_sb + h * p.q_sh + (int64_t)grow * p.q_st + scol;
    const float* db = p.dout + b * p.do_sb + h * p.do_sh + (int64_t)grow * p.do_st + scol;
    const float* ob = p.o + b * p.o_sb + h * p.o_sh + (int64_t)grow * p.o_st + scol;
#pragma unroll
    for (int i = 0; i < DT; ++i) {
      q4[i] = d4[i] = o4[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (grow < T) {
        q4[i] = *reinterpret_cast<const f32x4*>(qb + 32 * i);
        d4[i] = *reinterpret_cast<const f32x4*>(db + 32 * i);
        o4[i] = *reinterpret_cast<const f32x4*>(ob + 32 * i);
      }
    }
  }
  const float lrow = qvalid ? p.lse2[stat + qrow] : -INFINITY;
  const float neg_lse = lrow == -INFINITY ? -INFINITY : -lrow;

  const size_t row = (size_t)mb * nt + qt;
  f32::BlockWalk walk;
  walk.pidx = p.m.kv_idx + row * nt;
  walk.fidx = p.m.full_kv_idx + row * nt;
  walk.pslot = nullptr;
  walk.words = p.m.tile_bits + (size_t)uniform(p.m.kv_bits_off[row]) * kTileBitsWords;
  walk.woff = qloc * 4;
  walk.npart = uniform(p.m.kv_num[row]);
  walk.ntiles = walk.npart + uniform(p.m.full_kv_num[row]);
  walk.lane = lane;
  walk.wave = wave;
  walk.t0 = 0;
  walk.cnt = ((y >> 2) + y) & 3;
  walk.look((uint32_t)(qloc - n) * 4);
  const auto krs = f32::slice(p.k + b * p.k_sb + hk * p.k_sh, p.k_st, T, D);
  const auto vrs = f32::slice(p.v + b * p.v_sb + hk * p.v_sh, p.v_st, T, D);
  const int k_st4 = (int)p.k_st * 4, v_st4 = (int)p.v_st * 4;
  {
    // Delta = rowsum(O * dO): eight neighbouring threads hold a row
    float dl = 0.f;
#pragma unroll
    for (int i = 0; i < DT; ++i) {
      *reinterpret_cast<f32x4*>(lds + srow * P + scol + 32 * i) = q4[i];
      *reinterpret_cast<f32x4*>(lds + kOwn + srow * P + scol + 32 * i) = d4[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) dl = fmaf(o4[i][e], d4[i][e], dl);
    }
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) dl += __shfl_xor(dl, off, 64);
    if ((tid & 7) == 0) {
      row_delta[srow] = dl;
      if (grow < T) p.delta[stat + grow] = dl;
    }
  }
  walk.publish(flags);
  __syncthreads();
  walk.gather(flags);
  const float delta = row_delta[n];

  f32x16 dq[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) dq[dt] = f32x16{};

  // Units of a block: U of K rows (S), U of V rows (dP), 4 of K tokens (dQ).
  constexpr int U = D / 32, NU = 2 * U + 4;
  static_assert(NU % 4 == 0, "a block ends where the ring does");
  f32x4 x[4][4];  // ring: unit u in slot u % 4
  for (;;) {
    int base = 0, next;
    uint32_t w = 0, next_w;
    bool mixed = false, next_mixed;
    if (walk.m > 0) {
      walk.block(0, base, w, mixed);
      f32::load_row(x[0], krs, (base + n) * k_st4 + 16 * g, 0);
      f32::load_row(x[1], krs, (base + n) * k_st4 + 16 * g, 1);
    }
    for (int i = 0; i < walk.m; ++i) {
      int ln = lane;  // lane terms are made anew for each block (registers)
      asm volatile("" : "+v"(ln));
      const int g = ln >> 5, n = ln & 31;
      const float* q_own = lds + n * P + 4 * g;
      const float* do_own = q_own + kOwn;
      const int koff = n * k_st4 + 16 * g, voff = n * v_st4 + 16 * g;
      const int ktok = 4 * g * k_st4 + 4 * DT * n;
      f32::OwnPair own;
      f32::load_own(own, q_own, 0);
      f32x16 s = {}, dp = {};
      if (mixed) f32::seed_fill(s, ~w >> (4 * g));
      // (the last block's successor is itself: its rows are requested to no use)
      walk.block(min(i + 1, walk.m - 1), next, next_w, next_mixed);
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const int a = u + 2;  // unit to request
        if (a < U) f32::load_row(x[a & 3], krs, base * k_st4 + koff, a);
        else if (a < 2 * U) f32::load_row(x[a & 3], vrs, base * v_st4 + voff, a - U);
        else if (a < NU) f32::load_tok<D>(x[a & 3], krs, base * k_st4 + ktok, k_st4, a - 2 * U);
        else f32::load_row(x[a & 3], krs, next * k_st4 + koff, a - NU);
        if (u == 2 * U) {
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const float pv = fast_exp2(fmaf(s[e], c, neg_lse));
            dp[e] = pv * (dp[e] - delta);  // dS^T
          }
        }
        f32::fence();
        if (u < U) f32::dot_unit(s, x[u & 3], own, q_own, u == U - 1 ? do_own : nullptr, u);
        else if (u < 2 * U)
          f32::dot_unit(dp, x[u & 3], own, do_own, u == 2 * U - 1 ? do_own : nullptr, u - U);
        else f32::acc_unit<D>(dq, x[u & 3], dp, u - 2 * U);
        f32::fence();
      }
      base = next;
      w = next_w;
      mixed = next_mixed;
    }
    if (walk.t0 >= walk.ntiles) break;
    walk.look((uint32_t)(qloc - n) * 4);
    walk.publish(flags);
    __syncthreads();
    walk.gather(flags);
  }
  __syncthreads();  // Q and dO rows are no longer read
  f32::merge_store<D>(lds, dq, p.scale, p.dq + b * p.dq_sb + h * p.dq_sh + (int64_t)qrow * p.dq_st,
                      qvalid, wave, lane);
}

// dK, dV of one (b, kv head, 32 keys): S = Q K^T and dP = dO V^T with the
// keys in the lanes, dV^T += dO^T P, dK^T += Q^T dS, over every query head of
// the group and every query block of the column.
template <int D>
__global__ __launch_bounds__(kThreads, D == 64 ? 3 : 2) void bwd_dkdv_f32_kernel(BwdF32Params p) {
  constexpr int DT = D / 32;
  constexpr int P = f32::pitch<D>();
  constexpr int kOwn = f32::kRows * P;
  constexpr int kMerge = f32::merge_floats<D>();
  // K and V rows during the walk, then the merges of dK and of dV
  __shared__ __attribute__((aligned(16))) float lds[2 * kOwn > kMerge ? 2 * kOwn : kMerge];
  __shared__ __attribute__((aligned(16))) float stats[4][2][32];  // a wave's LSE and Delta
  __shared__ uint8_t flags[2][4][64];

  const int hk = blockIdx.x, b = blockIdx.z;
  const int tid = threadIdx.x, wave = uniform(tid >> 6), lane = tid & 63;
  const int g = lane >> 5, n = lane & 31;
  const int G = p.Hq / p.Hkv;
  const int mb = p.m.Bm > 1 ? b : 0;
  const int T = p.T, nt = p.m.nt;
  const int kt = uniform(p.m.col_order[(size_t)mb * nt + (blockIdx.y >> 2)]);
  const int kloc = 32 * (blockIdx.y & 3) + n;  // within a tile the earlier keys have more queries
  const int key = kt * kTile + kloc;
  if (key - n >= T) return;
  const bool kvalid = key < T;
  const float c = p.scale_log2;

  // K and V rows, requested before the tile list's chain of loads
  const int srow = tid >> 3, scol = 4 * (tid & 7);
  const int grow = key - n + srow;
  f32x4 k4[DT], v4[DT];
  {
    const float* kp = p.k + b * p.k_sb + hk * p.k_sh + (int64_t)grow * p.k_st + scol;
    const float* vp = p.v + b * p.v_sb + hk * p.v_sh + (int64_t)grow * p.v_st + scol;
#pragma unroll
    for (int i = 0; i < DT; ++i) {
      k4[i] = v4[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (grow < T) {
        k4[i] = *reinterpret_cast<const f32x4*>(kp + 32 * i);
        v4[i] = *reinterpret_cast<const f32x4*>(vp + 32 * i);
      }
    }
  }
  const size_t col = (size_t)mb * nt + kt;
  f32::BlockWalk walk;
  walk.pidx = p.m.q_idx + col * nt;
  walk.fidx = p.m.full_q_idx + col * nt;
  walk.pslot = p.m.q_bits_slot + col * nt;
  walk.words = p.m.tile_bits;
  walk.woff = kTile * 4 + kloc * 4;
  walk.npart = uniform(p.m.q_num[col]);
  walk.ntiles = walk.npart + uniform(p.m.full_q_num[col]);
  walk.lane = lane;
  walk.wave = wave;
  walk.t0 = 0;
  walk.cnt = ((blockIdx.y >> 2) + blockIdx.y) & 3;
  walk.look((uint32_t)(kTile + kloc - n) * 4);
#pragma unroll
  for (int i = 0; i < DT; ++i) {
    *reinterpret_cast<f32x4*>(lds + srow * P + scol + 32 * i) = k4[i];
    *reinterpret_cast<f32x4*>(lds + kOwn + srow * P + scol + 32 * i) = v4[i];
  }
  walk.publish(flags);
  __syncthreads();
  walk.gather(flags);

  f32x16 dk[DT], dv[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) { dk[dt] = f32x16{}; dv[dt] = f32x16{}; }
  const int q_st4 = (int)p.q_st * 4, d_st4 = (int)p.do_st * 4;

  for (int hh = 0; hh < G; ++hh) {
    const int h = hk * G + hh;
    const auto qrs = f32::slice(p.q + b * p.q_sb + h * p.q_sh, p.q_st, T, D);
    const auto drs = f32::slice(p.dout + b * p.do_sb + h * p.do_sh, p.do_st, T, D);
    // queries at or past T (masked) read an LSE and a Delta of zero
    const auto lrs = f32::row_stats(p.lse2 + ((size_t)b * p.Hq + h) * T, T);
    const auto ers = f32::row_stats(p.delta + ((size_t)b * p.Hq + h) * T, T);
    // Units of a block: U of Q rows (S), U of dO rows (dP), 4 of dO tokens
    // (dV), 4 of Q tokens (dK).
    constexpr int U = D / 32, NU = 2 * U + 8;
    static_assert(NU % 4 == 0, "a block ends where the ring does");
    f32x4 x[4][4];  // ring: unit u in slot u % 4
    for (;;) {
      int base = 0, next;
      uint32_t w = 0, next_w;
      bool mixed = false, next_mixed;
      float sl, sd;  // LSE and Delta of the block's query n
      // (without a block, block 0 of an empty list: tile 0, not used)
      walk.block(0, base, w, mixed);
      sl = f32::load1(lrs, 4 * (base + n));
      sd = f32::load1(ers, 4 * (base + n));
      f32::load_row(x[0], qrs, (base + n) * q_st4 + 16 * g, 0);
      f32::load_row(x[1], qrs, (base + n) * q_st4 + 16 * g, 1);
      for (int i = 0; i < walk.m; ++i) {
        // lane terms are made anew for each block: 128 of the 256 registers
        // are accumulators, and held across the loop these would spill
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int g = ln >> 5, n = ln & 31;
        const float* k_own = lds + n * P + 4 * g;
        const float* v_own = k_own + kOwn;
        const int qoff = n * q_st4 + 16 * g, doff = n * d_st4 + 16 * g;
        const int qtok = 4 * g * q_st4 + 4 * DT * n, dtok = 4 * g * d_st4 + 4 * DT * n;
        f32::OwnPair own;
        f32::load_own(own, k_own, 0);
        f32x16 s = {}, dp = {};
        if (mixed) f32::seed_fill(s, ~w >> (4 * g));
        // a fully masked row (LSE = -inf) has only -inf scores; clamping its
        // LSE keeps P at 0
        stats[wave][g][n] = g ? sd : fmaxf(sl, -3.402823466e38f);
        // (the last block's successor is itself: its rows are requested to no use)
        walk.block(min(i + 1, walk.m - 1), next, next_w, next_mixed);
        sl = f32::load1(lrs, 4 * (next + n));
        sd = f32::load1(ers, 4 * (next + n));
#pragma unroll
        for (int u = 0; u < NU; ++u) {
          const int a = u + 2;  // unit to request
          if (a < U) f32::load_row(x[a & 3], qrs, base * q_st4 + qoff, a);
          else if (a < 2 * U) f32::load_row(x[a & 3], drs, base * d_st4 + doff, a - U);
          else if (a < 2 * U + 4)
            f32::load_tok<D>(x[a & 3], drs, base * d_st4 + dtok, d_st4, a - 2 * U);
          else if (a < NU)
            f32::load_tok<D>(x[a & 3], qrs, base * q_st4 + qtok, q_st4, a - 2 * U - 4);
          else f32::load_row(x[a & 3], qrs, next * q_st4 + qoff, a - NU);
          if (u == 2 * U) {
            // P and dS; entry e is query base + acc_row(e, g)
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
              const f32x4 lse = *reinterpret_cast<const f32x4*>(&stats[wave][0][8 * e4 + 4 * g]);
              const f32x4 dl = *reinterpret_cast<const f32x4*>(&stats[wave][1][8 * e4 + 4 * g]);
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const int e = 4 * e4 + r;
                s[e] = fast_exp2(fmaf(s[e], c, -lse[r]));
                dp[e] = s[e] * (dp[e] - dl[r]);
              }
              f32::fence();
            }
          }
          f32::fence();
          if (u < U) f32::dot_unit(s, x[u & 3], own, k_own, u == U - 1 ? v_own : nullptr, u);
          else if (u < 2 * U)
            f32::dot_unit(dp, x[u & 3], own, v_own, u == 2 * U - 1 ? v_own : nullptr, u - U);
          else if (u < 2 * U + 4) f32::acc_unit<D>(dv, x[u & 3], s, u - 2 * U);
          else f32::acc_unit<D>(dk, x[u & 3], dp, u - 2 * U - 4);
          f32::fence();
        }
        base = next;
        w = next_w;
        mixed = next_mixed;
      }
      // the next 64 tiles, or the first ones for the next query head
      const bool over = walk.t0 >= walk.ntiles;
      if (over) {
        if (hh == G - 1 || walk.ntiles <= 64) break;
        walk.t0 = 0;
      }
      walk.look((uint32_t)(kTile + kloc - n) * 4);
      __syncthreads();
      walk.publish(flags);
      __syncthreads();
      walk.gather(flags);
      if (over) break;
    }
  }
  __syncthreads();  // K and V rows are no longer read
  f32::merge_store<D>(lds, dk, p.scale, p.dk + b * p.dk_sb + hk * p.dk_sh + (int64_t)key * p.dk_st,
                      kvalid, wave, lane);
  __syncthreads();
  f32::merge_store<D>(lds, dv, 1.f, p.dv + b * p.dv_sb + hk * p.dv_sh + (int64_t)key * p.dv_st,
                      kvalid, wave, lane);
}

hipError_t launch_attn_bwd_f32(const TensorView& q, const TensorView& k, const TensorView& v,
                               const TensorView& o, const TensorView& dout, const float* lse2,
                               float* delta, const TensorView& dq, const TensorView& dk,
                               const TensorView& dv, const AttnDims& dims, const MaskTables& mask,
                               hipStream_t stream) {
  BwdF32Params p;
  p.q = static_cast<const float*>(q.data); p.q_sb = q.sb; p.q_sh = q.sh; p.q_st = q.st;
  p.k = static_cast<const float*>(k.data); p.k_sb = k.sb; p.k_sh = k.sh; p.k_st = k.st;
  p.v = static_cast<const float*>(v.data); p.v_sb = v.sb; p.v_sh = v.sh; p.v_st = v.st;
  p.o = static_cast<const float*>(o.data); p.o_sb = o.sb; p.o_sh = o.sh; p.o_st = o.st;
  p.dout = static_cast<const float*>(dout.data);
  p.do_sb = dout.sb; p.do_sh = dout.sh; p.do_st = dout.st;
  p.dq = static_cast<float*>(dq.data); p.dq_sb = dq.sb; p.dq_sh = dq.sh; p.dq_st = dq.st;
  p.dk = static_cast<float*>(dk.data); p.dk_sb = dk.sb; p.dk_sh = dk.sh; p.dk_st = dk.st;
  p.dv = static_cast<float*>(dv.data); p.dv_sb = dv.sb; p.dv_sh = dv.sh; p.dv_st = dv.st;
  p.lse2 = lse2;
  p.delta = delta;
  p.B = dims.B; p.Hq = dims.Hq; p.Hkv = dims.Hkv; p.T = dims.T;
  p.scale = dims.scale;
  p.scale_log2 = dims.scale * kLog2e;
  p.m = mask;
  if (mask.nt == 0 || dims.B == 0 || dims.Hq == 0) return hipSuccess;
  const bool d64 = dims.D == 64;
  const dim3 gq(dims.Hq, 4 * mask.nt, dims.B), gk(dims.Hkv, 4 * mask.nt, dims.B);
  if (d64) hipLaunchKernelGGL(bwd_dq_f32_kernel<64>, gq, dim3(kThreads), 0, stream, p);
  else hipLaunchKernelGGL(bwd_dq_f32_kernel<128>, gq, dim3(kThreads), 0, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (d64) hipLaunchKernelGGL(bwd_dkdv_f32_kernel<64>, gk, dim3(kThreads), 0, stream, p);
  else hipLaunchKernelGGL(bwd_dkdv_f32_kernel<128>, gk, dim3(kThreads), 0, stream, p);
  return hipGetLastError();
}

}  // namespace t2t
