// Masked flash-attention forward for float32 inputs, gfx950 fp32 MFMA.
//
// The float32 form of the reference's math_attention
// (torch/_higher_order_ops/flex_attention.py:202-267): S = Q K^T * scale,
// P = softmax of the masked row, O = P V with P kept in float32 (the
// reference's P.to(dtype) is a no-op for float32), fully masked rows giving
// O = 0 and LSE = -inf.  Every product and sum is float32.
//
// One work-group per (b, query head, 32 queries), the key blocks dealt to its
// four waves (attn_f32.h); each wave keeps its own running max, sum and O,
// merged at the end.  S^T = K Q^T (keys in the accumulator rows, queries in
// the lanes), lazily rescaled softmax in the log2 domain, O^T += V^T P^T.
#include "attn_f32.h"

namespace t2t {

namespace {

struct FwdF32Params {
  const float* q; int64_t q_sb, q_sh, q_st;
  const float* k; int64_t k_sb, k_sh, k_st;
  const float* v; int64_t v_sb, v_sh, v_st;
  float* o; int64_t o_sb, o_sh, o_st;
  float* lse2;
  int B, Hq, Hkv, T;
  float scale_log2;
  MaskTables m;
};

}  // namespace

template <int D>
__global__ __launch_bounds__(kThreads, 3) void attn_fwd_f32_kernel(FwdF32Params p) {
  constexpr int DT = D / 32;
  constexpr int P = f32::pitch<D>();
  // Q rows during the walk, the merge of the four O accumulators after it
  constexpr int kOwn = f32::kRows * P, kMerge = f32::merge_floats<D>();
  __shared__ __attribute__((aligned(16))) float lds[kOwn > kMerge ? kOwn : kMerge];
  __shared__ float stat[2][4][32];  // running max and sum per wave and query
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
  const int qloc = 32 * (3 - (y & 3)) + n;  // within a tile the later queries see more keys
  const int qrow = qt * kTile + qloc;
  if (qrow - n >= T) return;
  const bool qvalid = qrow < T;
  const float c = p.scale_log2;

  // Q rows, requested before the tile list's chain of loads
  const int srow = tid >> 3, scol = 4 * (tid & 7);
  f32x4 q4[DT];
  {
    const float* qb = p.q + b * p.q_sb + h * p.q_sh + (int64_t)(qrow - n + srow) * p.q_st + scol;
#pragma unroll
    for (int i = 0; i < DT; ++i) {
      q4[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (qrow - n + srow < T) q4[i] = *reinterpret_cast<const f32x4*>(qb + 32 * i);
    }
  }
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
  walk.cnt = ((y >> 2) + y) & 3;  // no wave, hence no SIMD, always takes the odd blocks
  walk.look((uint32_t)(qloc - n) * 4);
  const auto krs = f32::slice(p.k + b * p.k_sb + hk * p.k_sh, p.k_st, T, D);
  const auto vrs = f32::slice(p.v + b * p.v_sb + hk * p.v_sh, p.v_st, T, D);
  const int k_st4 = (int)p.k_st * 4, v_st4 = (int)p.v_st * 4;
#pragma unroll
  for (int i = 0; i < DT; ++i)
    *reinterpret_cast<f32x4*>(lds + srow * P + scol + 32 * i) = q4[i];
  walk.publish(flags);
  __syncthreads();
  walk.gather(flags);

  f32x16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) oacc[dt] = f32x16{};
  float m_ref = -INFINITY, l_run = 0.f;

  // Units of a block: U of K rows (S), 4 of V tokens (P V).
  constexpr int U = D / 32, NU = U + 4, R = NU % 4 ? 3 : 4;
  static_assert(NU % R == 0, "a block ends where the ring does");
  f32x4 x[R][4];  // ring: unit u in slot u % R
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
      // lane terms are made anew for each block: held across the loop they
      // would take the kernel past the 168 registers of three waves per SIMD
      int ln = lane;
      asm volatile("" : "+v"(ln));
      const int g = ln >> 5, n = ln & 31;
      const float* own = lds + n * P + 4 * g;
      const int koff = n * k_st4 + 16 * g, voff = 4 * g * v_st4 + 4 * DT * n;
      f32::OwnPair qx;
      f32::load_own(qx, own, 0);
      f32x16 st = {};
      if (mixed) f32::seed_fill(st, ~w >> (4 * g));
      // (the last block's successor is itself: its rows are requested to no use)
      walk.block(min(i + 1, walk.m - 1), next, next_w, next_mixed);
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const int a = u + 2;  // unit to request
        if (a < U) f32::load_row(x[a % R], krs, base * k_st4 + koff, a);
        else if (a < NU) f32::load_tok<D>(x[a % R], vrs, base * v_st4 + voff, v_st4, a - U);
        else f32::load_row(x[a % R], krs, next * k_st4 + koff, a - NU);
        if (u == U) {
          float mx = st[0];
#pragma unroll
          for (int e = 1; e < 16; ++e) mx = fmaxf(mx, st[e]);
          mx = halves_max(mx);
          const bool move = (mx - m_ref) * c > 8.f;
          if (__ballot(move) != 0ull) {
            const float alpha = move ? fast_exp2((m_ref - mx) * c) : 1.f;
            l_run *= alpha;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) oacc[dt] *= alpha;
            m_ref = move ? mx : m_ref;
          }
          const float neg = m_ref == -INFINITY ? 0.f : -m_ref * c;
          float rs = 0.f;
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            st[e] = fast_exp2(fmaf(st[e], c, neg));
            rs += st[e];
          }
          l_run += rs;  // over the lane's own half of the keys
        }
        f32::fence();
        if (u < U) f32::dot_unit(st, x[u % R], qx, own, u == U - 1 ? own : nullptr, u);
        else f32::acc_unit<D>(oacc, x[u % R], st, u - U);
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

  // Merge: each wave's O and sum brought to the largest running max.
  l_run = halves_sum(l_run);
  if (g == 0) {
    stat[0][wave][n] = m_ref;
    stat[1][wave][n] = l_run;
  }
  __syncthreads();  // Q rows are no longer read either
  float m_all = stat[0][0][n];
#pragma unroll
  for (int u = 1; u < 4; ++u) m_all = fmaxf(m_all, stat[0][u][n]);
  float l_all = 0.f;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float mu = stat[0][u][n];  // -inf: the wave saw no allowed pair of this query
    if (mu != -INFINITY) l_all += stat[1][u][n] * fast_exp2((mu - m_all) * c);
  }
  const float alpha = m_ref == -INFINITY ? 0.f : fast_exp2((m_ref - m_all) * c);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) oacc[dt] *= alpha;
  const float inv_l = l_all > 0.f ? 1.f / l_all : 0.f;
  f32::merge_store<D>(lds, oacc, inv_l, p.o + b * p.o_sb + h * p.o_sh + (int64_t)qrow * p.o_st,
                      qvalid, wave, lane);
  if (qvalid && tid < 32)
    p.lse2[((size_t)b * p.Hq + h) * T + qrow] =
        l_all > 0.f ? m_all * c + __log2f(l_all) : -INFINITY;
}

hipError_t launch_attn_fwd_f32(const TensorView& q, const TensorView& k, const TensorView& v,
                               const TensorView& o, float* lse2, const AttnDims& dims,
                               const MaskTables& mask, hipStream_t stream) {
  FwdF32Params p;
  p.q = static_cast<const float*>(q.data); p.q_sb = q.sb; p.q_sh = q.sh; p.q_st = q.st;
  p.k = static_cast<const float*>(k.data); p.k_sb = k.sb; p.k_sh = k.sh; p.k_st = k.st;
  p.v = static_cast<const float*>(v.data); p.v_sb = v.sb; p.v_sh = v.sh; p.v_st = v.st;
  p.o = static_cast<float*>(o.data); p.o_sb = o.sb; p.o_sh = o.sh; p.o_st = o.st;
  p.lse2 = lse2;
  p.B = dims.B; p.Hq = dims.Hq; p.Hkv = dims.Hkv; p.T = dims.T;
  p.scale_log2 = dims.scale * kLog2e;
  p.m = mask;
  if (mask.nt == 0 || dims.B == 0 || dims.Hq == 0) return hipSuccess;
  dim3 grid(dims.Hq, 4 * mask.nt, dims.B);
  if (dims.D == 64)
    hipLaunchKernelGGL(attn_fwd_f32_kernel<64>, grid, dim3(kThreads), 0, stream, p);
  else
    hipLaunchKernelGGL(attn_fwd_f32_kernel<128>, grid, dim3(kThreads), 0, stream, p);
  return hipGetLastError();
}

}  // namespace t2t
