// Cross-entropy rows of a linear head, loss and gradient in one pass over the
// logits: for each row r of bf16 logits x (columns 0 .. V-1 of a row of ld),
//   loss[r] = logsumexp(x) - x[t]                        (t = target[r])
//   grad[r][j] = (softmax(x)[j] - [j == t]) * scale       (bf16, j < V)
//   grad[r][j] = 0                                        (V <= j < ld)
// with rows whose target equals ignore_index giving loss 0 and a zero
// gradient.  This is the per-chunk work of the reference's FusedLinearCELoss
// (tunalab, a Liger-style fused linear cross-entropy; constructed at
// model/modules/training_module.py:127-133 and called at :209): torch's
// F.cross_entropy(logits.float(), targets, ignore_index, reduction="sum") and
// its backward, with the gradient produced in the forward so the head's
// products for dX and dW follow without recomputing the logits.
//
// HBM bound: the row is read once and its gradient written once.  A row of up
// to 65536 columns is held in the registers of a 1024-thread work-group (1 to
// 8 pieces of 8 logits per thread; 7 and 28 registers at V = 50257, so that
// two such work-groups, 32 waves, run on a CU: one loads while the other
// computes or writes).  Row maximum, then the sum of exp2 against it, each
// combined across the wave by shuffles and across the waves through LDS; the
// gradient may overwrite the logits in place, since every read of a row
// happens before the barriers that precede its writes.  16384 rows of 50264:
// 933 -> 614 us, 5.4 TB/s, which is the rate of a large copy on this card
// (5.2 TB/s); 8192 rows of 40000 columns 356 -> 241 us, of 20000 201 -> 129
// us.  Wider rows are read twice, with a running (max, sum) per lane, and so
// are short ones, where 1024 threads have nothing to hold (16384 rows of 1000
// columns: 79 us read twice, 83 us held; of 4096: 124 and 93 us).
#include "attn_kernels.h"

namespace t2t {

namespace {

constexpr int kCeThreads = 512;
constexpr int kCeWaves = kCeThreads / 64;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  const __bf16 lo = (__bf16)a, hi = (__bf16)b;
  return (uint32_t)__builtin_bit_cast(uint16_t, lo) |
         ((uint32_t)__builtin_bit_cast(uint16_t, hi) << 16);
}

// (max, sum) pairs in log2 units: sum of exp2(v - max) over the values seen.
__device__ __forceinline__ void lse_add(float& m, float& s, float v) {
  if (v > m) {
    s = s * exp2f(m - v) + 1.f;
    m = v;
  } else {
    s += exp2f(v - m);
  }
}

__device__ __forceinline__ void lse_merge(float& m, float& s, float m2, float s2) {
  const float mm = fmaxf(m, m2);
  if (mm == -INFINITY) return;  // both empty
  s = s * exp2f(m - mm) + s2 * exp2f(m2 - mm);
  m = mm;
}

constexpr int kRegThreads = 1024;
constexpr int kRegWaves = kRegThreads / 64;

// Combines x over the work-group (every thread gets the result); red: LDS of
// kRegWaves floats, not in use by an earlier call.
template <bool Max>
__device__ __forceinline__ float wg_combine(float x, float* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float y = __shfl_xor(x, off, 64);
    x = Max ? fmaxf(x, y) : x + y;
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  float r = red[0];
#pragma unroll
  for (int w = 1; w < kRegWaves; ++w) r = Max ? fmaxf(r, red[w]) : r + red[w];
  return r;
}

// Makes the compiler unpack the row anew in each phase: 56 unpacked logits
// held from one to the next would spill.
template <int NP>
__device__ __forceinline__ void phase(uint4 (&q)[NP]) {
#pragma unroll
  for (int p = 0; p < NP; ++p)
    asm volatile("" : "+v"(q[p].x), "+v"(q[p].y), "+v"(q[p].z), "+v"(q[p].w));
}

// Rows of at most NP * 8 * kRegThreads columns.
template <int NP>
__global__ __launch_bounds__(kRegThreads, 8) void ce_rows_reg_kernel(
    const uint16_t* logits, uint16_t* grad, int64_t ld, int V,
    const int64_t* __restrict__ target, int64_t ignore_index, const float* __restrict__ scale,
    float* __restrict__ row_loss) {
  __shared__ float red[2][kRegWaves];
  const int64_t row = blockIdx.x;
  const uint4* x = reinterpret_cast<const uint4*>(logits + row * ld);
  const int nvec = (int)(ld / 8);
  uint4 q[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int i = threadIdx.x + p * kRegThreads;
    // columns past the row hold -inf: no share of the maximum or the sum
    q[p] = make_uint4(0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u);
    if (i < nvec) q[p] = x[i];
    if (i < nvec && 8 * i + 8 > V) {  // the row's padding columns too
      uint32_t w[4] = {q[p].x, q[p].y, q[p].z, q[p].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (8 * i + 2 * e >= V) w[e] = (w[e] & 0xffff0000u) | 0xff80u;
        if (8 * i + 2 * e + 1 >= V) w[e] = (w[e] & 0xffffu) | 0xff800000u;
      }
      q[p] = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  const int64_t t = target[row];
  const bool ignored = t == ignore_index;
  const bool valid = !ignored && t >= 0 && t < V;
  const float x_t = valid ? __uint_as_float((uint32_t)logits[row * ld + t] << 16) : 0.f;

  float m = -INFINITY;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const uint32_t w[4] = {q[p].x, q[p].y, q[p].z, q[p].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) m = fmaxf(fmaxf(m, bf16_lo(w[e])), bf16_hi(w[e]));
  }
  m = wg_combine<true>(m, red[0]);
  phase(q);
  // (an empty sum, 0, when every logit is -inf)
  const float neg = m == -INFINITY ? 0.f : -m * kLog2e;
  float s = 0.f;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const uint32_t w[4] = {q[p].x, q[p].y, q[p].z, q[p].w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      s += fast_exp2(fmaf(bf16_lo(w[e]), kLog2e, neg));
      s += fast_exp2(fmaf(bf16_hi(w[e]), kLog2e, neg));
    }
  }
  s = wg_combine<false>(s, red[1]);  // also orders every read of the row before the writes below
  phase(q);
  const float lse2 = __log2f(s) - neg;  // log2-sum-exp2 of x * log2 e

  if (threadIdx.x == 0) {
    float loss = 0.f;
    if (valid) loss = lse2 * kLn2 - x_t;
    else if (!ignored) loss = __builtin_nanf("");  // target outside [0, V)
    row_loss[row] = loss;
  }

  const float sc = valid ? *scale : 0.f;
  uint4* g = reinterpret_cast<uint4*>(grad + row * ld);
  const int tv = valid ? (int)(t >> 3) : -1;  // the piece that holds the target
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int i = threadIdx.x + p * kRegThreads;
    if (i >= nvec) break;
    const uint32_t w[4] = {q[p].x, q[p].y, q[p].z, q[p].w};
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float pa = fast_exp2(fmaf(bf16_lo(w[e]), kLog2e, -lse2));
      float pb = fast_exp2(fmaf(bf16_hi(w[e]), kLog2e, -lse2));
      if (i == tv) {
        if ((int)(t & 7) == 2 * e) pa -= 1.f;
        if ((int)(t & 7) == 2 * e + 1) pb -= 1.f;
      }
      o[e] = pack_bf16(pa * sc, pb * sc);
    }
    if (8 * i + 8 > V) {  // padding columns: zero, whatever the row holds
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (8 * i + 2 * e >= V) o[e] = 0u;
        else if (8 * i + 2 * e + 1 >= V) o[e] &= 0xffffu;
      }
    }
    g[i] = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

__global__ __launch_bounds__(kCeThreads) void ce_rows_kernel(
    const uint16_t* logits, uint16_t* grad, int64_t ld, int V,
    const int64_t* __restrict__ target, int64_t ignore_index, const float* __restrict__ scale,
    float* __restrict__ row_loss) {
  __shared__ float red_m[kCeWaves], red_s[kCeWaves];
  __shared__ float x_t;
  const int64_t row = blockIdx.x;
  const uint4* x = reinterpret_cast<const uint4*>(logits + row * ld);
  const int nvec = (int)(ld / 8);
  const int64_t t = target[row];
  const bool ignored = t == ignore_index;
  const bool valid = !ignored && t >= 0 && t < V;
  if (threadIdx.x == 0) x_t = valid ? __uint_as_float((uint32_t)logits[row * ld + t] << 16) : 0.f;

  float m = -INFINITY, s = 0.f;
  for (int i = threadIdx.x; i < nvec; i += kCeThreads) {
    const uint4 q = x[i];
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
    const int j0 = 8 * i;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (j0 + 2 * e < V) lse_add(m, s, bf16_lo(w[e]) * kLog2e);
      if (j0 + 2 * e + 1 < V) lse_add(m, s, bf16_hi(w[e]) * kLog2e);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float m2 = __shfl_xor(m, off, 64), s2 = __shfl_xor(s, off, 64);
    lse_merge(m, s, m2, s2);
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red_m[wave] = m;
    red_s[wave] = s;
  }
  __syncthreads();  // also orders every read of the row before the writes below
  m = red_m[0];
  s = red_s[0];
#pragma unroll
  for (int w = 1; w < kCeWaves; ++w) lse_merge(m, s, red_m[w], red_s[w]);
  const float lse2 = m + __log2f(s);  // log2-sum-exp2 of x * log2 e

  if (threadIdx.x == 0) {
    float loss = 0.f;
    if (valid) loss = lse2 * kLn2 - x_t;
    else if (!ignored) loss = __builtin_nanf("");  // target outside [0, V)
    row_loss[row] = loss;
  }

  const float sc = valid ? *scale : 0.f;
  uint4* g = reinterpret_cast<uint4*>(grad + row * ld);
  for (int i = threadIdx.x; i < nvec; i += kCeThreads) {
    const uint4 q = x[i];
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
    const int j0 = 8 * i;
    uint32_t o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int ja = j0 + 2 * e, jb = ja + 1;
      float pa = ja < V ? exp2f(bf16_lo(w[e]) * kLog2e - lse2) : 0.f;
      float pb = jb < V ? exp2f(bf16_hi(w[e]) * kLog2e - lse2) : 0.f;
      if (ja == t) pa -= 1.f;
      if (jb == t) pb -= 1.f;
      o[e] = pack_bf16(pa * sc, pb * sc);
    }
    g[i] = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

}  // namespace

hipError_t launch_ce_rows(const uint16_t* logits, uint16_t* grad, int64_t rows, int V, int64_t ld,
                          const int64_t* target, int64_t ignore_index, const float* scale,
                          float* row_loss, hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  const dim3 grid((unsigned)rows);
  // in registers from 2048 columns (two for each thread; between the widths
  // measured above) up to what eight pieces a thread hold
  const int64_t pieces = ld < 2 * kRegThreads ? 0 : (ld / 8 + kRegThreads - 1) / kRegThreads;
#define CE_REG(NP)                                                                             \
  hipLaunchKernelGGL(ce_rows_reg_kernel<NP>, grid, dim3(kRegThreads), 0, stream, logits, grad, \
                     ld, V, target, ignore_index, scale, row_loss)
  switch (pieces) {
    case 1: CE_REG(1); break;
    case 2: CE_REG(2); break;
    case 3: CE_REG(3); break;
    case 4: CE_REG(4); break;
    case 5: CE_REG(5); break;
    case 6: CE_REG(6); break;
    case 7: CE_REG(7); break;
    case 8: CE_REG(8); break;
    default:
      hipLaunchKernelGGL(ce_rows_kernel, grid, dim3(kCeThreads), 0, stream, logits, grad, ld, V,
                         target, ignore_index, scale, row_loss);
  }
#undef CE_REG
  return hipGetLastError();
}

}  // namespace t2t
