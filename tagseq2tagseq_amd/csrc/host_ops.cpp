// Host side of the per-layer calls, in C++: output allocation, the argument
// blocks of libt2t_attn.so's C entry points and the launch, on the tensors'
// own device and its current stream.
//
// What bounds it: a layer of a short sequence is host work -- at 512 tokens a
// forward and backward issue about fifty launches whose kernels take 0.26 ms,
// and through ctypes each of these wrappers cost 10 to 25 us (stream and
// device context objects, argument structures, tensor methods).  Here one
// costs 3 to 8 us: B1 H4 T1024 D64 float32 forward 29.7 -> 12.8 us a call,
// bf16 forward + backward at T 1537 156 -> 88, the mask of a 16k row 106 ->
// 64, a layer of 512 x 512 forward + backward 950 -> 750, twelve layers over
// 2048 tokens 3710 -> 2460.  The functions keep nothing from one call to the
// next.
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <tuple>
#include <vector>

#include "../../include/t2t_attn.h"

namespace {

using at::Tensor;

void* stream_of(const Tensor& t) {
  return at::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

void check(int rc, const char* what) {
  TORCH_CHECK(rc == T2T_OK, what, " failed (status ", rc, "): ", t2t_last_error());
}

// The kernels get plain addresses: one of host memory would fault the GPU.
template <typename... Ts>
void need_gpu(const Ts&... t) {
  TORCH_CHECK((t.is_cuda() && ...), "the gfx950 kernels need ROCm GPU tensors");
}

int weight_code(const Tensor& w) {
  TORCH_CHECK(w.scalar_type() == at::kBFloat16 || w.scalar_type() == at::kFloat,
              "weight dtype ", w.scalar_type(), " (bfloat16 or float32)");
  return w.scalar_type() == at::kFloat ? T2T_DTYPE_F32 : T2T_DTYPE_BF16;
}

// The attention kernels' code of q's dtype, which k, v and (backward) out and
// dout share: the kernels read what the code says, whatever the tensors hold.
template <typename... Ts>
int attention_code(const Tensor& q, const Ts&... others) {
  const at::ScalarType t = q.scalar_type();
  TORCH_CHECK_NOT_IMPLEMENTED(t == at::kBFloat16 || t == at::kFloat, "dtype ", t,
                              " is not supported (bfloat16 or float32)");
  TORCH_CHECK_VALUE(((others.scalar_type() == t) && ...), "attention operands differ in dtype");
  return t == at::kFloat ? T2T_DTYPE_F32 : T2T_DTYPE_BF16;
}

// [B, H, T, D] with unit stride along D; a dimension of size 1 is never stepped.
t2t_tensor view4(const Tensor& t) {
  TORCH_CHECK_VALUE(t.dim() == 4, "expected a 4-D [B, H, T, D] tensor, got shape ", t.sizes());
  TORCH_CHECK_VALUE(t.stride(3) == 1, "the head dimension (last) must have unit stride");
  return t2t_tensor{t.data_ptr(), t.size(0) == 1 ? 0 : t.stride(0),
                    t.size(1) == 1 ? 0 : t.stride(1), t.stride(2)};
}

// The rows [N, C] of t's last dimension as the kernels read them: unit column
// stride, row stride a multiple of 8 elements and a 16-byte aligned start;
// anything else is copied (rows that are contiguous but start between two such
// boundaries too, which contiguous() would hand back).
Tensor rows_of(const Tensor& t) {
  Tensor r = t.dim() == 2 ? t : t.reshape({-1, t.size(-1)});
  const bool ok = r.stride(1) == 1 && r.stride(0) % 8 == 0 &&
                  reinterpret_cast<uintptr_t>(r.data_ptr()) % 16 == 0;
  return ok ? r : r.clone(at::MemoryFormat::Contiguous);
}

const t2t_block_mask* mask_at(int64_t address) {
  return reinterpret_cast<const t2t_block_mask*>(static_cast<intptr_t>(address));
}

// ---- attention (mask: address of the caller's t2t_block_mask, alive during the call)

std::tuple<Tensor, Tensor> attn_fwd(const Tensor& q, const Tensor& k, const Tensor& v,
                                    int64_t mask, double scale) {
  const int dtype = attention_code(q, k, v);
  need_gpu(q, k, v);
  const c10::DeviceGuard guard(q.device());
  const int64_t B = q.size(0), Hq = q.size(1), T = q.size(2), D = q.size(3), Hkv = k.size(1);
  // [B, T, Hq, D] storage seen as [B, Hq, T, D]: the module's output
  // projection then reads token rows without a transpose copy
  Tensor out = at::empty({B, T, Hq, D}, q.options()).transpose(1, 2);
  Tensor lse2 = at::empty({B, Hq, T}, q.options().dtype(at::kFloat));
  const t2t_tensor qs = view4(q), ks = view4(k), vs = view4(v), os = view4(out);
  check(t2t_attn_fwd(&qs, &ks, &vs, &os, lse2.data_ptr<float>(), B, Hq, Hkv, T, D,
                     dtype, static_cast<float>(scale), mask_at(mask), stream_of(q)),
        "t2t_attn_fwd");
  return {out, lse2};
}

std::tuple<Tensor, Tensor, Tensor> attn_bwd(const Tensor& q, const Tensor& k, const Tensor& v,
                                            const Tensor& out, const Tensor& dout_in,
                                            const Tensor& lse2, int64_t mask, double scale) {
  const int dtype = attention_code(q, k, v, out, dout_in);
  need_gpu(q, k, v, out, dout_in, lse2);
  const c10::DeviceGuard guard(q.device());
  const int64_t B = q.size(0), Hq = q.size(1), T = q.size(2), D = q.size(3), Hkv = k.size(1);
  const Tensor dout = dout_in.stride(3) == 1 ? dout_in : dout_in.contiguous();
  Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(k.sizes(), k.options()),
         dv = at::empty(v.sizes(), v.options());
  Tensor delta = at::empty({B, Hq, T}, q.options().dtype(at::kFloat));
  const t2t_tensor qs = view4(q), ks = view4(k), vs = view4(v), os = view4(out),
                   ds = view4(dout), dqs = view4(dq), dks = view4(dk), dvs = view4(dv);
  check(t2t_attn_bwd(&qs, &ks, &vs, &os, &ds, lse2.data_ptr<float>(), delta.data_ptr<float>(),
                     &dqs, &dks, &dvs, B, Hq, Hkv, T, D, dtype,
                     static_cast<float>(scale), mask_at(mask), stream_of(q)),
        "t2t_attn_bwd");
  return {dq, dk, dv};
}

// ---- RMS normalisation

std::tuple<Tensor, Tensor> rms_norm(const Tensor& x, const Tensor& weight, double eps) {
  need_gpu(x, weight);
  const c10::DeviceGuard guard(x.device());
  const int64_t C = x.size(-1);
  const Tensor xr = rows_of(x), w = weight.contiguous();
  const int64_t N = xr.size(0);
  Tensor y = at::empty(x.sizes(), x.options());
  Tensor rstd = at::empty({N}, x.options().dtype(at::kFloat));
  check(t2t_rms_norm(xr.data_ptr(), xr.stride(0), w.data_ptr(), weight_code(w), y.data_ptr(), C,
                     rstd.data_ptr<float>(), N, C, static_cast<float>(eps), stream_of(x)),
        "t2t_rms_norm");
  return {y, rstd};
}

std::tuple<Tensor, Tensor> rms_norm_backward(const Tensor& dy, const Tensor& x,
                                             const Tensor& weight, const Tensor& rstd) {
  need_gpu(dy, x, weight, rstd);
  const c10::DeviceGuard guard(x.device());
  const int64_t C = x.size(-1);
  const Tensor xr = rows_of(x), dyr = rows_of(dy), w = weight.contiguous();
  const int64_t N = xr.size(0);
  Tensor dx = at::empty(x.sizes(), x.options());
  Tensor dw = at::empty(w.sizes(), w.options());
  const int64_t bytes = t2t_rms_norm_backward_workspace(N, C);
  Tensor ws = at::empty({std::max<int64_t>(1, bytes / 4)}, x.options().dtype(at::kFloat));
  check(t2t_rms_norm_backward(dyr.data_ptr(), dyr.stride(0), xr.data_ptr(), xr.stride(0),
                              w.data_ptr(), weight_code(w), rstd.data_ptr<float>(), dx.data_ptr(),
                              C, dw.data_ptr(), ws.data_ptr(), ws.numel() * 4, N, C,
                              stream_of(x)),
        "t2t_rms_norm_backward");
  return {dx, dw};
}

// ---- QKV split + rotary embedding

std::tuple<Tensor, Tensor, Tensor> qkv_rope(const Tensor& qkv_in, const Tensor& cos_in,
                                            const Tensor& sin_in, int64_t heads, int64_t pos0) {
  TORCH_CHECK_VALUE(qkv_in.dim() == 3, "qkv must be [B, T, 3 C], got shape ", qkv_in.sizes());
  TORCH_CHECK_VALUE(heads > 0, "num_heads=", heads, " must be positive");
  TORCH_CHECK_VALUE(qkv_in.size(2) % (3 * heads) == 0, "last dim ", qkv_in.size(2),
                    " is not 3 * num_heads * head_dim (num_heads=", heads, ")");
  TORCH_CHECK_NOT_IMPLEMENTED(qkv_in.scalar_type() == at::kBFloat16, "qkv dtype ",
                              qkv_in.scalar_type(), " is not supported (bfloat16 only)");
  need_gpu(qkv_in, cos_in, sin_in);
  const c10::DeviceGuard guard(qkv_in.device());
  const Tensor qkv = qkv_in.stride(2) == 1 ? qkv_in : qkv_in.contiguous();
  const Tensor cos = cos_in.contiguous(), sin = sin_in.contiguous();
  const int64_t B = qkv.size(0), T = qkv.size(1), D = qkv.size(2) / (3 * heads);
  Tensor q = at::empty({B, heads, T, D}, qkv.options()), k = at::empty_like(q),
         v = at::empty_like(q);
  const t2t_tensor qs{q.data_ptr(), q.stride(0), q.stride(1), q.stride(2)},
      ks{k.data_ptr(), k.stride(0), k.stride(1), k.stride(2)},
      vs{v.data_ptr(), v.stride(0), v.stride(1), v.stride(2)};
  check(t2t_qkv_rope(qkv.data_ptr(), qkv.stride(0), qkv.stride(1), B, T, heads, D,
                     cos.data_ptr<float>(), sin.data_ptr<float>(), cos.size(0), pos0, &qs, &ks,
                     &vs, stream_of(qkv)),
        "t2t_qkv_rope");
  return {q, k, v};
}

Tensor qkv_rope_backward(const Tensor& dq_in, const Tensor& dk_in, const Tensor& dv_in,
                         const Tensor& cos_in, const Tensor& sin_in, int64_t pos0) {
  for (const Tensor* t : {&dq_in, &dk_in, &dv_in})
    TORCH_CHECK_VALUE(t->dim() == 4, "expected a 4-D [B, H, T, D] gradient, got shape ",
                      t->sizes());
  need_gpu(dq_in, dk_in, dv_in, cos_in, sin_in);
  const c10::DeviceGuard guard(dq_in.device());
  const int64_t B = dq_in.size(0), H = dq_in.size(1), T = dq_in.size(2), D = dq_in.size(3);
  const Tensor dq = dq_in.stride(3) == 1 ? dq_in : dq_in.contiguous();
  const Tensor dk = dk_in.stride(3) == 1 ? dk_in : dk_in.contiguous();
  const Tensor dv = dv_in.stride(3) == 1 ? dv_in : dv_in.contiguous();
  const Tensor cos = cos_in.contiguous(), sin = sin_in.contiguous();
  Tensor dqkv = at::empty({B, T, 3 * H * D}, dq.options());
  const t2t_tensor qs{dq.data_ptr(), dq.stride(0), dq.stride(1), dq.stride(2)},
      ks{dk.data_ptr(), dk.stride(0), dk.stride(1), dk.stride(2)},
      vs{dv.data_ptr(), dv.stride(0), dv.stride(1), dv.stride(2)};
  check(t2t_qkv_rope_backward(&qs, &ks, &vs, cos.data_ptr<float>(), sin.data_ptr<float>(),
                              cos.size(0), pos0, B, T, H, D, dqkv.data_ptr(), dqkv.stride(0),
                              dqkv.stride(1), stream_of(dq)),
        "t2t_qkv_rope_backward");
  return dqkv;
}

// ---- SwiGLU

std::tuple<Tensor, Tensor> swiglu(const Tensor& gu) {
  need_gpu(gu);
  const c10::DeviceGuard guard(gu.device());
  const Tensor g2 = rows_of(gu);
  const int64_t N = g2.size(0), H = g2.size(1) / 2;
  std::vector<int64_t> shape = gu.sizes().vec();
  shape.back() = H;
  Tensor h = at::empty(shape, gu.options());
  check(t2t_swiglu(g2.data_ptr(), g2.stride(0), h.data_ptr(), H, N, H, stream_of(gu)),
        "t2t_swiglu");
  return {h, g2};
}

Tensor swiglu_backward(const Tensor& g2, const Tensor& dh, at::IntArrayRef shape) {
  need_gpu(g2, dh);
  const c10::DeviceGuard guard(g2.device());
  const int64_t N = g2.size(0), H = g2.size(1) / 2;
  const Tensor d2 = rows_of(dh);
  Tensor dgu = at::empty(shape, g2.options());
  check(t2t_swiglu_backward(g2.data_ptr(), g2.stride(0), d2.data_ptr(), d2.stride(0),
                            dgu.data_ptr(), 2 * H, N, H, stream_of(g2)),
        "t2t_swiglu_backward");
  return dgu;
}

// ---- linear map of token rows: x W^T, or x W (transposed)

Tensor linear(const Tensor& x, const Tensor& w, bool transposed) {
  need_gpu(x, w);
  const c10::DeviceGuard guard(x.device());
  const Tensor x2 = rows_of(x), w2 = rows_of(w);
  const int64_t M = x2.size(0), K = x2.size(1), N = w2.size(transposed ? 1 : 0);
  TORCH_CHECK(w2.size(transposed ? 0 : 1) == K, "weight ", w.sizes(), " does not take rows of ", K);
  std::vector<int64_t> shape = x.sizes().vec();
  shape.back() = N;
  Tensor y = at::empty(shape, x.options());
  check(t2t_linear(x2.data_ptr(), x2.stride(0), w2.data_ptr(), w2.stride(0), transposed,
                   y.data_ptr(), N, M, N, K, stream_of(x)),
        "t2t_linear");
  return y;
}

// ---- weight gradient dY^T X

Tensor wgrad(const Tensor& dy, const Tensor& x, at::ScalarType out_dtype) {
  need_gpu(dy, x);
  const c10::DeviceGuard guard(x.device());
  const Tensor d2 = rows_of(dy), x2 = rows_of(x);
  const int64_t K = d2.size(0), M = d2.size(1), N = x2.size(1);
  Tensor ws = at::empty({t2t_wgrad_workspace(M, N, K)}, x.options().dtype(at::kByte));
  Tensor out = at::empty({M, N}, x.options().dtype(out_dtype));
  check(t2t_wgrad(d2.data_ptr(), d2.stride(0), x2.data_ptr(), x2.stride(0), out.data_ptr(),
                  out_dtype == at::kFloat ? T2T_DTYPE_F32 : T2T_DTYPE_BF16, M, N, K,
                  ws.data_ptr(), ws.numel(), stream_of(x)),
        "t2t_wgrad");
  return out;
}

// ---- mask metadata

// The tables of t2t_mask_meta for doc [Bm, T] (int32) and words [Bm, W, T]
// (int64), in the order tile_class, the 13 tables of t2t_block_mask.  The
// index tables are views of one allocation; the bitmaps, which dwarf them,
// are their own.
std::vector<Tensor> mask_meta(const Tensor& doc, const Tensor& q_bits, const Tensor& kv_bits,
                              int64_t stream) {
  need_gpu(doc, q_bits, kv_bits);
  const c10::DeviceGuard guard(doc.device());
  const int64_t Bm = doc.size(0), T = doc.size(1), W = q_bits.size(1);
  const int64_t nt = (T + T2T_TILE - 1) / T2T_TILE;
  const auto i32 = doc.options().dtype(at::kInt);
  const int64_t row = Bm * nt, grid = Bm * nt * nt;
  const auto padded = [](int64_t n) { return (n + 15) / 16 * 16; };  // 64-byte starts
  Tensor pool = at::empty({7 * padded(row) + 5 * padded(grid)}, i32);
  int64_t at_ = 0;
  const auto take = [&](at::IntArrayRef shape, int64_t n) {
    Tensor t = pool.narrow(0, at_, n).view(shape);
    at_ += padded(n);
    return t;
  };
  std::vector<Tensor> t;
  t.reserve(14);
  t.push_back(at::empty({Bm, nt, nt}, doc.options().dtype(at::kChar)));
  for (int i = 0; i < 4; ++i) {  // kv, full_kv, q, full_q
    t.push_back(take({Bm, 1, nt}, row));
    t.push_back(take({Bm, 1, nt, nt}, grid));
  }
  t.push_back(take({Bm, nt}, row));       // row_order
  t.push_back(take({Bm, nt}, row));       // col_order
  t.push_back(take({Bm, nt}, row));       // kv_bits_off
  t.push_back(take({Bm, nt, nt}, grid));  // q_bits_slot
  const int64_t slots = std::max<int64_t>(1, Bm * nt * (nt + 1) / 2);
  t.push_back(at::empty({slots, 2, T2T_TILE, 4}, i32));
  const auto ptr = [&](int i) { return static_cast<int32_t*>(t[i].data_ptr()); };
  t2t_block_mask m{};
  m.mask_batch = Bm;
  m.num_tiles = nt;
  m.kv_num = ptr(1); m.kv_idx = ptr(2); m.full_kv_num = ptr(3); m.full_kv_idx = ptr(4);
  m.q_num = ptr(5); m.q_idx = ptr(6); m.full_q_num = ptr(7); m.full_q_idx = ptr(8);
  m.row_order = ptr(9); m.col_order = ptr(10); m.kv_bits_off = ptr(11); m.q_bits_slot = ptr(12);
  m.tile_bits = static_cast<uint32_t*>(t[13].data_ptr());
  m.tile_bits_slots = slots;
  check(t2t_mask_meta(static_cast<const int32_t*>(doc.data_ptr()),
                      W ? static_cast<const uint64_t*>(q_bits.data_ptr()) : nullptr,
                      W ? static_cast<const uint64_t*>(kv_bits.data_ptr()) : nullptr, Bm, T, W,
                      static_cast<int8_t*>(t[0].data_ptr()), &m,
                      reinterpret_cast<void*>(static_cast<intptr_t>(stream))),
        "t2t_mask_meta");
  return t;
}

// doc [B, T] and, when words > 0, q / kv words [B, words, T] (else undefined)
// from the device-resident lists (int32): spans at 0, grants at `grants`,
// the counts at `counts`, and link rows (uint64) at `links` (-1: none).
std::vector<Tensor> token_inputs(const Tensor& lists, int64_t grants, int64_t counts,
                                 int64_t links, int64_t B, int64_t T, int64_t words,
                                 int64_t max_spans, int64_t max_grants, bool has_grants,
                                 const std::vector<Tensor>& out) {
  TORCH_CHECK(out.empty() || words == 0 || out.size() == 3,
              "doc, q_bits and kv_bits are needed to overwrite ", words, " words a token");
  need_gpu(lists);
  const c10::DeviceGuard guard(lists.device());
  std::vector<Tensor> t = out;
  for (const Tensor& o : t) need_gpu(o);
  if (t.empty()) {
    t.push_back(at::empty({B, T}, lists.options()));
    if (words > 0)
      for (int i = 0; i < 2; ++i)
        t.push_back(at::empty({B, words, T}, lists.options().dtype(at::kLong)));
  }
  const int32_t* base = static_cast<const int32_t*>(lists.data_ptr());
  check(t2t_token_inputs(base, base + counts, max_spans, has_grants ? base + grants : nullptr,
                         has_grants ? base + counts + B : nullptr, max_grants,
                         links >= 0 ? reinterpret_cast<const uint64_t*>(base + links) : nullptr,
                         B, T, words, static_cast<int32_t*>(t[0].data_ptr()),
                         words > 0 ? static_cast<uint64_t*>(t[1].data_ptr()) : nullptr,
                         words > 0 ? static_cast<uint64_t*>(t[2].data_ptr()) : nullptr,
                         stream_of(lists)),
        "t2t_token_inputs");
  return t;
}

// ---- what may be watching a call

// Nothing but the caller sees the call, and the tensors are what their
// addresses say: no tracer, dispatch mode or function transform is active,
// and every argument is a torch.Tensor or Parameter itself (not a subclass)
// with plain memory of its own (not batched, nested, sparse or lazily
// negated).  A kernel called on addresses would be missing from a trace, and
// its output in it is the empty allocation.
bool plain_call(PyObject* const* args, Py_ssize_t n, bool recorded_counts) {
  constexpr c10::DispatchKeySet kIndirect{
      c10::DispatchKey::Batched,    c10::DispatchKey::FuncTorchBatched,
      c10::DispatchKey::Python,     c10::DispatchKey::NestedTensor,
      c10::DispatchKey::Negative,   c10::DispatchKey::Conjugate,
      c10::DispatchKey::ZeroTensor, c10::DispatchKey::Functionalize};
  if (torch::jit::tracer::isTracing() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
      c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
    return false;
  const bool grad = recorded_counts && c10::GradMode::is_enabled();
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (!THPVariable_CheckExact(args[i])) return false;
    const Tensor& t = THPVariable_Unpack(args[i]);
    if (t.key_set().has_any(kIndirect) || t.layout() != at::kStrided || !t.has_storage() ||
        (grad && t.requires_grad()))
      return false;
  }
  return true;
}

PyObject* plain(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return PyBool_FromLong(plain_call(args, n, false));
}

PyObject* unwatched(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return PyBool_FromLong(plain_call(args, n, true));
}

PyMethodDef kPredicates[] = {
    {"plain", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(plain)), METH_FASTCALL,
     "plain(*tensors): nothing but the caller sees a call on them"},
    {"unwatched", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(unwatched)),
     METH_FASTCALL, "plain(*tensors), and no graph records it"},
    {nullptr, nullptr, 0, nullptr}};

int64_t current_stream(int64_t device) {
  return reinterpret_cast<int64_t>(
      at::hip::getCurrentHIPStreamMasqueradingAsCUDA(static_cast<c10::DeviceIndex>(device))
          .stream());
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  // a launch may wait on a full queue, an allocation on the device: other
  // Python threads run meanwhile
  const auto no_gil = py::call_guard<py::gil_scoped_release>();
  m.def("attn_fwd", &attn_fwd, no_gil);
  m.def("attn_bwd", &attn_bwd, no_gil);
  m.def("rms_norm", &rms_norm, no_gil);
  m.def("rms_norm_backward", &rms_norm_backward, no_gil);
  m.def("qkv_rope", &qkv_rope, no_gil);
  m.def("qkv_rope_backward", &qkv_rope_backward, no_gil);
  m.def("swiglu", &swiglu, no_gil);
  m.def("swiglu_backward",
        [](const Tensor& g2, const Tensor& dh, const std::vector<int64_t>& shape) {
          return swiglu_backward(g2, dh, shape);
        }, no_gil);
  m.def("linear", &linear, no_gil);
  m.def("wgrad", [](const Tensor& dy, const Tensor& x, bool f32) {
    return wgrad(dy, x, f32 ? at::kFloat : at::kBFloat16);
  }, no_gil);
  m.def("mask_meta", &mask_meta, no_gil);
  m.def("token_inputs", &token_inputs, no_gil);
  m.def("current_stream", &current_stream);
  if (PyModule_AddFunctions(m.ptr(), kPredicates) != 0) throw py::error_already_set();
}
