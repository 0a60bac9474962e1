// Native host path of the eager operator calls: argument checks, output allocation, the C structs and the autograd node of
// chunk_palimpsa, in one extension call instead of some 25 us of Python per forward and 60 per forward and backward
// (one token of one sequence: 27 us a call, of which the kernel takes 5 and its launch 3).
//
// It serves the plain call, which is what the layers and a serving loop make: rows all bf16 or all fp32 and contiguous, head
// dims the kernels are compiled for, gates fp32 or bf16, states and per-head values fp32, everything on the current
// device.  For anything else the functions return None before they do anything and the caller takes its Python route,
// which converts and pads, or raises the error that the call deserves.
//
// The kernels are reached through the C ABI of palimpsa_hip.h, whose addresses the Python loader hands over once (bind).
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include "../../include/palimpsa_hip.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using OptT = std::optional<Tensor>;

struct Abi {
  int (*recurrent_fwd)(const PalDims*, const PalFwdTensors*, void*);
  int (*gla_recurrent_fwd)(const PalDims*, const PalFwdTensors*, void*);
  int (*chunk_fwd)(const PalDims*, const PalFwdTensors*, void*);
  int (*chunk_bwd)(const PalDims*, const PalFwdTensors*, const PalBwdTensors*, void*, size_t, void*);
  size_t (*chunk_bwd_workspace_bytes)(const PalDims*);
  int (*chunk_bwd_supported)(int32_t, int32_t, int32_t, uint32_t);
} abi;
py::handle raise_code;   // (code, where): raises what the Python routes raise for a code of the library

void bind(const std::vector<uintptr_t>& p, py::object check) {
  TORCH_CHECK(p.size() * sizeof(p[0]) == sizeof(abi), "bind: number of addresses");
  memcpy(&abi, p.data(), sizeof(abi));
  raise_code = check.release();   // held for the life of the process
}

// For the autograd node, whose backward runs on a thread of the engine: a Python exception that the engine carries over.
[[noreturn]] void fail(int rc, const char* where) {
  py::gil_scoped_acquire gil;
  try {
    raise_code(rc, where);
    PyErr_SetString(PyExc_RuntimeError, where);   // (not reached: the codes are errors)
  } catch (py::error_already_set& e) {
    e.restore();
  }
  python_error err;
  err.persist();
  throw err;
}

// kernel calls without the interpreter lock where the thread holds it (a launch may wait for room in the queue)
struct NoGil {
  PyThreadState* s;
  NoGil() : s(PyGILState_Check() ? PyEval_SaveThread() : nullptr) {}
  ~NoGil() { if (s) PyEval_RestoreThread(s); }
};

bool plain(const Tensor& t, const c10::Device& dev, at::ScalarType st) {
  return t.defined() && t.device() == dev && t.scalar_type() == st && t.layout() == at::kStrided &&
         !t.unsafeGetTensorImpl()->is_python_dispatch() && t.is_contiguous();
}
bool plain_opt(const OptT& t, const c10::Device& dev, at::ScalarType st) { return !t || plain(*t, dev, st); }

const void* ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return t.defined() ? (float*)t.mutable_data_ptr() : nullptr; }

// shapes and types of a call; ok = false: not plain
struct Call {
  bool ok = false;
  int64_t B = 0, T = 0, H = 0, Hq = 0, dk = 0, dv = 0, N = 0;
  at::ScalarType rows = at::kFloat;
  PalDims dims{};

  Call(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor* b, const Tensor& gt, const Tensor& g, const Tensor* Ip,
       double scale, int64_t n_seqs) {
    if (!q.defined() || q.device().type() != at::kCUDA || q.dim() != 4 || v.dim() != 4) return;
    const c10::Device dev = q.device();
    rows = q.scalar_type();
    if ((rows != at::kBFloat16 && rows != at::kFloat) || dev.index() != c10::hip::current_device()) return;
    if (!plain(q, dev, rows) || !plain(k, dev, rows) || !plain(v, dev, rows) || k.sizes() != q.sizes()) return;
    B = v.size(0); T = v.size(1); H = v.size(2); dv = v.size(3);
    Hq = q.size(2); dk = q.size(3);
    if (q.size(0) != B || q.size(1) != T || Hq < 1 || H % Hq != 0 || B * T == 0) return;
    if (dk % 16 || dv % 16 || dk < 16 || dv < 16 || dk > 256 || dv > 256) return;
    if (b && (!plain(*b, dev, rows) || b->sizes() != v.sizes())) return;
    const at::ScalarType gs = gt.scalar_type();
    if ((gs != at::kFloat && gs != at::kBFloat16) || !plain(gt, dev, gs) || gt.dim() != 3 || gt.size(0) != B || gt.size(1) != T ||
        gt.size(2) != H || ((uintptr_t)gt.const_data_ptr() & 3))
      return;
    if (!plain(g, dev, at::kFloat) || g.numel() != H || (Ip && (!plain(*Ip, dev, at::kFloat) || Ip->numel() != H))) return;
    if (B > INT32_MAX || T > INT32_MAX || H > INT32_MAX) return;
    N = n_seqs > 0 ? n_seqs : B;
    dims.batch = (int32_t)B; dims.seq_len = (int32_t)T; dims.n_seqs = (int32_t)N; dims.n_heads = (int32_t)H;
    dims.dk = (int32_t)dk; dims.dv = (int32_t)dv;
    dims.dtype = rows == at::kBFloat16 ? PAL_DTYPE_BF16 : PAL_DTYPE_F32;
    dims.gate_dtype = gs == at::kBFloat16 ? PAL_DTYPE_BF16 : PAL_DTYPE_F32;
    dims.var_dtype = PAL_DTYPE_F32;
    dims.scale = (float)scale;
    dims.n_qk_heads = (int32_t)Hq;
    ok = true;
  }
};

bool state_ok(const OptT& s, const c10::Device& dev, int64_t N, int64_t H, int64_t r, int64_t c) {
  return plain_opt(s, dev, at::kFloat) &&
         (!s || (s->dim() == 4 && s->size(0) == N && s->size(1) == H && s->size(2) == r && s->size(3) == c));
}

bool wants_grad(std::initializer_list<const Tensor*> ts, const OptT& a, const OptT& b) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->requires_grad()) return true;
  return (a && a->requires_grad()) || (b && b->requires_grad());
}

// No tracer (torch.jit.trace), functorch transform (vmap, grad, jvp) and no dispatch mode is listening on this thread: each
// would see the output allocations of a call but not the kernel that fills them.  (torch switches each of them on by a
// dispatch key that it includes for the thread.)
bool unobserved() {
  return (c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set).empty();
}

// A tensor with a forward-mode tangent (a dual number, whether or not it requires grad): the autograd Functions of the
// Python route refuse it, a plain kernel call would hand back results without a tangent, a derivative of zero.
bool has_tangent(std::initializer_list<const Tensor*> ts, const OptT& a, const OptT& b) {
  for (const Tensor* t : ts)
    if (t->defined() && t->_fw_grad(/*level=*/0).defined()) return true;
  return (a && a->_fw_grad(0).defined()) || (b && b->_fw_grad(0).defined());
}

void* stream_of(const c10::Device& dev) { return (void*)c10::hip::getCurrentHIPStream(dev.index()).stream(); }

// ---------------------------------------------------------------------------------------------- token-serial forward
// (o, o_var | None, final_mu | None, final_I | None), or None
py::object recurrent_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& b, const Tensor& gt, const Tensor& g,
                         const Tensor& Ip, double scale, const OptT& mu, const OptT& I, bool final_state, bool var,
                         int64_t mode_flags) {
  if (!unobserved() || mu.has_value() != I.has_value()) return py::none();
  if (wants_grad({&q, &k, &v, &b, &gt, &g, &Ip}, mu, I)) return py::none();
  if (has_tangent({&q, &k, &v, &b, &gt, &g, &Ip}, mu, I)) return py::none();
  Call c(q, k, v, &b, gt, g, &Ip, scale, 0);
  if (!c.ok) return py::none();
  switch (c.dk) {   // the head dims that the token-serial kernels are compiled for
    case 16: case 32: case 48: case 64: case 96: case 128: case 192: case 256: break;
    default: return py::none();
  }
  const c10::Device dev = q.device();
  if (!state_ok(mu, dev, c.N, c.H, c.dv, c.dk) || !state_ok(I, dev, c.N, c.H, c.dv, c.dk)) return py::none();
  const auto f32 = q.options().dtype(at::kFloat).requires_grad(false);
  Tensor o = at::empty(v.sizes(), v.options().requires_grad(false)), ov, fm, fI;
  if (var) ov = at::empty(v.sizes(), f32);
  if (final_state) {
    fm = at::empty({c.N, c.H, c.dv, c.dk}, f32);
    fI = at::empty({c.N, c.H, c.dv, c.dk}, f32);
  }
  c.dims.flags = (uint32_t)mode_flags | (mu ? PAL_FLAG_HAS_INIT : 0) | (final_state ? PAL_FLAG_STORE_FINAL : 0) | (var ? PAL_FLAG_HAS_VAR : 0);
  PalFwdTensors t{};
  t.q = ptr(q); t.k = ptr(k); t.v = ptr(v); t.b = ptr(b); t.gt = ptr(gt); t.g = (const float*)ptr(g); t.Ip = (const float*)ptr(Ip);
  t.o = o.mutable_data_ptr(); t.o_var = fptr(ov);
  if (mu) { t.init_mu = (const float*)ptr(*mu); t.init_I = (const float*)ptr(*I); }
  t.final_mu = fptr(fm); t.final_I = fptr(fI);
  int rc;
  { NoGil off; rc = abi.recurrent_fwd(&c.dims, &t, stream_of(dev)); }
  if (rc) return py::none();   // nothing was launched: the Python route says what is wrong
  auto opt = [](const Tensor& x) -> py::object { return x.defined() ? py::cast(x) : py::none(); };
  return py::make_tuple(o, opt(ov), opt(fm), opt(fI));
}

// the same without the precision state: (o, final | None), or None; states [N, H, dk, dv]
py::object gla_recurrent_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g, const Tensor& rate, double scale,
                             const OptT& S, bool final_state, int64_t mode_flags) {
  if (!unobserved() || wants_grad({&q, &k, &v, &g}, S, std::nullopt) || has_tangent({&q, &k, &v, &g}, S, std::nullopt)) return py::none();
  Call c(q, k, v, nullptr, g, rate, nullptr, scale, 0);
  if (!c.ok) return py::none();
  const c10::Device dev = q.device();
  if (!state_ok(S, dev, c.N, c.H, c.dk, c.dv)) return py::none();
  Tensor o = at::empty(v.sizes(), v.options().requires_grad(false)), fin;
  if (final_state) fin = at::empty({c.N, c.H, c.dk, c.dv}, q.options().dtype(at::kFloat).requires_grad(false));
  c.dims.flags = (uint32_t)mode_flags | (S ? PAL_FLAG_HAS_INIT : 0) | (final_state ? PAL_FLAG_STORE_FINAL : 0);
  PalFwdTensors t{};
  t.q = ptr(q); t.k = ptr(k); t.v = ptr(v); t.gt = ptr(g); t.g = (const float*)ptr(rate);
  t.o = o.mutable_data_ptr();
  if (S) t.init_mu = (const float*)ptr(*S);
  t.final_mu = fptr(fin);
  int rc;
  { NoGil off; rc = abi.gla_recurrent_fwd(&c.dims, &t, stream_of(dev)); }
  if (rc) return py::none();
  return py::make_tuple(o, fin.defined() ? py::cast(fin) : py::none());
}

// ------------------------------------------------------------------------------------------------------ chunked form
struct ChunkOut { Tensor o, ov, fm, fI, tile_mu, tile_I; };

// forward on tensors that Call has looked at; 0 or the library's code
int chunk_forward(Call& c, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& b, const Tensor& gt, const Tensor& g,
                  const Tensor& Ip, const Tensor& mu, const Tensor& I, bool var, uint32_t flags, const Tensor& meta,
                  const Tensor& cu, int64_t tiles, ChunkOut& out) {
  const auto f32 = q.options().dtype(at::kFloat).requires_grad(false);
  out.o = at::empty(v.sizes(), v.options().requires_grad(false));
  if (var) out.ov = at::empty(v.sizes(), v.options().requires_grad(false));
  out.fm = at::empty({c.N, c.H, c.dv, c.dk}, f32);
  out.fI = at::empty({c.N, c.H, c.dv, c.dk}, f32);
  out.tile_mu = at::empty({tiles, c.H, c.dv, c.dk}, f32);
  out.tile_I = at::empty({tiles, c.H, c.dv, c.dk}, f32);
  c.dims.total_chunks = (int32_t)tiles;
  c.dims.var_dtype = c.dims.dtype;
  c.dims.flags = flags | PAL_FLAG_STORE_FINAL;
  PalFwdTensors t{};
  t.q = ptr(q); t.k = ptr(k); t.v = ptr(v); t.b = ptr(b); t.gt = ptr(gt); t.g = (const float*)ptr(g); t.Ip = (const float*)ptr(Ip);
  t.o = out.o.mutable_data_ptr(); t.o_var = var ? out.ov.mutable_data_ptr() : nullptr;
  t.init_mu = (const float*)ptr(mu); t.init_I = (const float*)ptr(I);
  t.final_mu = fptr(out.fm); t.final_I = fptr(out.fI);
  if (cu.defined()) {
    t.cu_seqlens = (const int32_t*)ptr(cu);
    t.chunk_offsets = (const int32_t*)ptr(meta);
    t.chunk_table = t.chunk_offsets + c.N + 1;
  }
  t.chunk_mu = fptr(out.tile_mu); t.chunk_I = fptr(out.tile_I);
  NoGil off;
  return abi.chunk_fwd(&c.dims, &t, stream_of(q.device()));
}

// The autograd node: argument order and results of the Python Function's gradients (initial states included; gradients of
// the final states are ignored, chunk_palimpsa_forgetting_scalar.py:522 of the reference).
struct ChunkNode : torch::autograd::Function<ChunkNode> {
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                                                const Tensor& b, const Tensor& gt, const Tensor& g, const Tensor& Ip, const OptT& mu_,
                                                const OptT& I_, const OptT& meta_, const OptT& cu_, double scale, bool var,
                                                int64_t flags, int64_t tiles) {
    const Tensor mu = mu_.value_or(Tensor()), I = I_.value_or(Tensor()), meta = meta_.value_or(Tensor()), cu = cu_.value_or(Tensor());
    Call c(q, k, v, &b, gt, g, &Ip, scale, cu.defined() ? cu.numel() - 1 : 0);
    ChunkOut out;
    const int rc = chunk_forward(c, q, k, v, b, gt, g, Ip, mu, I, var, (uint32_t)flags, meta, cu, tiles, out);
    if (rc) fail(rc, "pal_chunk_fwd");
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({q, k, v, b, gt, g, Ip, mu, I, meta, cu, out.tile_mu, out.tile_I});
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["flags"] = flags;
    ctx->saved_data["var"] = var;
    ctx->saved_data["tiles"] = tiles;
    torch::autograd::variable_list r{out.o, out.fm, out.fI};
    if (var) r.push_back(out.ov);
    return r;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list gr) {
    const auto s = ctx->get_saved_variables();
    const Tensor &q = s[0], &k = s[1], &v = s[2], &b = s[3], &gt = s[4], &g = s[5], &Ip = s[6], &mu = s[7], &I = s[8], &meta = s[9],
                 &cu = s[10], &tile_mu = s[11], &tile_I = s[12];
    const c10::DeviceGuard guard(q.device());
    Call c(q, k, v, &b, gt, g, &Ip, ctx->saved_data["scale"].toDouble(), cu.defined() ? cu.numel() - 1 : 0);
    // what the forward saved has been through the saved-tensor hooks, which may hand back anything
    const int64_t tiles = ctx->saved_data["tiles"].toInt();
    const auto f32_as = [&](const Tensor& t, int64_t n) { return plain(t, q.device(), at::kFloat) && t.numel() == n * c.H * c.dv * c.dk; };
    const auto i32_as = [&](const Tensor& t, int64_t n) { return plain(t, q.device(), at::kInt) && t.numel() == n; };
    TORCH_CHECK_VALUE(c.ok && f32_as(tile_mu, tiles) && f32_as(tile_I, tiles) && mu.defined() == I.defined() &&
                          (!mu.defined() || (f32_as(mu, c.N) && f32_as(I, c.N))) &&
                          (!cu.defined() || (i32_as(cu, c.N + 1) && i32_as(meta, c.N + 1 + 4 * tiles))),
                      "chunk_palimpsa backward: a saved tensor came back in another shape, dtype, layout or device");
    Tensor d_o = gr[0].defined() ? gr[0].to(c.rows).contiguous() : at::zeros_like(v);
    Tensor d_ov;
    if (ctx->saved_data["var"].toBool() && gr[3].defined()) d_ov = gr[3].to(c.rows).contiguous();
    const auto f32 = q.options().dtype(at::kFloat).requires_grad(false);
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v), db = at::empty_like(b);
    Tensor dgt = at::empty(gt.sizes(), f32), dg = at::empty(g.sizes(), f32), dIp = at::empty(Ip.sizes(), f32), dmu, dI;
    if (mu.defined()) { dmu = at::empty_like(mu); dI = at::empty_like(I); }
    uint32_t flags = (uint32_t)ctx->saved_data["flags"].toInt() & ~(uint32_t)PAL_FLAG_HAS_VAR;
    if (d_ov.defined()) flags |= PAL_FLAG_HAS_VAR;
    c.dims.total_chunks = (int32_t)tiles;
    c.dims.var_dtype = c.dims.dtype;
    c.dims.flags = flags;
    PalFwdTensors t{};
    t.q = ptr(q); t.k = ptr(k); t.v = ptr(v); t.b = ptr(b); t.gt = ptr(gt); t.g = (const float*)ptr(g); t.Ip = (const float*)ptr(Ip);
    t.o = (void*)ptr(d_o);
    t.init_mu = (const float*)ptr(mu); t.init_I = (const float*)ptr(I);
    if (cu.defined()) {
      t.cu_seqlens = (const int32_t*)ptr(cu);
      t.chunk_offsets = (const int32_t*)ptr(meta);
      t.chunk_table = t.chunk_offsets + c.N + 1;
    }
    t.chunk_mu = fptr(tile_mu); t.chunk_I = fptr(tile_I);
    PalBwdTensors w{};
    w.d_o = ptr(d_o); w.d_o_var = ptr(d_ov);
    w.dq = dq.mutable_data_ptr(); w.dk = dk.mutable_data_ptr(); w.dv = dv.mutable_data_ptr(); w.db = db.mutable_data_ptr();
    w.dgt = fptr(dgt); w.dg = fptr(dg); w.dIp = fptr(dIp); w.d_init_mu = fptr(dmu); w.d_init_I = fptr(dI);
    const size_t bytes = abi.chunk_bwd_workspace_bytes(&c.dims);
    Tensor ws = at::empty({(int64_t)std::max<size_t>(bytes, 16)}, q.options().dtype(at::kByte).requires_grad(false));
    int rc;
    { NoGil off; rc = abi.chunk_bwd(&c.dims, &t, &w, ws.mutable_data_ptr(), bytes, stream_of(q.device())); }
    if (rc) fail(rc, "pal_chunk_bwd");
    if (gt.scalar_type() != at::kFloat) dgt = dgt.to(gt.scalar_type());
    const Tensor none;
    return {dq, dk, dv, db, dgt, dg, dIp, dmu, dI, none, none, none, none, none, none};
  }
};

// (o, o_var | None, final_mu, final_I), or None.  meta, cu: the packed tile table (palimpsa_amd._common.chunk_meta) and the
// sequence bounds of a packed batch; window: tiles beyond which one sequence without autograd is run in segments (Python).
py::object chunk_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& b, const Tensor& gt, const Tensor& g,
                     const Tensor& Ip, const OptT& mu, const OptT& I, double scale, bool var, int64_t mode_flags, const OptT& meta,
                     const OptT& cu, int64_t window_bytes) {
  if (!unobserved() || mu.has_value() != I.has_value() || meta.has_value() != cu.has_value()) return py::none();
  if (cu && (cu->dim() != 1 || cu->numel() < 2)) return py::none();
  if (has_tangent({&q, &k, &v, &b, &gt, &g, &Ip}, mu, I)) return py::none();
  Call c(q, k, v, &b, gt, g, &Ip, scale, cu ? cu->numel() - 1 : 0);
  if (!c.ok) return py::none();
  const c10::Device dev = q.device();
  if (!plain_opt(cu, dev, at::kInt) || !plain_opt(meta, dev, at::kInt)) return py::none();
  if (!state_ok(mu, dev, c.N, c.H, c.dv, c.dk) || !state_ok(I, dev, c.N, c.H, c.dv, c.dk)) return py::none();
  const int64_t tiles = cu ? (meta->numel() - c.N - 1) / 4 : (c.T + PAL_CHUNK - 1) / PAL_CHUNK * c.B;
  if (tiles < 1 || tiles > INT32_MAX) return py::none();
  const bool grad = wants_grad({&q, &k, &v, &b, &gt, &g, &Ip}, mu, I);
  if (!grad && !cu && c.B == 1 && tiles > std::max<int64_t>(16, window_bytes / (8 * c.H * c.dv * c.dk))) return py::none();
  const uint32_t flags = (uint32_t)mode_flags | (cu ? PAL_FLAG_VARLEN : 0) | (mu ? PAL_FLAG_HAS_INIT : 0) | (var ? PAL_FLAG_HAS_VAR : 0);
  if (grad) {
    if (abi.chunk_bwd_supported((int32_t)c.dk, (int32_t)c.dv, c.dims.dtype, (uint32_t)mode_flags)) return py::none();
    try {
      auto r = ChunkNode::apply(q, k, v, b, gt, g, Ip, mu, I, meta, cu, scale, var, (int64_t)flags, tiles);
      return py::make_tuple(r[0], var ? py::cast(r[3]) : py::none(), r[1], r[2]);
    } catch (python_error& e) {
      e.restore();
      throw py::error_already_set();
    }
  }
  ChunkOut out;
  const Tensor none;
  if (chunk_forward(c, q, k, v, b, gt, g, Ip, mu.value_or(none), I.value_or(none), var, flags | PAL_FLAG_OUTPUTS_ONLY, meta.value_or(none), cu.value_or(none),
                    tiles, out))
    return py::none();
  return py::make_tuple(out.o, var ? py::cast(out.ov) : py::none(), out.fm, out.fI);
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  // what this module was built from; the loader compares it before it binds the library
  m.attr("abi") = py::make_tuple(PAL_ABI_VERSION, sizeof(PalDims), sizeof(PalFwdTensors), sizeof(PalBwdTensors));
  m.attr("torch_version") = PAL_TORCH_VERSION;
  m.def("bind", &bind);
  m.def("recurrent_fwd", &recurrent_fwd);
  m.def("gla_recurrent_fwd", &gla_recurrent_fwd);
  m.def("chunk_fwd", &chunk_fwd);
}
