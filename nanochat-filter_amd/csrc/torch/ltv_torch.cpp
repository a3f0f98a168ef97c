// Host path of the bf16 filter for PyTorch: the fused op's autograd function
// and the decode step as native code over the C ABI.
//
// The kernels of a small training step take about 120 us on MI355X; the same
// calls made from a Python autograd function took 156 to 260 us of host time (its
// backward runs on the autograd engine's device thread, which has to take the
// interpreter lock from the thread that waits for it).  Here neither direction
// holds the lock.  The work -- buffers, launches, order, results -- is that of
// ops/ltv_hm_fast.py, which keeps the library op (torch.compile), the argument
// errors and the calls this file does not take: every entry returns None where an
// input is not the plain case, and Python then goes its own way.
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <cstdlib>
#include <map>
#include <mutex>
#include <tuple>
#include <utility>

#include "../../../include/nanochat_filter_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void check(int rc, const char* what) {
  static const char* names[] = {"LTV_OK", "LTV_ERR_INVALID_ARG", "LTV_ERR_UNSUPPORTED",
                                "LTV_ERR_HIP", "LTV_ERR_WORKSPACE"};
  if (rc == 0) return;
  const std::string name = rc > 0 && rc < 5 ? names[rc] : std::to_string(rc);
  TORCH_CHECK(false, what, " failed (", name, "): ", ltv_last_error());
}

void* current_stream(const Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

// ---------------------------------------------------------------------------
// Chain workspaces: those of nanochat_amd._native (one zeroed buffer per device
// and stream, shared with the Python calls on that stream), remembered here so
// that the interpreter is only entered for a stream's first buffer or a larger
// one.  _native drops them here too when it drops its own after an error.
//
// The buffers are Python's tensors: releasing one may take the interpreter lock,
// which a thread that wants `mu` may hold.  So none is released under `mu`, and
// `mu` is never waited for with the interpreter lock held.
// ---------------------------------------------------------------------------
using ChainKey = std::pair<int, void*>;  // device, stream
struct ChainCache {
  std::mutex mu;
  std::map<ChainKey, Tensor> bufs;
  uint64_t drops = 0;  // how often all of them were dropped
};
ChainCache& chain_cache() {
  static ChainCache* c = new ChainCache;  // (outlives the interpreter and the device)
  return *c;
}

// The remembered buffer if it is large enough, and the count of drops so far.
std::pair<Tensor, uint64_t> find_chain_workspace(const ChainKey& key, size_t bytes) {
  ChainCache& c = chain_cache();
  std::lock_guard<std::mutex> lk(c.mu);
  auto it = c.bufs.find(key);
  const bool hit = it != c.bufs.end() && (size_t)it->second.numel() >= bytes;
  return {hit ? it->second : Tensor(), c.drops};
}

// Remembers buf, unless the buffers were dropped since `drops` was read (buf may
// then be one of the dropped).  The one it replaces is released by the caller.
Tensor keep_chain_workspace(const ChainKey& key, Tensor buf, uint64_t drops) {
  ChainCache& c = chain_cache();
  std::lock_guard<std::mutex> lk(c.mu);
  if (c.drops == drops) std::swap(c.bufs[key], buf);
  return buf;
}

// (called with the interpreter lock)
void drop_chain_workspaces() {
  ChainCache& c = chain_cache();
  std::map<ChainKey, Tensor> old;
  pybind11::gil_scoped_release nogil;
  {
    std::lock_guard<std::mutex> lk(c.mu);
    old.swap(c.bufs);
    ++c.drops;
  }
  old.clear();
}

// An earlier chained launch failed: let _native reset the workspaces and raise.
void raise_on_chain_error() {
  const int code = ltv_chain_take_error();
  if (code == 0) return;
  pybind11::gil_scoped_acquire gil;
  pybind11::module_::import("nanochat_amd._native").attr("raise_chain_error")(code);
}

Tensor chain_workspace(const Tensor& like, void* stream, size_t bytes) {
  if (bytes == 0) return Tensor();
  raise_on_chain_error();
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  const bool capturing = hipStreamIsCapturing((hipStream_t)stream, &cs) != hipSuccess ||
                         cs != hipStreamCaptureStatusNone;
  const ChainKey key(like.device().index(), stream);
  uint64_t drops = 0;
  if (!capturing) {
    auto [kept, n] = find_chain_workspace(key, bytes);
    if (kept.defined()) return kept;
    drops = n;
  }
  Tensor buf;
  {
    pybind11::gil_scoped_acquire gil;
    buf = pybind11::module_::import("nanochat_amd._native")
              .attr("chain_workspace")(pybind11::cast(like).attr("device"), bytes)
              .cast<Tensor>();
  }
  if (!capturing) keep_chain_workspace(key, buf, drops);
  return buf;
}

// LTV_CHAIN_SYNC_CHECK: wait for a chained call and report its failure at once.
void chain_done(const Tensor& buf, void* stream) {
  if (!buf.defined()) return;
  const char* e = std::getenv("LTV_CHAIN_SYNC_CHECK");
  if (e == nullptr || *e == 0 || (e[0] == '0' && e[1] == 0)) return;
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)stream, &cs) != hipSuccess ||
      cs != hipStreamCaptureStatusNone)
    return;
  TORCH_CHECK(hipStreamSynchronize((hipStream_t)stream) == hipSuccess,
              "hipStreamSynchronize failed after a chained scan");
  raise_on_chain_error();
}

// ---------------------------------------------------------------------------
// The fused op
// ---------------------------------------------------------------------------
struct Spec {
  int B, T, C, NH, NKVH, Da, r, P, Q, K;
  int H() const { return NH + 2 * NKVH; }
  int D() const { return Da * r; }
  int F() const { return H() * (D() + Da); }
};

struct Strides {
  int64_t s[4];
  explicit Strides(const Tensor& t) {
    for (int64_t i = 0; i < t.dim(); ++i) s[i] = t.stride(i);
  }
  Strides(int64_t a, int64_t b, int64_t c, int64_t d = 0) : s{a, b, c, d} {}
};

// (b, h, d) strides of (B, H, D) inits, or of (H, D) ones shared by every sequence
Strides inits_strides(const Tensor& t) {
  return t.dim() == 2 ? Strides(0, t.stride(0), t.stride(1))
                      : Strides(t.stride(0), t.stride(1), t.stride(2));
}
int inits_code(const Tensor& t) {
  return t.scalar_type() == at::kFloat ? LTV_DTYPE_F32 : LTV_DTYPE_BF16;
}

// values, logits, packed weight, q, k, v
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor> forward_impl(
    const Tensor& x, const Tensor& weight, const Tensor& inits, const Tensor& bias,
    const Spec& c) {
  c10::OptionalDeviceGuard guard(x.device());
  void* st = current_stream(x);
  const int H = c.H(), D = c.D();
  const auto bf = x.options().dtype(at::kBFloat16).requires_grad(false);
  const int64_t Fp = ltv_qkv_packed_width(H, D, c.Da), Lp = ltv_qkv_logit_width(H, c.Da);
  Tensor wpack = at::empty({Fp, c.C}, bf);
  check(ltv_qkv_pack_weight(weight.scalar_type() == at::kFloat ? LTV_DTYPE_F32 : LTV_DTYPE_BF16,
                            weight.data_ptr(), wpack.data_ptr(), H, D, c.Da, c.C, st),
        "ltv_qkv_pack_weight");
  Tensor values = at::empty({c.B, H, c.T, D}, bf), logits = at::empty({c.B, c.T, Lp}, bf);
  check(ltv_qkv_project_forward(x.data_ptr(), wpack.data_ptr(), values.data_ptr(),
                                logits.data_ptr(), c.B, c.T, c.C, H, D, c.Da, st),
        "ltv_qkv_project_forward");
  Tensor q = at::empty({c.B, c.NH, c.T, D}, bf), k = at::empty({c.B, c.NKVH, c.T, D}, bf),
         v = at::empty({c.B, c.NKVH, c.T, D}, bf);
  const size_t bytes =
      c.P >= c.T ? ltv_hm_scan_forward_chain_workspace_size(LTV_DTYPE_BF16, c.B, c.T, c.NH,
                                                            c.NKVH, c.Da, c.r)
                 : 0;
  const Tensor cw = chain_workspace(x, st, bytes);
  const Strides vs(values), ls(logits.stride(0), c.Da, logits.stride(1), 1),
      is = inits_strides(inits), qs(q), ks(k), os(v);
  check(ltv_hm_look_back_scan_forward_split_ws(
            LTV_DTYPE_BF16, values.data_ptr(), vs.s, logits.data_ptr(), ls.s, inits.data_ptr(),
            is.s, inits_code(inits), bias.data_ptr<float>(), q.data_ptr(), qs.s, k.data_ptr(),
            ks.s, v.data_ptr(), os.s, cw.defined() ? cw.data_ptr() : nullptr,
            cw.defined() ? (size_t)cw.numel() : 0, c.B, c.T, c.NH, c.NKVH, c.Da, c.r, c.P, c.Q,
            c.K, 1, st),
        "ltv_hm_look_back_scan_forward_split_ws");
  chain_done(cw, st);
  return {values, logits, wpack, q, k, v};
}

variable_list backward_impl(const variable_list& saved, const variable_list& grads,
                            const Spec& c) {
  // (a saved-tensor hook may hand x and the scan's tensors back in another layout)
  const Tensor x = saved[0].contiguous();
  const Tensor &wpack = saved[1], &values = saved[2], &logits = saved[3], &inits = saved[4],
               &bias = saved[5];
  c10::OptionalDeviceGuard guard(x.device());
  void* st = current_stream(x);
  const int H = c.H(), D = c.D(), F = c.F();
  const auto bf = x.options().dtype(at::kBFloat16).requires_grad(false);
  const auto f32 = bf.dtype(at::kFloat);
  Tensor g[3];
  for (int i = 0; i < 3; ++i) {
    // upstream gradients keep their strides: the scan reads any layout
    g[i] = grads[i].defined() ? grads[i] : at::zeros_like(saved[6 + i]);
    if (g[i].scalar_type() != at::kBFloat16) g[i] = g[i].to(at::kBFloat16);
  }
  const int64_t Fp = wpack.size(0);
  Tensor gc = at::empty({c.B, c.T, Fp}, bf);
  Tensor gi = at::empty(inits.sizes(), inits.options().requires_grad(false));
  Tensor gb = at::empty({H, c.Da}, f32);
  const size_t wsb = ltv_hm_look_back_scan_backward_workspace_size(
      LTV_DTYPE_BF16, c.B, c.T, c.NH, c.NKVH, c.Da, c.r, c.P, c.Q, c.K);
  Tensor ws = at::empty({(int64_t)std::max<size_t>(wsb, 1)}, bf.dtype(at::kByte));
  size_t bytes = 0;
  if (c.P >= c.T &&
      ltv_hm_scan_backward_chain_pays(LTV_DTYPE_BF16, c.B, c.T, c.NH, c.NKVH, c.Da, c.r))
    bytes = ltv_hm_scan_backward_chain_workspace_size(LTV_DTYPE_BF16, c.B, c.T, c.NH, c.NKVH,
                                                      c.Da, c.r);
  const Tensor cw = chain_workspace(x, st, bytes);
  const Strides vs(values),
      ls(logits.stride(0), c.Da * logits.stride(2), logits.stride(1), logits.stride(2)),
      is = inits_strides(inits), gis = inits_strides(gi), hq(saved[6]), hk(saved[7]),
      hv(saved[8]), gq(g[0]), gk(g[1]), gv(g[2]);
  const Strides gvs(c.T * Fp, D, Fp, 1), gls(c.T * Fp, c.Da, Fp, 1);
  check(ltv_hm_look_back_scan_backward_split_ws(
            LTV_DTYPE_BF16, values.data_ptr(), vs.s, logits.data_ptr(), ls.s, inits.data_ptr(),
            is.s, inits_code(inits), bias.data_ptr<float>(), saved[6].data_ptr(), hq.s,
            saved[7].data_ptr(), hk.s, saved[8].data_ptr(), hv.s, g[0].data_ptr(), gq.s,
            g[1].data_ptr(), gk.s, g[2].data_ptr(), gv.s, gc.data_ptr(), gvs.s,
            static_cast<char*>(gc.data_ptr()) + (int64_t)H * D * 2, gls.s, (8 - F % 8) % 8,
            gi.data_ptr(), gis.s, gb.data_ptr<float>(), ws.data_ptr(), wsb,
            cw.defined() ? cw.data_ptr() : nullptr, cw.defined() ? (size_t)cw.numel() : 0, c.B,
            c.T, c.NH, c.NKVH, c.Da, c.r, c.P, c.Q, c.K, 1, st),
        "ltv_hm_look_back_scan_backward_split_ws");
  chain_done(cw, st);
  const int M = c.B * c.T;
  Tensor gx = at::empty({c.B, c.T, c.C}, bf), gw = at::empty({F, c.C}, f32);
  const size_t pwb = ltv_qkv_project_backward_workspace_size(M, c.C, H, D, c.Da);
  Tensor pws = at::empty({(int64_t)std::max<size_t>(pwb, 1)}, bf.dtype(at::kByte));
  check(ltv_qkv_project_backward_zero_padded(x.data_ptr(), wpack.data_ptr(), gc.data_ptr(),
                                             gx.data_ptr(), gw.data_ptr<float>(), pws.data_ptr(),
                                             pwb, M, c.C, H, D, c.Da, st),
        "ltv_qkv_project_backward_zero_padded");
  return {gx, gw, gi, gb};
}

class QkvFilter : public torch::autograd::Function<QkvFilter> {
 public:
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight,
                               const Tensor& inits, const Tensor& bias, int64_t NH, int64_t NKVH,
                               int64_t Da, int64_t r, int64_t P, int64_t Q, int64_t K) {
    const Spec c{(int)x.size(0), (int)x.size(1), (int)x.size(2), (int)NH, (int)NKVH, (int)Da,
                 (int)r,         (int)P,         (int)Q,         (int)K};
    auto [values, logits, wpack, q, k, v] = forward_impl(x, weight, inits, bias, c);
    ctx->save_for_backward({x, wpack, values, logits, inits, bias, q, k, v});
    ctx->saved_data["spec"] = std::vector<int64_t>{NH, NKVH, Da, r, P, Q, K};
    ctx->saved_data["weight_f32"] = weight.scalar_type() == at::kFloat;
    ctx->saved_data["bias_shape"] = bias.sizes().vec();
    ctx->set_materialize_grads(false);
    return {q, k, v};
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list saved = ctx->get_saved_variables();
    const auto a = ctx->saved_data["spec"].toIntVector();
    const Tensor& x = saved[0];
    const Spec c{(int)x.size(0), (int)x.size(1), (int)x.size(2), (int)a[0], (int)a[1], (int)a[2],
                 (int)a[3],      (int)a[4],      (int)a[5],      (int)a[6]};
    variable_list g = backward_impl(saved, grads, c);
    if (!ctx->saved_data["weight_f32"].toBool()) g[1] = g[1].to(at::kBFloat16);
    g[3] = g[3].view(ctx->saved_data["bias_shape"].toIntVector());
    g.resize(11);
    return g;
  }
};

bool plain(const Tensor& t) { return t.defined() && t.is_cuda() && t.layout() == at::kStrided; }

// Tensors of the ordinary kind, with no tracer, mode or transform looking on.
bool ordinary(at::ArrayRef<Tensor> ts) {
  return !at::areAnyTensorSubclassLike(ts) && !torch::jit::tracer::isTracing();
}

// (q, k, v), each (B, nh, T, D), or None where the inputs are not the plain case.
pybind11::object qkv_filter(const Tensor& x, const Tensor& weight, const Tensor& inits,
                            const Tensor& bias, int64_t NH, int64_t NKVH, int64_t Da, int64_t r,
                            int64_t P, int64_t Q, int64_t K) {
  const int64_t H = NH + 2 * NKVH, D = Da * r;
  if (!plain(x) || !plain(weight) || !plain(inits) || !plain(bias) ||
      !ordinary({x, weight, inits, bias}))
    return pybind11::none();
  const auto dev = x.device();
  auto f32_or_bf16 = [](const Tensor& t) {
    return t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16;
  };
  const bool ok =
      NH > 0 && NKVH > 0 && Da > 0 && r > 0 && x.dim() == 3 && x.numel() > 0 &&
      x.scalar_type() == at::kBFloat16 && x.is_contiguous() && weight.device() == dev &&
      weight.dim() == 2 && weight.size(0) == H * (D + Da) && weight.size(1) == x.size(2) &&
      f32_or_bf16(weight) && weight.is_contiguous() && inits.device() == dev &&
      f32_or_bf16(inits) &&
      ((inits.dim() == 2 && inits.size(0) == H && inits.size(1) == D) ||
       (inits.dim() == 3 && inits.size(0) == x.size(0) && inits.size(1) == H &&
        inits.size(2) == D)) &&
      bias.device() == dev && bias.scalar_type() == at::kFloat && bias.is_contiguous() &&
      bias.numel() == H * Da && x.size(0) * x.size(1) < (int64_t(1) << 31);
  if (!ok) return pybind11::none();
  variable_list out;
  {
    pybind11::gil_scoped_release nogil;
    out = QkvFilter::apply(x, weight, inits, bias, NH, NKVH, Da, r, P, Q, K);
  }
  return pybind11::make_tuple(out[0], out[1], out[2]);
}

// One decode step from the previous rows q, k, v (B, nh, D), which receive the
// new ones: the new rows as (B, 1, nh, D) views, or None where the inputs are
// not the plain case.
pybind11::object decode_rows(const Tensor& x, const Tensor& wpack, const Tensor& q,
                             const Tensor& k, const Tensor& v, const Tensor& bias, int64_t NH,
                             int64_t NKVH, int64_t Da, int64_t r) {
  const int64_t H = NH + 2 * NKVH, D = Da * r;
  if (!plain(x) || x.dim() != 3 || x.size(1) != 1 || x.size(0) == 0 ||
      x.scalar_type() != at::kBFloat16 || x.stride(2) != 1 || x.stride(0) % 8 != 0 ||
      x.requires_grad() || !plain(bias) || bias.scalar_type() != at::kFloat ||
      !bias.is_contiguous() || bias.numel() != H * Da || !ordinary({x, wpack, q, k, v, bias}))
    return pybind11::none();
  const int64_t B = x.size(0), C = x.size(2);
  const Tensor* prev[3] = {&q, &k, &v};
  int64_t st[6];
  for (int i = 0; i < 3; ++i) {
    const Tensor& t = *prev[i];
    if (!plain(t) || t.device() != x.device() || t.scalar_type() != at::kBFloat16 ||
        t.dim() != 3 || t.size(0) != B || t.size(1) != (i == 0 ? NH : NKVH) || t.size(2) != D ||
        t.stride(2) != 1)
      return pybind11::none();
    st[2 * i] = t.stride(0);
    st[2 * i + 1] = t.stride(1);
  }
  if (!plain(wpack) || wpack.device() != x.device() || bias.device() != x.device() ||
      wpack.scalar_type() != at::kBFloat16 || wpack.dim() != 2 || !wpack.is_contiguous() ||
      wpack.size(0) != ltv_qkv_packed_width(H, D, Da) || wpack.size(1) != C)
    return pybind11::none();
  c10::OptionalDeviceGuard guard(x.device());
  Tensor out = at::empty({B, 1, H, D}, x.options());
  const int rc = ltv_qkv_decode_step_rows(
      x.data_ptr(), x.stride(0), wpack.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), st,
      bias.data_ptr<float>(), out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), st,
      (int)B, (int)C, (int)NH, (int)NKVH, (int)D, (int)Da, 1, current_stream(x));
  check(rc, "ltv_qkv_decode_step_rows");
  return pybind11::make_tuple(out.narrow(2, 0, NH), out.narrow(2, NH, NKVH),
                              out.narrow(2, NH + NKVH, NKVH));
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("qkv_filter", &qkv_filter);
  m.def("decode_rows", &decode_rows);
  m.def("drop_chain_workspaces", &drop_chain_workspaces);
  // the workspace cache by itself, any tensors (its locking is tested without a device)
  m.def("_find_chain_workspace", [](int device, int64_t stream, size_t bytes) {
    return find_chain_workspace({device, reinterpret_cast<void*>(stream)}, bytes);
  }, pybind11::call_guard<pybind11::gil_scoped_release>());
  m.def("_keep_chain_workspace", [](int device, int64_t stream, Tensor buf, uint64_t drops) {
    keep_chain_workspace({device, reinterpret_cast<void*>(stream)}, std::move(buf), drops);
  }, pybind11::call_guard<pybind11::gil_scoped_release>());
}
