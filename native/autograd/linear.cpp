// The autograd node of kgs.ops.Linear for layers that the host bounds: forward and backward each in
// one call, the backward pass without the interpreter.
//
// A small layer's kernels take less time than the host's work for them: three layers of 64 rows, 512 - 2048 -
// 512, forward 67 us and with the backward pass 329 as Python autograd.Functions (the engine's thread takes
// the interpreter's lock for each node and again after each launch), 28 and 153 here; a training step of
// them 411 / 207, of which the kernels are 115. The kernels and their order are those of
// kgs/ops/gemm.py's _LinearFn, so are the results; that one stays for what this one hands back: products
// that run on transposed copies (tr_slices 0: such sizes keep the GPU busy for longer than the
// host), operands that only the element-wise kernel reads, empty ones, and whatever has to see a Python
// function (tracing, functorch transforms, forward-mode tangents, dispatch modes, tensor subclasses).
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <string>

namespace {

// libkgs_kernels.so's entry points, bound from the library that Python loaded
typedef int (*NtAuto)(const void*, const void*, void*, const void*, int, int, int, int, int, int, int, float*, hipStream_t);
typedef int (*NtPadded)(const void*, const void*, void*, const void*, int, int, int, int, int, int, int, void*, hipStream_t);
typedef int (*NtAct)(const void*, const void*, void*, void*, const void*, int, int, int, int, int, int, int, float*, hipStream_t);
typedef int (*PadRows)(const void*, void*, long, int, long, const void*, void*, long, int, long, hipStream_t);
typedef int (*ActGrad)(const void*, const void*, void*, void*, float*, void*, int, int, int, int, hipStream_t);
typedef int (*Tr)(const void*, const void*, void*, int, int, int, int, int, int, int, int, int, float*, hipStream_t);
typedef int (*TrPair)(const void*, const void*, const void*, void*, void*, int, int, int, int, int, int, int, int, float*, float*, hipStream_t);
typedef long (*Scratch)(int, int, int);
typedef long (*PaddedScratch)(int, int, int, int, int);
typedef int (*Parts)(int, int);
typedef int (*TrSlices)(int, int, int, int, int);

struct Entries {
  NtAuto nt_auto;
  NtPadded nt_padded;
  NtAct nt_act;
  PadRows pad_rows;
  ActGrad act_grad;
  Tr tr;
  TrPair tr_pair;
  Scratch scratch;
  PaddedScratch padded_scratch;
  Parts parts;
  TrSlices tr_slices;
} so;

constexpr int NONE = 0, BIAS = 1, GELU = 2, SILU = 4;  // the kernels' epilogues

void check(int rc, const char* what, long m, long n, long k) {
  TORCH_CHECK(rc == 0, what, "[", m, "x", n, "x", k, "]: error ", rc);
}

at::Tensor fresh(const at::Tensor& like, at::IntArrayRef size, at::ScalarType type = at::kBFloat16) {
  return at::empty(size, like.options().dtype(type));
}

template <class T = void>
T* ptr(const at::Tensor& t) {
  return t.defined() ? (T*)t.data_ptr() : nullptr;
}

bool rows16(const at::Tensor& t) { return t.stride(0) % 8 == 0 && (uintptr_t)t.data_ptr() % 16 == 0; }

bool odd(const at::Tensor& t) { return t.size(1) % 8 || !rows16(t); }

// kgs/ops/gemm.py _pads: whether odd rows are copied into padded ones for the fast tiles
bool pads(long m, long n, long k) { return k > (m * n <= 4096 ? 128 : std::min(m, n) <= 96 ? 64 : 32); }

// Zero-padded copies of the matrices whose rows are not whole, aligned 16-byte chunks; one launch.
void even(at::Tensor* a, at::Tensor* b, hipStream_t s) {
  at::Tensor* both[2] = {a, b};
  at::Tensor src[2], *dst[2];
  int n = 0;
  for (at::Tensor* t : both)
    if (t && odd(*t)) {
      src[n] = *t;
      *t = fresh(*t, {t->size(0), (t->size(1) + 7) / 8 * 8});
      dst[n++] = t;
    }
  if (!n) return;
  const bool two = n > 1;
  check(so.pad_rows(ptr(src[0]), ptr(*dst[0]), src[0].size(0), (int)src[0].size(1), src[0].stride(0), two ? ptr(src[1]) : nullptr,
                    two ? ptr(*dst[1]) : nullptr, two ? src[1].size(0) : 0, two ? (int)src[1].size(1) : 0,
                    two ? src[1].stride(0) : 0, s),
        "pad_rows", src[0].size(0), src[0].size(1), n);
}

// act(a . b^T + bias)
at::Tensor product(const at::Tensor& a, const at::Tensor& b, at::Tensor bias, int epi, hipStream_t s) {
  const int m = (int)a.size(0), n = (int)b.size(0), k = (int)a.size(1), lda = (int)a.stride(0), ldb = (int)b.stride(0);
  if (epi == NONE && bias.defined()) epi = BIAS;
  if (epi && !bias.defined()) bias = at::zeros({n}, a.options());
  const at::Tensor out = fresh(a, {m, n});
  const bool oa = odd(a), ob = odd(b);
  if (oa || ob) {
    const at::Tensor ws = fresh(a, {std::max(4L, so.padded_scratch(m, n, k, oa, ob))}, at::kFloat);
    check(so.nt_padded(ptr(a), ptr(b), ptr(out), ptr(bias), m, n, k, lda, ldb, n, epi, ptr(ws), s), "gemm_nt", m, n, k);
  } else {
    const long need = so.scratch(m, n, k);
    const at::Tensor ws = need ? fresh(a, {need}, at::kFloat) : at::Tensor();
    check(so.nt_auto(ptr(a), ptr(b), ptr(out), ptr(bias), m, n, k, lda, ldb, n, epi, ptr<float>(ws), s), "gemm_nt", m, n, k);
  }
  return out;
}

// room for the ns partial sums of an [m, n] product in K slices, none for a whole one
at::Tensor slices(const at::Tensor& like, int ns, long m, long n) {
  return ns > 1 ? fresh(like, {ns * m * ((n + 7) / 8 * 8)}, at::kFloat) : at::Tensor();
}

// op(a) . b over k on tiles that read K-major operands in place (a: [k, m] if ta; b: [k, n]), a's rows lda apart
at::Tensor product_tr(const at::Tensor& a, int lda, const at::Tensor& b, int m, int n, int k, int ta, hipStream_t s) {
  const int ns = so.tr_slices(m, n, k, ta, 1);
  const at::Tensor out = fresh(a, {m, n});
  const at::Tensor ws = slices(a, ns, m, n);
  check(so.tr(ptr(a), ptr(b), ptr(out), m, n, k, lda, (int)b.stride(0), n, ta, 1, ns, ptr<float>(ws), s), "gemm_tr", m, n, k);
  return out;
}

// product_tr is the way to a product whose operands' rows are lda and ldb long (once padded)
bool by_tr(long m, long n, long k, long lda, long ldb, int ta) {
  return (k + 128) * std::max(lda, ldb) < 1L << 30 && so.tr_slices((int)m, (int)n, (int)k, ta, 1) > 0;
}

long padded(const at::Tensor& t) { return odd(t) ? (t.size(1) + 7) / 8 * 8 : t.stride(0); }

// A matrix that a kernel may read without Python's having a say
bool plain(const at::Tensor& t, int64_t dim) {
  return t.defined() && t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.layout() == at::kStrided && t.dim() == dim &&
         t.numel() > 0 && t.stride(dim - 1) == 1 && !t.unsafeGetTensorImpl()->key_set().has(c10::DispatchKey::Python) &&
         !t._fw_grad(0).defined();
}

// A saved tensor as the kernels read it: hooks may have put another one in its place
at::Tensor loaded(const at::Tensor& t, int64_t m, int64_t n, const at::Tensor& gy) {
  TORCH_CHECK(t.is_cuda() && t.device() == gy.device() && t.scalar_type() == at::kBFloat16 && t.dim() == 2 && t.size(0) == m &&
                  t.size(1) == n,
              "linear backward: a saved tensor came back as ", t.toString(), " ", t.sizes(), " on ", t.device());
  return t.stride(1) == 1 && t.stride(0) >= n ? t : t.contiguous();
}

struct LinearNode : torch::autograd::Function<LinearNode> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& x, const at::Tensor& w,
                            const std::optional<at::Tensor>& given, int64_t act, bool train) {
    const at::Tensor bias = given ? *given : at::Tensor();
    const c10::DeviceGuard guard(x.device());
    const hipStream_t s = c10::hip::getCurrentHIPStream(x.get_device()).stream();
    ctx->saved_data["act"] = act;
    if (act == NONE || !train) {
      ctx->save_for_backward({x, w, bias, at::Tensor()});
      return product(x, w, bias, (int)act, s);
    }
    // training keeps the pre-activation for the backward pass
    at::Tensor a = x, b = w;
    if (odd(a) || odd(b)) even(&a, &b, s);
    const int m = (int)a.size(0), n = (int)b.size(0), k = (int)a.size(1);
    const at::Tensor z = fresh(x, {m, n}), y = fresh(x, {m, n});
    const long need = so.scratch(m, n, k);
    const at::Tensor ws = need ? fresh(x, {need}, at::kFloat) : at::Tensor();
    check(so.nt_act(ptr(a), ptr(b), ptr(z), ptr(y), ptr(bias), m, n, k, (int)a.stride(0), (int)b.stride(0), n, (int)act,
                    ptr<float>(ws), s),
          "gemm_nt_act", m, n, k);
    ctx->save_for_backward({x, w, bias, z});
    return y;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const at::Tensor gy = grads[0].contiguous(), bias = saved[2];
    const c10::DeviceGuard guard(gy.device());
    const hipStream_t s = c10::hip::getCurrentHIPStream(gy.get_device()).stream();
    const int m = (int)gy.size(0), n = (int)gy.size(1), k = (int)saved[0].size(1), ld = (n + 7) / 8 * 8;
    at::Tensor x = loaded(saved[0], m, k, gy), w = loaded(saved[1], n, k, gy);
    const at::Tensor z = saved[3].defined() ? loaded(saved[3], m, n, gy).contiguous() : at::Tensor();
    const int act = z.defined() ? (int)ctx->saved_data["act"].toInt() : NONE;
    const bool need_x = ctx->needs_input_grad(0), need_w = ctx->needs_input_grad(1),
               need_b = bias.defined() && ctx->needs_input_grad(2);
    // the gradient through the activation, in rows of whole 16-byte chunks, and its column sums
    const bool copy = act != NONE || ld != n || (uintptr_t)gy.data_ptr() % 16;
    const at::Tensor gz = copy ? fresh(gy, {m, ld}) : gy, gb = need_b ? fresh(gy, {n}) : at::Tensor();
    if (copy || need_b) {
      const int parts = need_b ? so.parts(m, n) : 1;
      const at::Tensor part = parts > 1 ? fresh(gy, {parts, n}, at::kFloat) : at::Tensor();
      check(so.act_grad(ptr(gy), act ? ptr(z) : nullptr, copy ? ptr(gz) : nullptr, nullptr, ptr<float>(part), ptr(gb), m, n, ld, act, s),
            "act_grad", m, n, 0);
    }
    even(need_w ? &x : nullptr, need_x ? &w : nullptr, s);
    at::Tensor gx, gw;
    if (need_x && need_w) {  // both from one launch
      const int nsx = so.tr_slices(m, k, n, 0, 1), nsw = so.tr_slices(n, k, m, 1, 1);
      gx = fresh(gz, {m, k});
      gw = fresh(gz, {n, k});
      const at::Tensor wsx = slices(gz, nsx, m, k), wsw = slices(gz, nsw, n, k);
      check(so.tr_pair(ptr(gz), ptr(w), ptr(x), ptr(gx), ptr(gw), m, n, k, ld, (int)w.stride(0), (int)x.stride(0), nsx, nsw,
                       ptr<float>(wsx), ptr<float>(wsw), s),
            "gemm_tr_pair", m, n, k);
      return {gx, gw, gb, at::Tensor(), at::Tensor()};
    }
    if (need_x) gx = product_tr(gz, ld, w, m, k, n, 0, s);  // dX[m, k] = dY[m, n] . W[n, k]
    if (need_w) gw = product_tr(gz, ld, x, n, k, m, 1, s);  // dW[n, k] = dY[m, n]^T . X[m, k]
    return {gx, gw, gb, at::Tensor(), at::Tensor()};
  }
};

// A functorch transform is running on this thread (its thread-local storage stays behind when it has ended)
bool transforming() {
  return c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerBackMode);
}

// act(x . w^T + bias), or None where kgs/ops/gemm.py's _LinearFn has to run it (or say what is wrong)
std::optional<at::Tensor> linear(const at::Tensor& x, const at::Tensor& w, const std::optional<at::Tensor>& b, int64_t act) {
  const at::Tensor bias = b ? *b : at::Tensor();
  if (!(act == NONE || (act >= GELU && act <= SILU)) || !plain(x, 2) || !plain(w, 2) || (b && !plain(bias, 1))) return {};
  if (torch::jit::tracer::isTracing() || transforming() || c10::impl::TorchDispatchModeTLS::any_modes_set()) return {};
  const long m = x.size(0), k = x.size(1), n = w.size(0), lim = 1L << 22;
  if (w.size(1) != k || w.device() != x.device() || (b && (bias.numel() != n || bias.device() != x.device()))) return {};
  if (m >= 1L << 24 || x.stride(0) < k || w.stride(0) < k || std::max({n, x.stride(0), w.stride(0)}) >= lim) return {};
  if ((odd(x) || odd(w)) && !pads(m, n, k)) return {};
  const bool gx = x.requires_grad(), gw = w.requires_grad(), train = gx || gw || (b && bias.requires_grad());
  const long ld = (n + 7) / 8 * 8;
  if (train && at::GradMode::is_enabled() &&
      ((gx && !by_tr(m, k, n, ld, padded(w), 0)) || (gw && !by_tr(n, k, m, ld, padded(x), 1))))
    return {};
  return LinearNode::apply(x, w, b, act, train);
}

template <class F>
void bind(F& f, const py::dict& d, const char* name) {
  f = (F)d[name].cast<uintptr_t>();
}

}  // namespace

PYBIND11_MODULE(_autograd, mod) {
  mod.def("bind", [](const py::dict& d) {
    bind(so.nt_auto, d, "kgs_gemm_bf16_nt_auto");
    bind(so.nt_padded, d, "kgs_gemm_bf16_nt_padded");
    bind(so.nt_act, d, "kgs_gemm_bf16_nt_act");
    bind(so.pad_rows, d, "kgs_pad_rows_bf16");
    bind(so.act_grad, d, "kgs_act_grad");
    bind(so.tr, d, "kgs_gemm_bf16_tr");
    bind(so.tr_pair, d, "kgs_gemm_bf16_tr_pair");
    bind(so.scratch, d, "kgs_gemm_bf16_nt_scratch");
    bind(so.padded_scratch, d, "kgs_gemm_bf16_nt_padded_scratch");
    bind(so.parts, d, "kgs_act_grad_parts");
    bind(so.tr_slices, d, "kgs_gemm_bf16_tr_slices");
  }, "The kernels' addresses by name; to be called once, first.");
  mod.def("linear", &linear, py::arg("x"), py::arg("w"), py::arg("bias"), py::arg("act"), py::call_guard<py::gil_scoped_release>());
}
