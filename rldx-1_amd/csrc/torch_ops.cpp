// Native dispatch of the torch.library operators (rldx_amd/ops.py) on the GPU.
//
// The operators are defined, with their argument checks, fake implementations
// and autograd behaviour, in Python; a call there spends 15-19 us of host time
// (dispatcher -> Python twice, checks, ctypes) on kernels that run 8-12 us.
// This library registers C++ kernels under the CUDA and AutogradCUDA keys of the
// same operators: the common forms of a call (the tensors' types and layouts
// below) are checked and launched here, everything else -- other layouts, wrong
// arguments, inputs that need a gradient -- is handed to the Python
// implementation, which keeps its behaviour and its error messages.
#include <ATen/core/Tensor.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/Event.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include <atomic>
#include <cmath>
#include <memory>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "rldx_amd.h"

namespace {

using at::Tensor;
using c10::SymInt;
using OptTensor = std::optional<Tensor>;

// ---- argument forms the native path takes ----
bool bf16(const Tensor& t) { return t.is_cuda() && t.scalar_type() == at::kBFloat16; }
bool rows2d(const Tensor& t) { return bf16(t) && t.dim() == 2 && t.stride(1) == 1; }
bool vec(const Tensor& t, int64_t n) { return bf16(t) && t.numel() == n && t.is_contiguous(); }
bool table(const Tensor& t, int64_t rows, int64_t cols) {  // fp32 [>= rows, cols]
  return t.is_cuda() && t.scalar_type() == at::kFloat && t.dim() == 2 && t.is_contiguous() && t.size(0) >= rows &&
         t.size(1) == cols;
}
template <class... T>
bool one_device(const Tensor& a, const T&... rest) {
  return ((rest.device() == a.device()) && ...);
}
hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
Tensor bytes_like(const Tensor& t, int64_t n) {
  return at::empty({n < 16 ? 16 : n}, t.options().dtype(at::kByte));
}

// ---- dispatch helpers ----
template <class Sig>
c10::TypedOperatorHandle<Sig> handle(const char* name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").template typed<Sig>();
}
// the Python implementation (registered for every backend; the CPU key's table entry is it)
constexpr c10::DispatchKeySet kPython(c10::DispatchKey::CPU);

bool needs_autograd(const Tensor& t) {
  if (!t.defined() || t.unsafeGetTensorImpl()->autograd_meta() == nullptr) return false;
  return (c10::GradMode::is_enabled() && t.requires_grad()) || t._fw_grad(0).defined();
}
bool needs_autograd(const OptTensor& t) { return t.has_value() && needs_autograd(*t); }
template <class T>
bool needs_autograd(const T&) { return false; }

// The AutogradCUDA kernel of an operator: no input needs a gradient -> the
// kernel below autograd; otherwise the Python autograd implementation (any other
// backend's autograd table entry), which refuses the backward pass.
template <class Tag, class Sig>
struct Autograd;
template <class Tag, class R, class... A>
struct Autograd<Tag, R(A...)> {
  static R call(c10::DispatchKeySet ks, A... a) {
    static auto op = handle<R(A...)>(Tag::name);
    if ((needs_autograd(a) || ...)) return op.redispatch(ks.add(c10::DispatchKey::AutogradXPU), a...);
    return op.redispatch(ks & c10::after_autograd_keyset, a...);
  }
};
template <class Tag, class R, class... A>
R python(A... a) {
  static auto op = handle<R(A...)>(Tag::name);
  return op.redispatch(kPython, a...);
}

#define RLDX_OP(TAG, NAME) \
  struct TAG {             \
    static constexpr const char* name = NAME; \
  }

// ---------------------------------------------------------------------------
// VLM, vision, memory attention
// ---------------------------------------------------------------------------
RLDX_OP(Gqa, "rldx_backbone::fused_attention");
Tensor gqa(const Tensor& qkv, const Tensor& qw, const Tensor& qwr, const Tensor& kw, const Tensor& kwr,
           const Tensor& cos, const Tensor& sin, SymInt hq_, SymInt hkv_, SymInt d_) {
  const int64_t hq = hq_.guard_int(__FILE__, __LINE__), hkv = hkv_.guard_int(__FILE__, __LINE__),
                D = d_.guard_int(__FILE__, __LINE__);
  if (rows2d(qkv) && one_device(qkv, qw, kw, cos, sin) && vec(qw, D) && vec(kw, D) && rows2d(cos) && rows2d(sin)) {
    const int64_t M = qkv.size(0);
    if (M > 0 && hq > 0 && hkv > 0 && D > 0 && qkv.size(1) >= (hq + 2 * hkv) * D && cos.size(0) == M &&
        cos.size(1) == D && sin.sizes() == cos.sizes() && sin.stride(0) == cos.stride(0)) {
      const c10::OptionalDeviceGuard guard(qkv.device());
      const int64_t need = rldx_llm_fused_attention_workspace_bytes(M, hkv, D);
      if (need >= 0) {
        Tensor out = at::empty({M, hq * D}, qkv.options()), ws = bytes_like(qkv, need);
        if (rldx_llm_fused_attention_bf16(qkv.data_ptr(), qkv.stride(0), qw.data_ptr(), kw.data_ptr(), cos.data_ptr(),
                                          sin.data_ptr(), cos.stride(0), 1, out.data_ptr(), hq * D, M, hq, hkv, D,
                                          1e-6f, ws.data_ptr(), ws.numel(), stream_of(qkv)) == hipSuccess)
          return out;
      }
    }
  }
  return python<Gqa, Tensor, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                const Tensor&, SymInt, SymInt, SymInt>(qkv, qw, qwr, kw, kwr, cos, sin, hq_, hkv_, d_);
}

RLDX_OP(Vit, "rldx_backbone::vision_attention");
Tensor vit(const Tensor& qkv, const Tensor& cos, const Tensor& sin, const Tensor& cu, double scaling, SymInt h_,
           SymInt d_) {
  const int64_t H = h_.guard_int(__FILE__, __LINE__), D = d_.guard_int(__FILE__, __LINE__);
  if (rows2d(qkv) && qkv.is_contiguous() && one_device(qkv, cos, sin, cu) && qkv.size(1) == 3 * H * D && H > 0 && D > 0 &&
      cu.scalar_type() == at::kInt && cu.dim() == 1 && cu.numel() >= 2 && cu.is_contiguous()) {
    const int64_t M = qkv.size(0), S = cu.numel() - 1;
    if (M > 0 && table(cos, M, D) && table(sin, M, D) && cos.size(0) == M && sin.size(0) == M) {
      const c10::OptionalDeviceGuard guard(qkv.device());
      const int64_t need = rldx_vision_attention_workspace_bytes(M, S, H, D);
      if (need >= 0) {
        Tensor out = at::empty({M, H * D}, qkv.options()), ws = bytes_like(qkv, need);
        if (rldx_vision_attention_bf16(qkv.data_ptr(), cos.data_ptr<float>(), sin.data_ptr<float>(),
                                       cu.data_ptr<int32_t>(), S, out.data_ptr(), M, H, D, static_cast<float>(scaling),
                                       ws.data_ptr(), ws.numel(), stream_of(qkv)) == hipSuccess)
          return out;
      }
    }
  }
  return python<Vit, Tensor, const Tensor&, const Tensor&, const Tensor&, const Tensor&, double, SymInt, SymInt>(
      qkv, cos, sin, cu, scaling, h_, d_);
}

RLDX_OP(Mem, "mem::fused_attention");
Tensor mem(const Tensor& qkv, const Tensor& cos, const Tensor& sin, SymInt h_, SymInt d_, SymInt b_) {
  const int64_t H = h_.guard_int(__FILE__, __LINE__), D = d_.guard_int(__FILE__, __LINE__),
                B = b_.guard_int(__FILE__, __LINE__);
  if (rows2d(qkv) && qkv.is_contiguous() && one_device(qkv, cos, sin) && H > 0 && B > 0 &&
      (D == 64 || D == 128 || D == 256) && qkv.size(0) > 0 && qkv.size(1) == 3 * H * D) {
    const int64_t M = qkv.size(0);
    if (vec(cos, M * D) && vec(sin, M * D) && cos.dim() == 2 && sin.dim() == 2 && cos.size(0) == M && sin.size(0) == M) {
      const c10::OptionalDeviceGuard guard(qkv.device());
      Tensor out = at::empty({M, H * D}, qkv.options());
      if (rldx_memory_attention_bf16(qkv.data_ptr(), cos.data_ptr(), sin.data_ptr(), out.data_ptr(), M, H, D, B,
                                     stream_of(qkv)) == hipSuccess)
        return out;
    }
  }
  return python<Mem, Tensor, const Tensor&, const Tensor&, const Tensor&, SymInt, SymInt, SymInt>(qkv, cos, sin, h_, d_,
                                                                                                  b_);
}

// ---------------------------------------------------------------------------
// MSAT joint attention
// ---------------------------------------------------------------------------
// Rows [first, first + n) of packed QKV (2-D rows, or contiguous with leading
// dimensions) as a stream; cos / sin: rope tables or null.
bool qkv_rows(const Tensor& t) { return bf16(t) && t.dim() >= 2 && (t.dim() == 2 ? t.stride(1) == 1 : t.is_contiguous()); }
int64_t rows_of(const Tensor& t) { return t.dim() == 2 ? t.size(0) : t.numel() / t.size(-1); }
int64_t ld_of(const Tensor& t) { return t.dim() == 2 ? t.stride(0) : t.size(-1); }

bool stream(const Tensor& ref, const Tensor& qkv, int64_t first, int64_t n, int64_t inner, const Tensor& qw,
            const Tensor& kw, const Tensor* cos, const Tensor* sin, int64_t D, rldx_msat_stream_t& s) {
  if (n < 0 || first < 0 || !one_device(ref, qkv, qw, kw) || !vec(qw, D) || !vec(kw, D) || qkv.numel() == 0 ||
      !qkv_rows(qkv) || qkv.size(-1) < 3 * inner || rows_of(qkv) < first + n)
    return false;
  if (cos && (!one_device(ref, *cos, *sin) || !table(*cos, n, D / 2) || !table(*sin, n, D / 2) ||
              cos->sizes() != sin->sizes()))
    return false;
  s = rldx_msat_stream_t{static_cast<const char*>(qkv.data_ptr()) + first * ld_of(qkv) * 2, ld_of(qkv), n,
                         qw.data_ptr(), kw.data_ptr(), cos ? cos->data_ptr<float>() : nullptr,
                         cos ? sin->data_ptr<float>() : nullptr, cos ? cos->stride(0) : 0};
  return true;
}

// QK norm + RoPE + K/V tiles, then the attention; an undefined tensor if the call is not one of the native forms.
Tensor joint(const Tensor& ref, const rldx_msat_stream_t* s, int n, const OptTensor& mask, int64_t H, int64_t D) {
  int64_t M = 0;
  for (int i = 0; i < n; ++i) M += s[i].rows;
  if (M == 0 || H <= 0 || !(D == 64 || D == 128)) return Tensor();
  const float* mp = nullptr;
  if (mask.has_value()) {
    const Tensor& m = *mask;
    if (!one_device(ref, m) || m.scalar_type() != at::kFloat || !(m.dim() == 1 || (m.dim() == 2 && m.size(0) == 1)) ||
        m.stride(-1) != 1 || m.size(-1) != M)
      return Tensor();
    mp = m.data_ptr<float>();
  }
  const c10::OptionalDeviceGuard guard(ref.device());
  const int64_t elems = rldx_attention_kv_packed_elems(M, D), inner = H * D;
  Tensor q = at::empty({H, M, D}, ref.options()), kvp = at::empty({H, elems}, ref.options()),
         out = at::empty({1, M, inner}, ref.options());
  hipStream_t st = stream_of(ref);
  if (rldx_msat_qkv_norm_rope_bf16(s, n, H, D, q.data_ptr(), nullptr, nullptr, M * D, D, kvp.data_ptr(), elems, 1e-6f,
                                   st) != hipSuccess)
    return Tensor();
  const int64_t ps[2] = {H * elems, elems}, qs[3] = {H * M * D, M * D, D}, os[3] = {M * inner, D, inner};
  const float scale = static_cast<float>(1.0 / std::sqrt(static_cast<double>(D)));
  const hipError_t e =
      mp ? rldx_attention_packed_fwd_mask_bf16(q.data_ptr(), kvp.data_ptr(), ps, out.data_ptr(), 0, 1, H, H, M, M, D, qs,
                                               os, mp, 0, scale, 0, st)
         : rldx_attention_packed_fwd_bf16(q.data_ptr(), kvp.data_ptr(), ps, out.data_ptr(), 0, 1, H, H, M, M, D, qs, os,
                                          nullptr, 0, scale, 0, st);
  return e == hipSuccess ? out : Tensor();
}

RLDX_OP(Ds2, "ds::fused_attention_2way");
Tensor ds2(const Tensor& sa, const Tensor& vl, const Tensor& qsa, const Tensor& ksa, const Tensor& qvl,
           const Tensor& kvl, const Tensor& cos, const Tensor& sin, SymInt nsa_, SymInt nvl_, SymInt h_, SymInt d_) {
  const int64_t nsa = nsa_.guard_int(__FILE__, __LINE__), nvl = nvl_.guard_int(__FILE__, __LINE__),
                H = h_.guard_int(__FILE__, __LINE__), D = d_.guard_int(__FILE__, __LINE__);
  rldx_msat_stream_t s[2];
  if (stream(sa, vl, 0, nvl, H * D, qvl, kvl, nullptr, nullptr, D, s[0]) &&
      stream(sa, sa, 0, nsa, H * D, qsa, ksa, &cos, &sin, D, s[1])) {
    Tensor o = joint(sa, s, 2, std::nullopt, H, D);
    if (o.defined()) return o;
  }
  return python<Ds2, Tensor, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                const Tensor&, const Tensor&, SymInt, SymInt, SymInt, SymInt>(sa, vl, qsa, ksa, qvl, kvl, cos, sin, nsa_,
                                                                              nvl_, h_, d_);
}

RLDX_OP(Ds3, "ds::fused_attention_3way");
Tensor ds3(const Tensor& sa, const Tensor& vl, const Tensor& p, const Tensor& qsa, const Tensor& ksa, const Tensor& qvl,
           const Tensor& kvl, const Tensor& qp, const Tensor& kp, const Tensor& sc, const Tensor& ss, const Tensor& pc,
           const Tensor& psn, SymInt nsa_, SymInt nvl_, SymInt np_, SymInt h_, SymInt d_, const OptTensor& mask) {
  const int64_t nsa = nsa_.guard_int(__FILE__, __LINE__), nvl = nvl_.guard_int(__FILE__, __LINE__),
                np = np_.guard_int(__FILE__, __LINE__), H = h_.guard_int(__FILE__, __LINE__),
                D = d_.guard_int(__FILE__, __LINE__);
  rldx_msat_stream_t s[3];
  if (stream(sa, vl, 0, nvl, H * D, qvl, kvl, nullptr, nullptr, D, s[0]) &&
      stream(sa, sa, 0, nsa, H * D, qsa, ksa, &sc, &ss, D, s[1]) &&
      stream(sa, p, 0, np, H * D, qp, kp, &pc, &psn, D, s[2])) {
    Tensor o = joint(sa, s, 3, mask, H, D);
    if (o.defined()) return o;
  }
  return python<Ds3, Tensor, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                SymInt, SymInt, SymInt, SymInt, SymInt, const OptTensor&>(sa, vl, p, qsa, ksa, qvl, kvl, qp, kp, sc, ss,
                                                                          pc, psn, nsa_, nvl_, np_, h_, d_, mask);
}

RLDX_OP(Ss2, "ss::fused_attention_2way");
Tensor ss2(const Tensor& x, const Tensor& qw, const Tensor& kw, const Tensor& cos, const Tensor& sin, SymInt nsa_,
           SymInt h_, SymInt d_) {
  const int64_t nsa = nsa_.guard_int(__FILE__, __LINE__), H = h_.guard_int(__FILE__, __LINE__),
                D = d_.guard_int(__FILE__, __LINE__);
  if (x.numel() > 0 && qkv_rows(x) && nsa > 0 && rows_of(x) > nsa) {
    const int64_t nv = rows_of(x) - nsa;
    rldx_msat_stream_t s[2];
    if (stream(x, x, 0, nv, H * D, qw, kw, nullptr, nullptr, D, s[0]) &&
        stream(x, x, nv, nsa, H * D, qw, kw, &cos, &sin, D, s[1])) {
      Tensor o = joint(x, s, 2, std::nullopt, H, D);
      if (o.defined()) return o;
    }
  }
  return python<Ss2, Tensor, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, SymInt, SymInt,
                SymInt>(x, qw, kw, cos, sin, nsa_, h_, d_);
}

RLDX_OP(Ss3, "ss::fused_attention_3way");
Tensor ss3(const Tensor& x, const Tensor& p, const Tensor& qx, const Tensor& kx, const Tensor& qp, const Tensor& kp,
           const Tensor& sc, const Tensor& ss, const Tensor& pc, const Tensor& psn, SymInt nx_, SymInt nsa_, SymInt np_,
           SymInt h_, SymInt d_, const OptTensor& mask) {
  const int64_t nx = nx_.guard_int(__FILE__, __LINE__), nsa = nsa_.guard_int(__FILE__, __LINE__),
                np = np_.guard_int(__FILE__, __LINE__), H = h_.guard_int(__FILE__, __LINE__),
                D = d_.guard_int(__FILE__, __LINE__);
  rldx_msat_stream_t s[3];
  if (nsa > 0 && nx > nsa && np > 0 && stream(x, x, 0, nx - nsa, H * D, qx, kx, nullptr, nullptr, D, s[0]) &&
      stream(x, x, nx - nsa, nsa, H * D, qx, kx, &sc, &ss, D, s[1]) &&
      stream(x, p, 0, np, H * D, qp, kp, &pc, &psn, D, s[2])) {
    Tensor o = joint(x, s, 3, mask, H, D);
    if (o.defined()) return o;
  }
  return python<Ss3, Tensor, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                const Tensor&, const Tensor&, const Tensor&, const Tensor&, SymInt, SymInt, SymInt, SymInt, SymInt,
                const OptTensor&>(x, p, qx, kx, qp, kp, sc, ss, pc, psn, nx_, nsa_, np_, h_, d_, mask);
}

// ---------------------------------------------------------------------------
// SwiGLU, fused MLP, residual + norm
// ---------------------------------------------------------------------------
RLDX_OP(Swiglu, "rldx_amd::swiglu");
Tensor swiglu(const Tensor& x) {
  if (bf16(x) && x.dim() >= 1 && x.is_contiguous() && x.numel() > 0 && x.size(-1) % 2 == 0) {
    const c10::OptionalDeviceGuard guard(x.device());
    const int64_t n = x.size(-1) / 2, rows = x.numel() / (2 * n);
    auto shape = x.sizes().vec();
    shape.back() = n;
    Tensor out = at::empty(shape, x.options());
    if (rldx_swiglu_bf16(x.data_ptr(), 2 * n, nullptr, out.data_ptr(), n, rows, n, stream_of(x)) == hipSuccess) return out;
  }
  return python<Swiglu, Tensor, const Tensor&>(x);
}

// Packed weights of ss::fused_mlp_swiglu.  Python packs a weight, keeps the packed
// copy for as long as the weight lives and enters it here; forget() takes it out
// when the weight dies.  The weak reference keeps the address from being another
// tensor's meanwhile, and the version, the data pointer, the sizes and the strides
// must be the packed ones (`w.data = w.data[:rows]` changes the sizes alone).
// Made: the launch that wrote the copy.  Work on another stream waits for its event; a
// stream capture takes the copy only when it is complete, because a replay waits for
// nothing outside its graph.
struct Made {
  c10::Event event{c10::DeviceType::CUDA};
  c10::Stream stream;
  std::atomic<bool> done{false};
  explicit Made(c10::Stream s) : stream(s) { event.record(s); }
  void again(c10::Stream s) {
    stream = s;
    done = false;
    event.record(s);
  }
};
struct Packed {
  c10::weak_intrusive_ptr<c10::TensorImpl> w;
  uint32_t version;
  const void* data;
  std::vector<int64_t> sizes, strides;
  Tensor packed;
  std::shared_ptr<Made> made;  // null: host memory
};
std::mutex g_packed_mutex;
std::unordered_map<int64_t, Packed>& packed_weights() {
  static auto* m = new std::unordered_map<int64_t, Packed>();  // (never destroyed: entries may outlive the runtime's exit)
  return *m;
}
c10::Stream current_stream(const Tensor& t) {
  return c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getStream(t.device());
}
// Events of forgotten copies, at most 16: a new one costs 15-20 us of a first call.  (Under the mutex.)
std::vector<std::shared_ptr<Made>>& spare_events() {
  static auto* v = new std::vector<std::shared_ptr<Made>>();
  return *v;
}
std::shared_ptr<Made> made_on(c10::Stream s) {
  std::shared_ptr<Made> m;
  {
    const std::lock_guard<std::mutex> lock(g_packed_mutex);
    auto& v = spare_events();
    for (size_t i = 0; i < v.size() && !m; ++i)
      if (v[i]->stream.device_index() == s.device_index()) {
        m = std::move(v[i]);
        v.erase(v.begin() + static_cast<std::ptrdiff_t>(i));
      }
  }
  if (!m) return std::make_shared<Made>(s);
  m->again(s);
  return m;
}
void spare(std::shared_ptr<Made>& m) {  // (nobody else reads it: it came out of the table, and no call holds it)
  if (m && m.use_count() == 1 && spare_events().size() < 16) spare_events().push_back(std::move(m));
}
int64_t key_of(const Tensor& w) { return reinterpret_cast<int64_t>(w.unsafeGetTensorImpl()); }

void remember_packed(const Tensor& w, const Tensor& packed) {
  if (w.is_inference()) return;  // no version counter
  Packed p{c10::weak_intrusive_ptr<c10::TensorImpl>(w.getIntrusivePtr()), static_cast<uint32_t>(w._version()),
           w.data_ptr(), w.sizes().vec(), w.strides().vec(), packed,
           packed.is_cuda() ? made_on(current_stream(packed)) : nullptr};
  std::optional<Packed> old;  // freed outside the lock: the last reference to a tensor of Python's takes the GIL
  const std::lock_guard<std::mutex> lock(g_packed_mutex);
  auto [it, inserted] = packed_weights().try_emplace(key_of(w), std::move(p));
  if (inserted) return;
  old.emplace(std::move(it->second));
  spare(old->made);
  it->second = std::move(p);
}
void forget_packed(int64_t key) {
  std::optional<Packed> old;  // freed outside the lock, as above
  const std::lock_guard<std::mutex> lock(g_packed_mutex);
  auto it = packed_weights().find(key);
  if (it == packed_weights().end()) return;
  old.emplace(std::move(it->second));
  spare(old->made);
  packed_weights().erase(it);
}
// Whether work on the current stream can read a copy; makes the stream wait for it where it has to.
bool readable(const Tensor& packed, Made& m) {
  const c10::Stream cur = current_stream(packed);
  if (!m.done) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream_of(packed), &capture) != hipSuccess) return false;
    {
      // (a query ends no capture, neither this stream's nor another thread's)
      c10::hip::HIPStreamCaptureModeGuard relaxed(hipStreamCaptureModeRelaxed);
      m.done = m.event.query();
    }
    if (!m.done && capture != hipStreamCaptureStatusNone) return false;
    if (!m.done && cur != m.stream) m.event.block(cur);
  }
  if (cur != m.stream) packed.record_stream(cur);
  return true;
}
OptTensor packed_of(const Tensor& w) {
  if (w.is_inference()) return std::nullopt;
  Tensor packed;
  std::shared_ptr<Made> made;
  {
    const std::lock_guard<std::mutex> lock(g_packed_mutex);
    auto it = packed_weights().find(key_of(w));
    if (it == packed_weights().end()) return std::nullopt;
    const Packed& p = it->second;
    if (p.w.expired() || p.data != w.data_ptr() || p.version != static_cast<uint32_t>(w._version()) ||
        w.sizes() != p.sizes || w.strides() != p.strides)
      return std::nullopt;
    packed = p.packed;
    made = p.made;
  }
  if (made && !readable(packed, *made)) return std::nullopt;
  return packed;
}

RLDX_OP(Mlp, "ss::fused_mlp_swiglu");
Tensor mlp(const Tensor& x, const Tensor& w, const Tensor& bias, SymInt split_) {
  const int64_t split = split_.guard_int(__FILE__, __LINE__);
  if (split <= 1 && rows2d(x) && x.size(0) > 0 && bf16(w) && w.dim() == 2 && w.size(0) % 2 == 0 &&
      one_device(x, w, bias) && vec(bias, w.size(0)) && w.size(1) == x.size(1)) {
    const OptTensor pw = packed_of(w);
    if (pw.has_value()) {
      const c10::OptionalDeviceGuard guard(x.device());
      const int64_t M = x.size(0), K = x.size(1), n = w.size(0);
      Tensor a = at::empty({(M + 31) / 32 * 32 * K}, x.options()), out = at::empty({M, n / 2}, x.options());
      hipStream_t st = stream_of(x);
      const rldx_gemm_group_t g{a.data_ptr(), M, pw->data_ptr(), bias.data_ptr(), out.data_ptr(), n / 2, nullptr, 0};
      if (rldx_act_pack_bf16(x.data_ptr(), x.stride(0), M, K, a.data_ptr(), st) == hipSuccess &&
          rldx_grouped_gemm_bf16(&g, 1, n, K, RLDX_GEMM_EPI_SWIGLU, st) == hipSuccess)
        return out;
    }
  }
  return python<Mlp, Tensor, const Tensor&, const Tensor&, const Tensor&, SymInt>(x, w, bias, split_);
}

using Two = std::tuple<Tensor, Tensor>;
// new = hidden + residual [+ deepstack]; normed = RMSNorm(new): outputs shaped like hidden, or undefined
Two add_rmsnorm(const Tensor& h, const Tensor& r, const Tensor* ds, const Tensor& w) {
  if (bf16(h) && bf16(r) && (!ds || bf16(*ds)) && h.dim() >= 1 && h.numel() > 0 && one_device(h, r, w) &&
      (!ds || ds->device() == h.device()) && h.is_contiguous() && r.is_contiguous() && (!ds || ds->is_contiguous()) &&
      r.numel() == h.numel() && (!ds || ds->numel() == h.numel()) && w.dim() == 1 && vec(w, h.size(-1))) {
    const c10::OptionalDeviceGuard guard(h.device());
    const int64_t D = h.size(-1), M = h.numel() / D;
    Tensor nh = at::empty(h.sizes(), h.options()), nm = at::empty(h.sizes(), h.options());
    if (rldx_add_rmsnorm_bf16(h.data_ptr(), r.data_ptr(), ds ? ds->data_ptr() : nullptr, w.data_ptr(), nh.data_ptr(),
                              nm.data_ptr(), M, D, 1e-6f, stream_of(h)) == hipSuccess)
      return {nh, nm};
  }
  return {};
}
template <class Tag>
Two add2(const Tensor& h, const Tensor& r, const Tensor& w) {
  Two o = add_rmsnorm(h, r, nullptr, w);
  return std::get<0>(o).defined() ? o : python<Tag, Two, const Tensor&, const Tensor&, const Tensor&>(h, r, w);
}
RLDX_OP(Add2, "rldx_backbone::fused_epilogue_add2_rmsnorm");
RLDX_OP(MemAdd2, "mem::fused_epilogue_add2_rmsnorm");
RLDX_OP(Add3, "rldx_backbone::fused_epilogue_add3_rmsnorm");
Two add3(const Tensor& h, const Tensor& r, const Tensor& ds, const Tensor& w) {
  Two o = add_rmsnorm(h, r, &ds, w);
  return std::get<0>(o).defined()
             ? o
             : python<Add3, Two, const Tensor&, const Tensor&, const Tensor&, const Tensor&>(h, r, ds, w);
}

// the autograd kernel of an operator with native kernel F
template <class Tag, class R, class... A>
constexpr auto autograd_of(R (*)(A...)) { return &Autograd<Tag, R(A...)>::call; }

#define RLDX_IMPL(M, NAME, TAG, FN) M.impl(NAME, TORCH_FN((FN)))
#define RLDX_AUTOGRAD(M, NAME, TAG, FN) M.impl(NAME, autograd_of<TAG>(FN))

}  // namespace

#define RLDX_BACKBONE(X, M)                                       \
  X(M, "fused_attention", Gqa, gqa);                              \
  X(M, "vision_attention", Vit, vit);                             \
  X(M, "fused_epilogue_add2_rmsnorm", Add2, add2<Add2>);          \
  X(M, "fused_epilogue_add3_rmsnorm", Add3, add3)
#define RLDX_MEM(X, M)               \
  X(M, "fused_attention", Mem, mem); \
  X(M, "fused_epilogue_add2_rmsnorm", MemAdd2, add2<MemAdd2>)
#define RLDX_DS(X, M)                     \
  X(M, "fused_attention_2way", Ds2, ds2); \
  X(M, "fused_attention_3way", Ds3, ds3)
#define RLDX_SS(X, M)                     \
  X(M, "fused_attention_2way", Ss2, ss2); \
  X(M, "fused_attention_3way", Ss3, ss3); \
  X(M, "fused_mlp_swiglu", Mlp, mlp)

TORCH_LIBRARY_IMPL(rldx_backbone, CUDA, m) { RLDX_BACKBONE(RLDX_IMPL, m); }
TORCH_LIBRARY_IMPL(rldx_backbone, AutogradCUDA, m) { RLDX_BACKBONE(RLDX_AUTOGRAD, m); }
TORCH_LIBRARY_IMPL(mem, CUDA, m) { RLDX_MEM(RLDX_IMPL, m); }
TORCH_LIBRARY_IMPL(mem, AutogradCUDA, m) { RLDX_MEM(RLDX_AUTOGRAD, m); }
TORCH_LIBRARY_IMPL(ds, CUDA, m) { RLDX_DS(RLDX_IMPL, m); }
TORCH_LIBRARY_IMPL(ds, AutogradCUDA, m) { RLDX_DS(RLDX_AUTOGRAD, m); }
TORCH_LIBRARY_IMPL(ss, CUDA, m) { RLDX_SS(RLDX_IMPL, m); }
TORCH_LIBRARY_IMPL(ss, AutogradCUDA, m) { RLDX_SS(RLDX_AUTOGRAD, m); }
TORCH_LIBRARY_IMPL(rldx_amd, CUDA, m) { RLDX_IMPL(m, "swiglu", Swiglu, swiglu); }
TORCH_LIBRARY_IMPL(rldx_amd, AutogradCUDA, m) { RLDX_AUTOGRAD(m, "swiglu", Swiglu, swiglu); }

TORCH_LIBRARY(rldx_native, m) {
  m.def("remember_packed(Tensor w, Tensor packed) -> ()", &remember_packed);
  m.def("forget_packed(int key) -> ()", &forget_packed);
  m.def("packed_of(Tensor w) -> Tensor?", &packed_of);
}
