// pybind11 torch extension `dhellam_amd._host`: the host path of the Python operators (dhellam_amd/operators,
// dhellam_amd/_Clib.py) in native code.  One call per operator: it checks the tensors, makes the results and the
// scratch on the stream the operator runs on, and calls the C ABI (include/dhellam_hip.h).
//
// What bounds a small operator is the host: with its checks, allocations, stream switches and ctypes call in Python an
// operator took 20-25 us to issue (seven bandwidth operators on 64 tokens: 178 us of host time for 28 us of kernels).
// torch.cuda.current_stream() alone is 7 us, entering and leaving torch.cuda.stream() another 5.  From here the same seven
// take 56 us to issue (8 us each, most of it the kernel launch), and the pass went from 151 to 41 us.
//
// Conventions: `stream` is None (torch's current stream) or a torch.cuda.Stream, under which results and scratch are
// allocated; a failed argument check raises AssertionError where the Python operator asserted and RuntimeError
// otherwise; the GIL is released around the library call, as ctypes does.
#include <torch/extension.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Stream.h>

#include <array>
#include <map>
#include <algorithm>
#include <mutex>
#include <optional>
#include <tuple>
#include <vector>

#include "dhellam_hip.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;
using OptStream = py::object;      // None, a torch.cuda.Stream, or a raw handle

[[noreturn]] void assertion(const char *msg) {
  PyErr_SetString(PyExc_AssertionError, msg);
  throw py::error_already_set();
}
#define PY_ASSERT(cond, msg) \
  do {                       \
    if (!(cond)) assertion(msg); \
  } while (0)

int dt(const Tensor &t) {
  switch (t.scalar_type()) {
    case at::kFloat: return DH_F32;
    case at::kBFloat16: return DH_BF16;
    case at::kHalf: return DH_F16;
    default: TORCH_CHECK(false, "unsupported dtype ", t.scalar_type());
  }
}

void need_gpu(std::initializer_list<const Tensor *> ts) {
  for (const Tensor *t : ts) TORCH_CHECK(t->is_cuda(), "dhellam operators need tensors on the GPU");
}

// Runs fn() -> status without the GIL and raises its error.  `own`: the lock of a shared scratch buffer, held meanwhile:
// the kernels of one call that hand each other data through it must not have those of another thread's call on the same
// stream between them.  It is taken and given back without the GIL, so that no thread waits for one holding the other.
template <typename F> void launch(F &&fn, std::mutex *own = nullptr) {
  int rc;
  {
    py::gil_scoped_release nogil;
    std::unique_lock<std::mutex> lock;
    if (own) lock = std::unique_lock<std::mutex>(*own);
    rc = fn();
  }
  TORCH_CHECK(rc == 0, "dhellam_hip error ", rc, ": ", dh_last_error());
}

// The stream an operator runs on: torch's current one, or the given one made current while this object lives (as
// `with torch.cuda.stream(s)` does), so that allocations belong to it.
class On {
 public:
  explicit On(const OptStream &s) {
    if (THPStream_Check(s.ptr())) {
      const c10::hip::HIPStream want = of(s);
      if (want != c10::hip::getCurrentHIPStream()) guard_.emplace(want.unwrap());
      raw_ = want.stream();
    } else if (s.is_none()) {
      raw_ = c10::hip::getCurrentHIPStream().stream();
    } else {      // a handle: launched there, allocations stay with the current stream
      raw_ = (hipStream_t)s.cast<uint64_t>();
    }
  }
  // The runtime masquerades as CUDA in Python and is HIP in c10: same stream, other device type.
  static c10::hip::HIPStream of(const OptStream &s) {
    auto *t = (THPStream *)s.ptr();
    return c10::hip::HIPStream(c10::Stream::unpack3(t->stream_id, (c10::DeviceIndex)t->device_index, c10::DeviceType::HIP));
  }
  void *get() const { return raw_; }

 private:
  std::optional<c10::hip::HIPStreamGuard> guard_;
  hipStream_t raw_;
};

const void *ptr(const OptTensor &t) { return t.has_value() ? t->data_ptr() : nullptr; }
void *mptr(const OptTensor &t) { return t.has_value() ? t->data_ptr() : nullptr; }

// Scratch kept per (device, stream) and purpose: kernels on one stream are ordered, so consecutive calls may share it
// (calls of several threads one after the other: `own`); it grows to the largest call seen, the replaced buffer staying with
// the calls that hold it.  Never freed at exit: the allocator may be gone by then.
enum Scratch { kNorm, kGemm, kAttnBwd, kGrouped, kScratchKinds };
struct Key {
  int device;
  void *stream;
  bool operator<(const Key &o) const { return device != o.device ? device < o.device : stream < o.stream; }
};
std::mutex g_scratch_mu;
struct Buffer {
  Tensor t;
  std::mutex own;
};
std::map<Key, Buffer> &scratch_map(int kind) {
  static auto *maps = new std::array<std::map<Key, Buffer>, kScratchKinds>();
  return (*maps)[kind];
}
struct Held {
  Tensor t;
  std::mutex *own;
  void *data_ptr() const { return t.data_ptr(); }
  int64_t numel() const { return t.numel(); }
};
Held scratch(Scratch kind, int64_t bytes, const Tensor &like, void *stream) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  Buffer &b = scratch_map(kind)[Key{like.device().index(), stream}];
  if (!b.t.defined() || b.t.numel() < bytes) b.t = at::empty({bytes}, like.options().dtype(at::kByte));
  return {b.t, &b.own};
}
// (device index, stream handle) of the scratch buffers of one kind that exist.
std::vector<std::pair<int, uint64_t>> scratch_keys(int kind) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  std::vector<std::pair<int, uint64_t>> r;
  for (auto &kv : scratch_map(kind)) r.emplace_back(kv.first.device, (uint64_t)kv.first.stream);
  return r;
}

uint64_t stream_ptr(const OptStream &s) {
  if (THPStream_Check(s.ptr())) return (uint64_t)On::of(s).stream();
  return (uint64_t)c10::hip::getCurrentHIPStream().stream();
}

// ---- norm ---------------------------------------------------------------------------------------------------------
// -> (ln_out like inp, mu or None, rsigma, sum or None)
std::tuple<Tensor, OptTensor, Tensor, OptTensor> norm_fwd(const Tensor &inp, const Tensor &weight, const OptTensor &bias,
                                                          double eps, bool zero_centered, const OptTensor &residual,
                                                          OptTensor sum_out, const OptTensor &ln_out,
                                                          const OptStream &stream) {
  PY_ASSERT(inp.is_cuda(), "dhellam needs a GPU.");
  const int64_t cols = weight.numel();
  PY_ASSERT(inp.dim() > 0 && inp.size(-1) == cols, "LayerNorm not possible");
  PY_ASSERT(inp.is_contiguous() && weight.is_contiguous(), "norm: input and weight must be contiguous");
  const int64_t rows = cols ? inp.numel() / cols : 0;
  const int type = dt(inp);
  On on(stream);
  Tensor y;
  if (ln_out.has_value()) {
    PY_ASSERT(ln_out->is_contiguous() && ln_out->numel() == inp.numel() && ln_out->scalar_type() == inp.scalar_type(),
              "norm: ln_out must be contiguous, of the input's size and type");
    y = ln_out->view(inp.sizes());
  } else {
    y = at::empty(inp.sizes(), inp.options());
  }
  const auto f32 = inp.options().dtype(at::kFloat);
  Tensor rsigma = at::empty({rows}, f32);
  OptTensor mu;
  if (bias.has_value()) mu = at::empty({rows}, f32);
  if (!residual.has_value()) {
    launch([&] {
      return dh_norm_fwd(inp.data_ptr(), weight.data_ptr(), ptr(bias), y.data_ptr(), (float *)mptr(mu),
                         rsigma.data_ptr<float>(), rows, cols, (float)eps, zero_centered, type, on.get());
    });
    return {y, mu, rsigma, std::nullopt};
  }
  PY_ASSERT(residual->is_contiguous() && residual->numel() == inp.numel() && residual->scalar_type() == inp.scalar_type(),
            "norm: residual must be contiguous, of the input's size and type");
  if (!sum_out.has_value()) sum_out = at::empty(residual->sizes(), residual->options());
  PY_ASSERT(sum_out->is_contiguous() && sum_out->numel() == inp.numel() && sum_out->scalar_type() == inp.scalar_type(),
            "norm: sum_out must be contiguous, of the input's size and type");
  launch([&] {
    return dh_add_norm_fwd(inp.data_ptr(), residual->data_ptr(), sum_out->data_ptr(), weight.data_ptr(), ptr(bias),
                           y.data_ptr(), (float *)mptr(mu), rsigma.data_ptr<float>(), rows, cols, (float)eps,
                           zero_centered, type, on.get());
  });
  return {y, mu, rsigma, sum_out};
}

// -> (dinp like inp, dgamma, dbeta or None)
std::tuple<Tensor, Tensor, OptTensor> norm_bwd(const Tensor &dy, const Tensor &inp, const OptTensor &mu,
                                               const Tensor &rsigma, const Tensor &weight, bool zero_centered,
                                               const OptTensor &add, const OptTensor &dgamma_out,
                                               const OptTensor &dbeta_out, const OptTensor &dgrad_out,
                                               const OptStream &stream) {
  PY_ASSERT(inp.is_cuda(), "dhellam needs a GPU.");
  const int64_t cols = weight.numel();
  PY_ASSERT(inp.dim() > 0 && inp.size(-1) == cols, "LayerNorm not possible");
  PY_ASSERT(inp.is_contiguous() && dy.is_contiguous() && dy.numel() == inp.numel(),
            "norm: input and gradient must be contiguous and of one size");
  const int64_t rows = cols ? inp.numel() / cols : 0;
  const int type = dt(inp);
  PY_ASSERT(!add.has_value() || (add->is_contiguous() && add->numel() == inp.numel()),
            "norm: add_to_dgrad must be contiguous, of the input's size");
  On on(stream);
  Tensor dx;
  if (dgrad_out.has_value()) {
    PY_ASSERT(dgrad_out->is_contiguous() && dgrad_out->numel() == inp.numel() &&
                  dgrad_out->scalar_type() == inp.scalar_type(),
              "norm: dgrad_out must be contiguous, of the input's size and type");
    dx = dgrad_out->view(inp.sizes());
  } else {
    dx = at::empty(inp.sizes(), inp.options());
  }
  const bool accumulate = dgamma_out.has_value();
  PY_ASSERT(!accumulate || dgamma_out->scalar_type() == weight.scalar_type(), "dgamma_out must have the weight's dtype");
  PY_ASSERT(!dbeta_out.has_value() || dbeta_out->scalar_type() == weight.scalar_type(),
            "dbeta_out must have the weight's dtype");
  Tensor dgamma = accumulate ? *dgamma_out : at::empty_like(weight);
  OptTensor dbeta;
  if (mu.has_value()) {
    PY_ASSERT(dbeta_out.has_value() == accumulate, "pass both or neither of dgamma_out/dbeta_out");
    dbeta = dbeta_out.has_value() ? *dbeta_out : at::empty_like(weight);
  }
  const Held ws = scratch(kNorm, (int64_t)dh_norm_bwd_workspace_bytes(rows, cols), inp, on.get());
  launch([&] {
    return dh_norm_bwd(dy.data_ptr(), inp.data_ptr(), (const float *)ptr(mu), rsigma.data_ptr<float>(),
                       weight.data_ptr(), ptr(add), dx.data_ptr(), dgamma.data_ptr(), mptr(dbeta), ws.data_ptr(),
                       (size_t)ws.numel(), rows, cols, zero_centered, accumulate, type, on.get());
  }, ws.own);
  return {dx, dgamma, dbeta};
}

// ---- SwiGLU, residual add, RoPE -------------------------------------------------------------------------------------
bool transposable(int64_t rows, int64_t f, std::initializer_list<const Tensor *> ts) {
  if (!(rows > 0 && f > 0 && rows % 8 == 0 && f % 8 == 0 && rows < 64 * 65535)) return false;
  const auto type = (*ts.begin())->scalar_type();
  if (type != at::kBFloat16 && type != at::kHalf) return false;
  for (const Tensor *t : ts)
    if (t->scalar_type() != type || (uintptr_t)t->data_ptr() % 16 != 0) return false;
  return true;
}

// -> (out, its transpose or None)
std::tuple<Tensor, OptTensor> swiglu_fwd(const Tensor &y, bool with_transposed, const OptStream &stream) {
  PY_ASSERT(y.is_cuda() && y.is_contiguous() && y.dim() > 0 && y.size(-1) % 2 == 0,
            "swiglu: input must be a contiguous GPU tensor with an even last dimension");
  const int64_t f = y.size(-1) / 2, rows = f ? y.numel() / (2 * f) : 0;
  const int type = dt(y);
  On on(stream);
  auto sizes = y.sizes().vec();
  sizes.back() = f;
  Tensor out = at::empty(sizes, y.options());
  OptTensor ot;
  if (with_transposed && transposable(rows, f, {&y, &out})) {
    ot = at::empty({f, rows}, y.options());
    launch([&] { return dh_swiglu_fwd_t(y.data_ptr(), out.data_ptr(), ot->data_ptr(), rows, f, type, on.get()); });
  } else {
    launch([&] { return dh_swiglu_fwd(y.data_ptr(), out.data_ptr(), rows, f, type, on.get()); });
  }
  return {out, ot};
}

// -> (dy, its transpose or None)
std::tuple<Tensor, OptTensor> swiglu_bwd(const Tensor &g, const Tensor &y, const OptTensor &o, bool with_transposed,
                                         const OptStream &stream) {
  PY_ASSERT(y.is_cuda() && y.is_contiguous() && g.is_contiguous() && y.dim() > 0 && y.size(-1) % 2 == 0,
            "swiglu: inputs must be contiguous GPU tensors with an even last dimension");
  const int64_t f = y.size(-1) / 2, rows = f ? y.numel() / (2 * f) : 0;
  PY_ASSERT(g.numel() == rows * f, "grad shape does not match swiglu input");
  const int type = dt(y);
  On on(stream);
  Tensor out = o.has_value() ? *o : at::empty(y.sizes(), y.options());
  PY_ASSERT(out.is_contiguous() && out.sizes() == y.sizes(), "swiglu: o must be contiguous, of the input's shape");
  OptTensor ot;
  if (with_transposed && transposable(rows, f, {&y, &g, &out})) {
    ot = at::empty({2 * f, rows}, y.options());
    launch([&] {
      return dh_swiglu_bwd_t(g.data_ptr(), y.data_ptr(), out.data_ptr(), ot->data_ptr(), rows, f, type, on.get());
    });
  } else {
    launch([&] { return dh_swiglu_bwd(g.data_ptr(), y.data_ptr(), out.data_ptr(), rows, f, type, on.get()); });
  }
  return {out, ot};
}

Tensor residual_add(const Tensor &x, const Tensor &residual, const OptTensor &out, const OptStream &stream) {
  PY_ASSERT(x.is_cuda() && x.is_contiguous() && residual.is_contiguous(), "bda: tensors must be contiguous on the GPU");
  PY_ASSERT(x.numel() == residual.numel() && x.scalar_type() == residual.scalar_type(), "bda: sizes or types differ");
  const Tensor &dst = out.has_value() ? *out : x;
  PY_ASSERT(dst.is_contiguous() && dst.numel() == x.numel() && dst.scalar_type() == x.scalar_type(),
            "bda: out must be contiguous, of the input's size and type");
  const int type = dt(x);
  On on(stream);
  launch([&] { return dh_residual_add(x.data_ptr(), residual.data_ptr(), dst.data_ptr(), x.numel(), type, on.get()); });
  return dst;
}

int64_t head_rows_stride(const Tensor &t) {
  PY_ASSERT(t.dim() == 3 && t.stride(2) == 1 && t.stride(1) == t.size(2), "expected [tokens, heads, d] with contiguous heads");
  return t.stride(0);
}

std::tuple<Tensor, OptTensor> rope(const Tensor &q, const OptTensor &k, const Tensor &inv_freq, const OptTensor &positions,
                                   int64_t seq_len, bool backward, bool inplace, const OptStream &stream) {
  PY_ASSERT(q.is_cuda(), "rope: tensors must be on the GPU");
  const int64_t qs = head_rows_stride(q), d = q.size(2);
  PY_ASSERT(!positions.has_value() || (positions->scalar_type() == at::kInt && positions->numel() == q.size(0)),
            "rope: positions must be int32, one per token");
  int64_t ks = 0;
  if (k.has_value()) {
    ks = head_rows_stride(*k);
    PY_ASSERT(k->size(0) == q.size(0) && k->size(2) == d && k->scalar_type() == q.scalar_type(), "rope: q and k differ");
  }
  const int type = dt(q);
  On on(stream);
  Tensor qo = inplace ? q : at::empty(q.sizes(), q.options());
  OptTensor ko;
  if (k.has_value()) ko = inplace ? *k : at::empty(k->sizes(), k->options());
  launch([&] {
    return dh_rope(q.data_ptr(), ptr(k), qo.data_ptr(), mptr(ko), inv_freq.data_ptr<float>(),
                   (const int32_t *)ptr(positions), q.size(0), (int)q.size(1), k.has_value() ? (int)k->size(1) : 0, (int)d,
                   qs, ks, head_rows_stride(qo), ko.has_value() ? head_rows_stride(*ko) : 0, seq_len, backward, type, on.get());
  });
  return {qo, ko};
}

// ---- dense GEMM, transpose ------------------------------------------------------------------------------------------
constexpr int64_t kGemmWorkspace = 32 << 20;

bool dense_ok(std::initializer_list<const Tensor *> ts) {
  for (const Tensor *t : ts)
    if (!(t->is_cuda() && t->dim() == 2 && t->is_contiguous())) return false;
  return true;
}

void gemm_on(const Tensor &A, const Tensor &B, const Tensor &D, bool transa, bool transb, bool accumulate,
             const OptTensor &workspace, int64_t workspace_bytes, void *st) {
  TORCH_CHECK(dense_ok({&A, &B, &D}), "dense_gemm: operands must be contiguous 2-D GPU tensors");
  TORCH_CHECK(A.scalar_type() == B.scalar_type() && (D.scalar_type() == A.scalar_type() || D.scalar_type() == at::kFloat),
              "dense_gemm: operand types ", A.scalar_type(), ", ", B.scalar_type(), " -> ", D.scalar_type(), " not supported");
  const int64_t m = transa ? A.size(0) : A.size(1), n = transb ? B.size(1) : B.size(0);
  TORCH_CHECK(D.size(0) == n && D.size(1) == m, "dense_gemm: output is ", D.sizes(), ", the product is [", n, ", ", m, "]");
  Held ws{{}, nullptr};
  if (!workspace.has_value() || !workspace->is_cuda() || workspace_bytes <= 0) {
    ws = scratch(kGemm, kGemmWorkspace, A, st);
    workspace_bytes = ws.numel();
  } else {
    TORCH_CHECK((int64_t)workspace->nbytes() >= workspace_bytes, "dense_gemm: workspace tensor smaller than workspaceSize");
    ws.t = *workspace;
  }
  if ((transa ? A.size(1) : A.size(0)) == 0) {
    if (!accumulate) D.zero_();
    return;
  }
  const int type = dt(A), out_type = dt(D);
  launch([&] {
    if (transa && transb)      // refused by dh_gemm as by the reference's cublas_gemm; the library's own entry for it
      return dh_gemm_tt(A.data_ptr(), B.data_ptr(), D.data_ptr(), A.size(0), A.size(1), B.size(0), B.size(1), accumulate,
                        type, out_type, ws.data_ptr(), (size_t)workspace_bytes, st);
    return dh_gemm(A.data_ptr(), B.data_ptr(), D.data_ptr(), A.size(0), A.size(1), B.size(0), B.size(1), transa, transb,
                   accumulate, type, out_type, ws.data_ptr(), (size_t)workspace_bytes, st);
  }, ws.own);
}

void dense_gemm(const Tensor &A, const Tensor &B, const Tensor &D, bool transa, bool transb, bool accumulate,
                const OptTensor &workspace, int64_t workspace_bytes, const OptStream &stream) {
  On on(stream);
  gemm_on(A, B, D, transa, transb, accumulate, workspace, workspace_bytes, on.get());
}

// input [..., K] @ weight [N, K]^T in `output` (made here if not given); None where dh_gemm does not take the operands.
OptTensor linear(const Tensor &input, const Tensor &weight, OptTensor output, const OptStream &stream) {
  if (!input.is_contiguous() || !input.is_cuda() || input.dim() < 1 || !dense_ok({&weight}) ||
      weight.scalar_type() != input.scalar_type() || input.size(-1) != weight.size(1) ||
      (output.has_value() && !(output->is_contiguous() && output->scalar_type() == input.scalar_type())))
    return std::nullopt;
  const int64_t n = weight.size(0), k = weight.size(1), rows = k ? input.numel() / k : 0;
  if (k == 0) return std::nullopt;
  On on(stream);
  if (!output.has_value()) {
    auto sizes = input.sizes().vec();
    sizes.back() = n;
    output = at::empty(sizes, input.options());
  }
  gemm_on(weight, input.view({rows, k}), output->view({-1, n}), true, false, false, std::nullopt, 0, on.get());
  return output;
}

// B [T, k] @ A^T (transa, A [m, k]) or B @ A (A [k, m]) in `out`, made here if not given
Tensor matmul(const Tensor &A, const Tensor &B, const OptTensor &out, bool transa, const OptStream &stream) {
  TORCH_CHECK(A.dim() == 2 && B.dim() == 2, "dense_gemm: operands must be contiguous 2-D GPU tensors");
  On on(stream);
  Tensor d = out.has_value() ? *out : at::empty({B.size(0), transa ? A.size(0) : A.size(1)}, B.options());
  gemm_on(A, B, d, transa, false, false, std::nullopt, 0, on.get());
  return d;
}

// 16-bit matrices that the grouped kernel takes with one group: rows of whole 16-byte pieces, aligned.
bool grouped_ok(const Tensor &x, at::ScalarType type) {
  return x.is_cuda() && x.dim() == 2 && x.is_contiguous() && x.scalar_type() == type && (type == at::kBFloat16 || type == at::kHalf) &&
         x.size(1) % 8 == 0 && (uintptr_t)x.data_ptr() % 16 == 0;
}

// The row lengths (elements) that the grouped kernel's tiles address: longer ones have a kernel there for a few rows only.
constexpr int64_t kGroupedMaxRow = (1 << 22) - 8;

// Data gradient grad [T, N] @ weight [N, K] as given: whether the grouped kernel with one group is the faster one.  It splits
// long reductions of few rows over the chip and needs no whole slices; the library's kernels for this layout are at their
// best where N is short and the result small.  us, library / here, of sweeps over N = 1000 to 50304, K = 64 to 8192, T = 1 to 16384:
//   N >= 16000: 32000 x 1024 at 8, 200, 1000, 4096, 16384 94 / 21, 101 / 33, 174 / 68, 336 / 214, 800 / 738; x 4096 at 8, 1000, 4096, 16384 122 / 50,
//     323 / 211, 769 / 719, 3058 / 2923
//   more than 125 rows for every column of a narrow result, store after store: 8192 x 64 at 6000, 16384 1.18 and 0.52 times as fast, x 128
//     at 12000, 16384 1.09 and 0.60; from N = 12000 on only up to 64 columns (32000 x 64 at 16384 0.94, x 128 1.21 times)
//   results of up to 65536 values, where there is little to split (not the narrowest, where the library is slow as well, and not
//     those with rows of 4096 and more): 5120 x 256 at 48, 256 10.6 / 12, 10.8 / 13.9, 8192 x 1024 at 16, 48, 65 0.82, 0.84, 1.35 times; from 9000
//     on here again (12288 x 256 at 1, 200 1.04, 1.36 times).  At exactly 64 rows the library's choice is a poor one: 8192 x 1024
//     36 / 17, 5120 x 256 25 / 13, where 63 and 65 rows are 0.8 times as fast here
//   5120 <= N < 16000, by K T: 8192 x 1024 at 100, 1000, 1904 1.5 times, 44 / 31, 58 / 43, at 3000 65 / 64; x 2048 at 1000 58 / 45,
//     at 1904 71 / 73, at 3000 94 / 112; x 3584 at 768 84 / 57, at 1000 70 / 70; 7168 x 8192 at 200 50 / 41, at 512 64 / 68;
//     and again where 256x256 tiles fill the chip: 7168 x 8192 at 1904, 4096 173 / 164, 346 / 330, 8192 x 3584 at 4096 184 / 180
//   N that is no multiple of 64: to 1152 all (1000 x 1024 at 8, 1904, 16384 10.6 / 8.1, 15 / 11, 43 / 36); from 2900 on by the size of the
//     result as above, up to 5900 (4008 x 256 at 128, 512, 1000 0.86, 1.41 times, 20 / 16, 6008 x 128 at 256 0.96); in between large results,
//     and from 1440 on few rows and narrow long results (1256 x 1024 at 8, 1000, 8192 0.93, 0.87, 1.18 times; 1504 x 512 at 32, 1000,
//     8192 1.08, 0.94, 0.79, x 128 at 512, 1000 0.97, 1.40; 2008 x 1024 at 64, 1000, 4096, 8192 1.42, 0.84, 0.83, 1.09)
//   below: the library (3072 x 1024 at 1000 18 / 21, 1280 x 8192 at 1904 38 / 41)
// Over the 2254 products of the sweeps 23 are more than 5 % slower here than by the library, none of them by 20 %.
bool dgrad_grouped(int64_t t, int64_t n, int64_t k) {
  if (t <= 0 || n < 1000 || n > kGroupedMaxRow || k > kGroupedMaxRow) return false;
  const int64_t size = t * k;
  const bool ragged = n % 64 != 0;
  if (ragged && n < 1152) return true;
  if (t > 125 * k && (n < 12000 || k <= 64)) return false;
  if (n >= 16000) return true;
  if (ragged && n < 2900)
    return size > (n < 1440 ? 2000000 : 4300000) || (n >= 1440 && (t <= 56 || t == 64 || (t >= 1000 && k > 64 && k < 256)));
  if (!ragged && n < 5120) return false;
  if (size <= 65536 && k > 64 && k < 4096 && t != 64 && n < (ragged ? 5900 : 9000)) return false;
  return ragged || size <= 2800000 || size >= 14000000;
}

// Weight gradient dY [T, N]^T X [T, K]: the same question.  The library reads both operands along their strided dimension
// here, its slowest layout (one of them materialised transposed first gains 10 % and costs most of that); the grouped kernel's
// LDS transpose reads cost it nothing, and it adds to what is there without a read of its own.  us accumulating, library (the
// better of its two layouts) / here, N, K at T = 200, 1000, 1904, 4096: 7168, 8192 76 / 62, 154 / 125, 244 / 197, 411 / 378;
// 8192, 3584 40 / 32, 79 / 61, 124 / 97, 205 / 190; 32000, 2048 at 512, 1064, 4096 93 / 85, 164 / 135, 442 / 432; 1280, 8192 (160
// tiles) 18 / 15, 40 / 30, 54 / 45, but 80 / 84: few tiles of many whole slices stay with the library, as does 8192, 1024 (128 tiles)
// 14 / 16, 31 / 29, 44 / 44, 69 / 83.  Few rows, T = 16, 64, 100: 32000, 4096 126 / 96, 121 / 103, 145 / 112; 4096, 4096 18 / 13, 16 / 14,
// 21 / 15; 1280, 8192 14 / 11, 13 / 11, 26 / 12.  Small weights of few rows: 3072, 1024 at 64, 256, 368 10.4 / 7.6, 10.5 / 9.4, 12.4 / 10.5, at 512
// 12.2 / 12.4.
// Narrow weights fill a part of their tiles only, and the rest is computed all the same: long reductions are better off with the
// library.  N, K with the share of the 256x256 tiles that is output, times as fast here, T = 24, 64, 200, 1000, 2000, 4096: 100000, 8
// (0.03) 12.7, 1.48, 1.23, 1.28, 1.33, 1.01; 32, 100000 (0.12) 8.2, 0.98, 1.03, 1.64, 1.57, 1.08; 50304, 64 (0.25) 1.27, 1.25, 1.02, 1.10, 0.98, 0.84; 50304, 96
// (0.37) 1.56, 1.39, 1.30, 1.29, 1.01, 0.86; 128, 50304 (0.50) 1.85, 1.66, 1.53, 1.23, 0.97, 0.84; 264, 30000 (0.51) 2.2, 2.0, 1.83, 1.43, 1.25, 0.85; 50304, 192
// (0.75) 1.34 at 32, 1.41, 1.30, 1.36, 1.13.
bool wgrad_grouped(int64_t t, int64_t n, int64_t k) {
  const int64_t tiles = (n + 255) / 256 * ((k + 255) / 256);
  if (t <= 0 || n > kGroupedMaxRow || k > kGroupedMaxRow) return false;
  if (tiles < 160) return t <= 384 && n * k <= 3200000;
  if ((tiles < 224 && t % 64 == 0 && t >= 2048) || 2 * t * std::max(n, k) >= (int64_t)1 << 31) return false;
  const double share = (double)(n * k) / (double)(tiles * 65536);
  return share >= 0.7 || t <= (std::min(n, k) <= 128 ? 1500 : 3500);
}

// out [N, K] (+)= grad [T, N]^T @ data [T, K] by the grouped kernel; false, and nothing done, where it is not the faster one or does
// not take the operands.
bool wgrad(const Tensor &grad, const Tensor &data, const Tensor &out, bool accumulate, const OptStream &stream) {
  const auto type = grad.scalar_type();
  if (!grouped_ok(grad, type) || !grouped_ok(data, type) || !grouped_ok(out, type)) return false;
  const int64_t t = grad.size(0), n = grad.size(1), k = data.size(1);
  if (data.size(0) != t || out.size(0) != n || out.size(1) != k || !wgrad_grouped(t, n, k)) return false;
  On on(stream);
  const Held ws = scratch(kGrouped, (int64_t)dh_grouped_gemm_workspace_bytes(), grad, on.get());
  launch([&] {
    return dh_grouped_gemm_tn_ws(grad.data_ptr(), data.data_ptr(), out.data_ptr(), nullptr, 1, t, n, k, accumulate, dt(grad),
                                 ws.data_ptr(), (size_t)ws.numel(), on.get());
  }, ws.own);
  return true;
}

Tensor dgrad(const Tensor &grad, const Tensor &weight, const OptTensor &out, const OptStream &stream) {
  const auto type = grad.scalar_type();
  if (grouped_ok(grad, type) && grouped_ok(weight, type) && grad.size(1) == weight.size(0) &&
      dgrad_grouped(grad.size(0), weight.size(0), weight.size(1)) &&
      (!out.has_value() || (grouped_ok(*out, type) && out->sizes() == at::IntArrayRef({grad.size(0), weight.size(1)})))) {
    const int64_t t = grad.size(0), n = weight.size(0), k = weight.size(1);
    On on(stream);
    Tensor d = out.has_value() ? *out : at::empty({t, k}, grad.options());
    const Held ws = scratch(kGrouped, (int64_t)dh_grouped_gemm_workspace_bytes(), grad, on.get());
    launch([&] {
      return dh_grouped_gemm_nn(grad.data_ptr(), weight.data_ptr(), d.data_ptr(), nullptr, 1, t, k, n, dt(grad), ws.data_ptr(),
                                (size_t)ws.numel(), on.get());
    }, ws.own);
    return d;
  }
  return matmul(weight, grad, out, false, stream);
}

Tensor transpose_2d(const Tensor &src, const OptTensor &out, const OptStream &stream) {
  need_gpu({&src});
  TORCH_CHECK(src.dim() == 2 && src.stride(1) == 1, "transpose_2d: src must be 2-D with unit inner stride");
  const int64_t rows = src.size(0), cols = src.size(1);
  const int type = dt(src);
  On on(stream);
  Tensor o;
  if (out.has_value()) {
    o = *out;
    TORCH_CHECK(o.dim() == 2 && o.size(0) == cols && o.size(1) == rows && o.stride(1) == 1 && o.scalar_type() == src.scalar_type(),
                "transpose_2d: out must be [cols, rows] of src's dtype with unit inner stride");
  } else {
    o = at::empty({cols, rows}, src.options());
  }
  launch([&] {
    return dh_transpose_2d(src.data_ptr(), o.data_ptr(), rows, cols, src.stride(0), o.stride(0), type, on.get());
  });
  return o;
}

// ---- attention ------------------------------------------------------------------------------------------------------
int64_t token_stride(const Tensor &t) {
  TORCH_CHECK(t.dim() == 3 && t.stride(2) == 1 && t.stride(1) == t.size(2),
              "attention tensors must be [tokens, heads, d] with contiguous (heads, d)");
  return t.stride(0);
}

// -> (out, lse)
std::tuple<Tensor, Tensor> attn_fwd(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &cu_q,
                                    const Tensor &cu_k, int max_q, int max_k, double scale, bool causal,
                                    const OptStream &stream) {
  need_gpu({&q, &k, &v, &cu_q, &cu_k});
  TORCH_CHECK(cu_q.scalar_type() == at::kInt && cu_k.scalar_type() == at::kInt, "cu_seqlens must be int32");
  const int64_t qs = token_stride(q), ks = token_stride(k), vs = token_stride(v);
  const int b = (int)cu_q.numel() - 1, type = dt(q);
  On on(stream);
  Tensor out = at::empty(q.sizes(), q.options());
  Tensor lse = at::empty({b, q.size(1), max_q}, q.options().dtype(at::kFloat));
  launch([&] {
    return dh_attn_fwd_total(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr<float>(), cu_q.data_ptr<int>(),
                             cu_k.data_ptr<int>(), 0, 0, b, max_q, max_k, q.size(0), (int)q.size(1), (int)k.size(1),
                             (int)q.size(2), qs, ks, vs, token_stride(out), (float)scale, causal, type, on.get());
  });
  return {out, lse};
}

// dq, dk, dv and (optional) delta are the caller's; with accumulate_dq this call's dq is added to what dq holds.
void attn_bwd(const Tensor &dout, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &out, const Tensor &lse,
              const Tensor &dq, const Tensor &dk, const Tensor &dv, const OptTensor &delta, const Tensor &cu_q,
              const Tensor &cu_k, int max_q, int max_k, double scale, bool causal, bool accumulate_dq,
              const OptStream &stream) {
  need_gpu({&dout, &q, &k, &v, &out, &lse, &dq, &dk, &dv, &cu_q, &cu_k});
  TORCH_CHECK(!delta.has_value() || delta->is_cuda(), "dhellam operators need tensors on the GPU");
  TORCH_CHECK(cu_q.scalar_type() == at::kInt && cu_k.scalar_type() == at::kInt, "cu_seqlens must be int32");
  const int b = (int)cu_q.numel() - 1, hq = (int)q.size(1), hk = (int)k.size(1), d = (int)q.size(2), type = dt(q);
  On on(stream);
  const size_t bytes = dh_attn_bwd_workspace_bytes(q.size(0), k.size(0), b, max_q, hq, hk, d, type);
  const Held ws = scratch(kAttnBwd, (int64_t)bytes, q, on.get());
  launch([&] {
    return dh_attn_bwd_acc(dout.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr<float>(),
                           dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), (float *)mptr(delta), ws.data_ptr(),
                           (size_t)ws.numel(), cu_q.data_ptr<int>(), cu_k.data_ptr<int>(), b, max_q, max_k, q.size(0),
                           k.size(0), hq, hk, d, token_stride(q), token_stride(k), token_stride(v), token_stride(out),
                           token_stride(dout), token_stride(dq), token_stride(dk), token_stride(dv), (float)scale, causal,
                           accumulate_dq, type, on.get());
  }, ws.own);
}

// ---- attention on the packed projection, as a layer calls it: split, RoPE (inv_freq given), attention in one call ------------
// Packed rows are [q heads of the group | k | v] per kv group; one group: q, k, v are views, several: contiguous copies.
// -> (out [T, hq, d], q, k, v, lse)
std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor> attn_fwd_packed(const Tensor &qkv, const Tensor &cu_q, const Tensor &cu_k, int64_t hq,
                                                                   int64_t hk, int64_t d, int seq, double scale,
                                                                   const OptTensor &inv_freq, const OptStream &stream) {
  TORCH_CHECK(qkv.dim() == 2 && qkv.is_contiguous() && qkv.size(1) == (hq + 2 * hk) * d && hq % hk == 0, "packed qkv: [T, (hq + 2 hk) d]");
  On on(stream);
  const int64_t t = qkv.size(0), r = hq / hk;
  Tensor q, k, v;
  if (hk == 1) {
    q = qkv.as_strided({t, hq, d}, {qkv.size(1), d, 1});
    k = qkv.as_strided({t, 1, d}, {qkv.size(1), d, 1}, qkv.storage_offset() + hq * d);
    v = qkv.as_strided({t, 1, d}, {qkv.size(1), d, 1}, qkv.storage_offset() + (hq + 1) * d);
  } else {
    const Tensor g = qkv.view({t, hk, (r + 2) * d});
    q = g.narrow(2, 0, r * d).contiguous().view({t, hq, d});
    k = g.narrow(2, r * d, d).contiguous();
    v = g.narrow(2, (r + 1) * d, d).contiguous();
  }
  if (inv_freq.has_value()) rope(q, k, *inv_freq, std::nullopt, seq, false, true, stream);
  auto [out, lse] = attn_fwd(q, k, v, cu_q, cu_k, seq, seq, scale, true, stream);
  return {out, q, k, v, lse};
}

// -> the packed gradient [T, (hq + 2 hk) d]
Tensor attn_bwd_packed(const Tensor &dout, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &out, const Tensor &lse,
                       const Tensor &cu_q, const Tensor &cu_k, int seq, double scale, const OptTensor &inv_freq,
                       const OptStream &stream) {
  const int64_t t = q.size(0), hq = q.size(1), hk = k.size(1), d = q.size(2), r = hq / hk, width = (hq + 2 * hk) * d;
  On on(stream);
  Tensor packed = at::empty({t, width}, q.options()), dq, dk, dv;
  if (hk == 1) {
    dq = packed.as_strided({t, hq, d}, {width, d, 1});
    dk = packed.as_strided({t, 1, d}, {width, d, 1}, hq * d);
    dv = packed.as_strided({t, 1, d}, {width, d, 1}, (hq + 1) * d);
  } else {
    dq = at::empty(q.sizes(), q.options());
    dk = at::empty(k.sizes(), k.options());
    dv = at::empty(v.sizes(), v.options());
  }
  attn_bwd(dout.view({t, hq, d}), q, k, v, out, lse, dq, dk, dv, std::nullopt, cu_q, cu_k, seq, seq, scale, true, false, stream);
  if (inv_freq.has_value()) rope(dq, dk, *inv_freq, std::nullopt, seq, true, true, stream);
  if (hk != 1) {
    Tensor to = packed.view({t, hk, (r + 2) * d});
    at::cat_out(to, {dq.view({t, hk, r * d}), dk, dv}, 2);
  }
  return packed;
}

// ---- context-parallel ring steps, causal, batch 1: one call each, on halves addressed in place ---------------------------
// q [1, 2, c, hq, d], kv [2, 1, 2, c, hk, d]; step 0 is the diagonal, steps up to the rank take the first half of the visiting
// keys, later ones the second half of the queries.  A step in Python is a dozen views, a halved cu_seqlens (a kernel each) and
// for the backward a copy of half of lse: 40 us of host time forward and 55 us backward, 12 and 17 us from here.
struct RingStep {
  bool fits = false, half_q = false, half_k = false;
  int64_t c = 0, hq = 0, hk = 0, d = 0;
  RingStep(const Tensor &q, const Tensor &kv, const Tensor &cu_q, const Tensor &cu_k, int step, int rank) {
    for (const Tensor *cu : {&cu_q, &cu_k})
      if (!(cu->is_cuda() && cu->scalar_type() == at::kInt && cu->numel() == 2 && cu->is_contiguous())) return;
    if (!(q.is_cuda() && kv.is_cuda() && q.dim() == 5 && kv.dim() == 6 && q.is_contiguous() && kv.is_contiguous() &&
          q.scalar_type() == kv.scalar_type() && (q.scalar_type() == at::kBFloat16 || q.scalar_type() == at::kHalf)))
      return;
    c = q.size(2);
    hq = q.size(3);
    d = q.size(4);
    hk = kv.size(4);
    fits = q.size(0) == 1 && q.size(1) == 2 && kv.size(0) == 2 && kv.size(1) == 1 && kv.size(2) == 2 && kv.size(3) == c &&
           kv.size(5) == d && c > 0 && (d == 64 || d == 96 || d == 128 || d == 192 || d == 256) &&
           (uintptr_t)q.data_ptr() % 16 == 0 && (uintptr_t)kv.data_ptr() % 16 == 0;
    half_k = step > 0 && step <= rank;
    half_q = step > rank;
    if (step == 0) half_q = false;
  }
  int64_t rows_q() const { return half_q ? c : 2 * c; }
  int64_t rows_k() const { return half_k ? c : 2 * c; }
};
char *at_row(const Tensor &t, int64_t row, int64_t heads, int64_t d) { return (char *)t.data_ptr() + row * heads * d * t.element_size(); }

// -> (out [rows, hq, d], lse [1, hq, rows]), or None where the operands are not of that form
py::object ring_fwd(const Tensor &q, const Tensor &kv, const Tensor &cu_q, const Tensor &cu_k, int64_t max_q, int64_t max_k,
                    int step, int rank, double scale, const OptStream &stream) {
  const RingStep r(q, kv, cu_q, cu_k, step, rank);
  if (!r.fits || max_q != 2 * r.c || max_k != 2 * r.c) return py::none();
  const int type = dt(q);
  const int64_t nq = r.rows_q(), nk = r.rows_k(), qs = r.hq * r.d, ks = r.hk * r.d;
  On on(stream);
  Tensor out = at::empty({nq, r.hq, r.d}, q.options()), lse = at::empty({1, r.hq, nq}, q.options().dtype(at::kFloat));
  launch([&] {
    return dh_attn_fwd_halves(at_row(q, r.half_q ? r.c : 0, r.hq, r.d), kv.data_ptr(), at_row(kv, 2 * r.c, r.hk, r.d), out.data_ptr(),
                              lse.data_ptr<float>(), cu_q.data_ptr<int>(), cu_k.data_ptr<int>(), r.half_q, r.half_k, 1, (int)nq,
                              (int)nk, (int)r.hq, (int)r.hk, (int)r.d, qs, ks, ks, qs, (float)scale, step == 0, type, on.get());
  });
  return py::make_tuple(out, lse);
}

// -> (dq like q, dkv like kv), or None; a step's dq is stored by the backward's first call and added by the later ones
py::object ring_bwd(const Tensor &dout, const Tensor &out, const Tensor &q, const OptTensor &dq_in, const Tensor &kv, const Tensor &lse,
                    const Tensor &cu_q, const Tensor &cu_k, int64_t max_q, int64_t max_k, int step, int rank, bool first, double scale,
                    const OptStream &stream) {
  const RingStep r(q, kv, cu_q, cu_k, step, rank);
  const auto like_q = [&](const Tensor &t) {
    return t.is_cuda() && t.is_contiguous() && t.numel() == q.numel() && t.scalar_type() == q.scalar_type();
  };
  if (!r.fits || max_q != 2 * r.c || max_k != 2 * r.c || !like_q(dout) || !like_q(out) || !lse.is_cuda() || !lse.is_contiguous() ||
      lse.scalar_type() != at::kFloat || lse.numel() != 2 * r.c * r.hq || (dq_in.has_value() && !like_q(*dq_in)))
    return py::none();
  const int type = dt(q);
  const int64_t nq = r.rows_q(), nk = r.rows_k(), q_at = r.half_q ? r.c : 0, qs = r.hq * r.d, ks = r.hk * r.d;
  On on(stream);
  Tensor dq = dq_in.has_value() ? *dq_in : at::empty(q.sizes(), q.options());
  Tensor dkv = at::empty(kv.sizes(), kv.options());
  if (r.half_k) dkv.select(2, 1).zero_();
  if (first && r.half_q) dq.select(1, 0).zero_();      // the first contribution to these rows is an addition
  const size_t bytes = dh_attn_bwd_workspace_bytes(nq, nk, 1, (int)nq, (int)r.hq, (int)r.hk, (int)r.d, type);
  const Held ws = scratch(kAttnBwd, (int64_t)bytes, q, on.get());
  launch([&] {
    return dh_attn_bwd_halves(at_row(dout, q_at, r.hq, r.d), at_row(q, q_at, r.hq, r.d), kv.data_ptr(), at_row(kv, 2 * r.c, r.hk, r.d),
                              at_row(out, q_at, r.hq, r.d), lse.data_ptr<float>() + q_at, at_row(dq, q_at, r.hq, r.d), dkv.data_ptr(),
                              at_row(dkv, 2 * r.c, r.hk, r.d), nullptr, ws.data_ptr(), (size_t)ws.numel(), cu_q.data_ptr<int>(),
                              cu_k.data_ptr<int>(), r.half_q, r.half_k, (int)(2 * r.c), 1, (int)nq, (int)nk, nq, nk, (int)r.hq, (int)r.hk,
                              (int)r.d, qs, ks, ks, qs, qs, qs, ks, ks, (float)scale, step == 0, !first, type, on.get());
  }, ws.own);
  return py::make_tuple(dq, dkv);
}

// Running log-sum-exp of a ring: a copy of the first step's, or `next` folded into it in place (half: its second half of rows).
Tensor ring_lse(const OptTensor &running, const Tensor &next, bool half, const OptStream &stream) {
  On on(stream);
  if (!running.has_value()) return next.clone();
  Tensor dst = *running;
  if (half) dst = dst.narrow(-1, dst.size(-1) / 2, dst.size(-1) / 2);
  at::logaddexp_out(dst, dst, next);
  return *running;
}

void attn_merge(const std::vector<Tensor> &outs, const std::vector<Tensor> &lses, const std::vector<int> &row_begin,
                const std::vector<int> &rows, const Tensor &out, const Tensor &lse, const OptStream &stream) {
  const size_t n = outs.size();
  PY_ASSERT(lses.size() == n && row_begin.size() == n && rows.size() == n, "merge: one entry per step in every list");
  PY_ASSERT(lse.dim() == 3 && out.dim() == 3, "merge: out [b*sq, hq, d], lse [b, hq, sq]");
  const int64_t b = lse.size(0), hq = lse.size(1), sq = lse.size(2), d = out.size(2);
  std::vector<const void *> po(n);
  std::vector<const float *> pl(n);
  for (size_t s = 0; s < n; ++s) {
    PY_ASSERT(outs[s].is_contiguous() && lses[s].is_contiguous() && lses[s].scalar_type() == at::kFloat,
              "merge: partial results must be contiguous, lse in fp32");
    PY_ASSERT(outs[s].sizes() == at::IntArrayRef({b * rows[s], hq, d}) && lses[s].sizes() == at::IntArrayRef({b, hq, (int64_t)rows[s]}),
              "merge: a partial result has the wrong shape");
    po[s] = outs[s].data_ptr();
    pl[s] = lses[s].data_ptr<float>();
  }
  PY_ASSERT(out.is_contiguous() && lse.is_contiguous(), "merge: out and lse must be contiguous");
  const int type = dt(out);
  On on(stream);
  launch([&] {
    return dh_attn_merge(po.data(), pl.data(), row_begin.data(), rows.data(), (int)n, out.data_ptr(), lse.data_ptr<float>(),
                         (int)b, (int)sq, (int)hq, (int)d, type, on.get());
  });
}

// attn_merge into new tensors: (out [b * sq, hq, d], lse [b, hq, sq])
std::tuple<Tensor, Tensor> attn_merge_new(const std::vector<Tensor> &outs, const std::vector<Tensor> &lses,
                                          const std::vector<int> &row_begin, const std::vector<int> &rows, int64_t b, int64_t sq,
                                          const OptStream &stream) {
  PY_ASSERT(!outs.empty() && outs.size() == lses.size() && outs[0].dim() == 3, "merge: one entry per step in every list");
  On on(stream);
  Tensor out = at::empty({b * sq, outs[0].size(1), outs[0].size(2)}, outs[0].options());
  Tensor lse = at::empty({b, outs[0].size(1), sq}, lses[0].options());
  attn_merge(outs, lses, row_begin, rows, out, lse, stream);
  return {out, lse};
}

// ---- MoE ------------------------------------------------------------------------------------------------------------
std::tuple<Tensor, Tensor> moe_route(const Tensor &logits, int k, const OptStream &stream) {
  PY_ASSERT(logits.is_cuda() && logits.scalar_type() == at::kFloat && logits.is_contiguous() && logits.dim() == 2,
            "route_topk: logits must be a contiguous fp32 [T, E] GPU tensor");
  const int64_t t = logits.size(0);
  On on(stream);
  Tensor idx = at::empty({t, k}, logits.options().dtype(at::kInt)), gates = at::empty({t, k}, logits.options());
  launch([&] {
    return dh_moe_route_topk(logits.data_ptr<float>(), idx.data_ptr<int>(), gates.data_ptr<float>(), t, (int)logits.size(1), k,
                             on.get());
  });
  return {idx, gates};
}

// -> (tokens_per_expert, expert_offsets, sorted_idx, dest_row)
std::tuple<Tensor, Tensor, Tensor, Tensor> moe_sort(const Tensor &topk_idx, int experts, const OptStream &stream) {
  PY_ASSERT(topk_idx.is_cuda() && topk_idx.scalar_type() == at::kInt && topk_idx.is_contiguous() && topk_idx.dim() == 2,
            "sort_assignments: topk_idx must be a contiguous int32 [T, k] GPU tensor");
  const int64_t n = topk_idx.numel();
  On on(stream);
  const auto opt = topk_idx.options();
  Tensor tpe = at::empty({experts}, opt), offs = at::empty({experts + 1}, opt), order = at::empty({n}, opt), dest = at::empty({n}, opt);
  Tensor ws = at::empty({(int64_t)dh_moe_sort_workspace_bytes(n, experts)}, opt.dtype(at::kByte));
  launch([&] {
    return dh_moe_sort(topk_idx.data_ptr<int>(), tpe.data_ptr<int>(), offs.data_ptr<int>(), order.data_ptr<int>(),
                       dest.data_ptr<int>(), ws.data_ptr(), (size_t)ws.numel(), n, experts, on.get());
  });
  return {tpe, offs, order, dest};
}

Tensor moe_gather(const Tensor &x, const Tensor &sorted_idx, const OptTensor &row_scale, const Tensor &offs, int e_lo, int e_hi,
                  int64_t max_rows, int k, const OptStream &stream) {
  PY_ASSERT(x.is_cuda() && x.is_contiguous() && x.dim() == 2, "permute: rows must be a contiguous 2-D GPU tensor");
  const int type = dt(x);
  On on(stream);
  Tensor out = at::empty({max_rows, x.size(1)}, x.options());      // the kernel zeroes the unused rows
  launch([&] {
    return dh_moe_gather_rows(x.data_ptr(), sorted_idx.data_ptr<int>(), (const float *)ptr(row_scale), out.data_ptr(),
                              offs.data_ptr<int>(), e_lo, e_hi, max_rows, k, x.size(1), type, on.get());
  });
  return out;
}

Tensor moe_scatter(const Tensor &y, const Tensor &dest_row, const OptTensor &gates, const Tensor &offs, int e_lo, int e_hi,
                   int64_t tokens, int k, const OptStream &stream) {
  PY_ASSERT(y.is_cuda() && y.is_contiguous() && y.dim() == 2, "unpermute: rows must be a contiguous 2-D GPU tensor");
  const int type = dt(y);
  On on(stream);
  Tensor out = at::empty({tokens, y.size(1)}, y.options());
  launch([&] {
    return dh_moe_scatter_rows(y.data_ptr(), dest_row.data_ptr<int>(), (const float *)ptr(gates), out.data_ptr(),
                               offs.data_ptr<int>(), e_lo, e_hi, tokens, k, y.size(1), type, on.get());
  });
  return out;
}

// -> (dy [max_rows, H], dgates [T, k])
std::tuple<Tensor, Tensor> moe_unpermute_bwd(const Tensor &dout, const Tensor &y, const Tensor &sorted_idx, const Tensor &dest_row,
                                             const Tensor &gates, const Tensor &offs, int e_lo, int e_hi, int64_t max_rows,
                                             int64_t tokens, int k, const OptStream &stream) {
  PY_ASSERT(dout.is_cuda() && dout.is_contiguous() && dout.dim() == 2, "unpermute: rows must be a contiguous 2-D GPU tensor");
  PY_ASSERT(y.is_contiguous() && y.dim() == 2 && y.size(1) == dout.size(1) && y.scalar_type() == dout.scalar_type(),
            "unpermute: expert outputs must be rows like dout's");
  const int type = dt(dout);
  On on(stream);
  Tensor dy = at::empty({max_rows, dout.size(1)}, dout.options());
  Tensor dg = at::empty({tokens, k}, dout.options().dtype(at::kFloat));
  launch([&] {
    return dh_moe_unpermute_bwd(dout.data_ptr(), y.data_ptr(), sorted_idx.data_ptr<int>(), dest_row.data_ptr<int>(),
                                gates.data_ptr<float>(), dy.data_ptr(), dg.data_ptr<float>(), offs.data_ptr<int>(), e_lo, e_hi,
                                max_rows, tokens, k, dout.size(1), type, on.get());
  });
  return {dy, dg};
}

// c [R, N] = per group a [R, K] times b [G, N, K]^T (transposed) or b [G, K, N]
Tensor grouped_gemm(const Tensor &a, const Tensor &b, const Tensor &offs, std::optional<int64_t> max_rows, const OptTensor &out,
                    bool transposed, const OptStream &stream) {
  PY_ASSERT(a.dim() == 2 && b.dim() == 3 && a.is_contiguous() && b.is_contiguous(), "grouped_gemm: contiguous a [R, K], b [G, ., .]");
  const int64_t g = b.size(0), n = b.size(transposed ? 1 : 2), k = b.size(transposed ? 2 : 1), held = a.size(0);
  PY_ASSERT(a.size(1) == k && offs.numel() == g + 1, "grouped_gemm: shapes differ");
  const int type = dt(a);
  On on(stream);
  // rows past the last group are zeroed by the library; everything else is written
  Tensor c = out.has_value() ? *out : at::empty({held, n}, a.options());
  const int64_t rows = max_rows.value_or(held);
  if (!out.has_value() && rows < held) c.narrow(0, rows, held - rows).zero_();
  const Held ws = scratch(kGrouped, (int64_t)dh_grouped_gemm_workspace_bytes(), a, on.get());      // split-k pieces
  launch([&] {
    return (transposed ? dh_grouped_gemm_nt : dh_grouped_gemm_nn)(a.data_ptr(), b.data_ptr(), c.data_ptr(), offs.data_ptr<int>(),
                                                                  (int)g, rows, n, k, type, ws.data_ptr(),
                                                                  (size_t)ws.numel(), on.get());
  }, ws.own);
  return c;
}

// c [G, M, N] (+)= per group a [R, M]^T b [R, N]
Tensor grouped_gemm_tn(const Tensor &a, const Tensor &b, const Tensor &offs, const OptTensor &out, bool accumulate,
                       const OptStream &stream) {
  PY_ASSERT(a.dim() == 2 && b.dim() == 2 && a.is_contiguous() && b.is_contiguous() && a.size(0) == b.size(0),
            "grouped_gemm_tn: contiguous a [R, M], b [R, N]");
  PY_ASSERT(out.has_value() || !accumulate, "grouped_gemm_tn: nothing to accumulate into");
  const int64_t g = offs.numel() - 1, m = a.size(1), n = b.size(1);
  const int type = dt(a);
  On on(stream);
  Tensor c = out.has_value() ? *out : at::empty({g, m, n}, a.options());
  const Held ws = scratch(kGrouped, (int64_t)dh_grouped_gemm_workspace_bytes(), a, on.get());
  launch([&] {
    return dh_grouped_gemm_tn_ws(a.data_ptr(), b.data_ptr(), c.data_ptr(), offs.data_ptr<int>(), (int)g, a.size(0), m, n,
                                 accumulate, type, ws.data_ptr(), (size_t)ws.numel(), on.get());
  }, ws.own);
  return c;
}

// The SwiGLU expert FFN on permuted rows -> (y [R, H], h [R, 2F], a [R, F]).
std::tuple<Tensor, Tensor, Tensor> expert_ffn_fwd(const Tensor &xp, const Tensor &w1, const Tensor &w2, const Tensor &offs,
                                                  const OptStream &stream) {
  Tensor h = grouped_gemm(xp, w1, offs, std::nullopt, std::nullopt, true, stream);
  Tensor a = std::get<0>(swiglu_fwd(h, false, stream));
  return {grouped_gemm(a, w2, offs, std::nullopt, std::nullopt, true, stream), h, a};
}

// Its backward -> (dxp, dw1, dw2).  w1t / w2t: the weights' resident transposes, if kept: the data gradients then run in
// the forward's layout.  dw1 / dw2 are accumulated into when given.
std::tuple<Tensor, Tensor, Tensor> expert_ffn_bwd(const Tensor &dy, const Tensor &xp, const Tensor &w1, const Tensor &w2,
                                                  const OptTensor &w1t, const OptTensor &w2t, const Tensor &offs, const Tensor &h,
                                                  const Tensor &a, const OptTensor &dw1, const OptTensor &dw2,
                                                  const OptStream &stream) {
  Tensor da = grouped_gemm(dy, w2t.has_value() ? *w2t : w2, offs, std::nullopt, std::nullopt, w2t.has_value(), stream);
  Tensor g2 = grouped_gemm_tn(dy, a, offs, dw2, dw2.has_value(), stream);
  Tensor dh = std::get<0>(swiglu_bwd(da, h, std::nullopt, false, stream));
  Tensor dxp = grouped_gemm(dh, w1t.has_value() ? *w1t : w1, offs, std::nullopt, std::nullopt, w1t.has_value(), stream);
  return {dxp, grouped_gemm_tn(dh, xp, offs, dw1, dw1.has_value(), stream), g2};
}

// ---- head -----------------------------------------------------------------------------------------------------------
Tensor embedding_fwd(const Tensor &vocab, const Tensor &ids, int64_t vocab_start) {
  need_gpu({&vocab, &ids});
  PY_ASSERT(vocab.dim() == 2 && vocab.is_contiguous() && ids.scalar_type() == at::kLong, "embedding: contiguous table, int64 ids");
  const Tensor i = ids.contiguous();
  auto sizes = i.sizes().vec();
  sizes.push_back(vocab.size(1));
  const int type = dt(vocab);
  On on(py::none{});
  Tensor out = at::empty(sizes, vocab.options());
  launch([&] {
    return dh_embedding_fwd(vocab.data_ptr(), i.data_ptr<int64_t>(), i.numel(), vocab.size(1), vocab.size(0), vocab_start, type,
                            out.data_ptr(), on.get());
  });
  return out;
}

void embedding_bwd(const Tensor &dout_in, const Tensor &ids_in, const Tensor &grad, int64_t vocab_start) {
  need_gpu({&grad, &dout_in, &ids_in});
  const Tensor dout = dout_in.contiguous(), ids = ids_in.contiguous();
  PY_ASSERT(grad.dim() == 2 && grad.is_contiguous() && ids.scalar_type() == at::kLong && dout.numel() == ids.numel() * grad.size(1),
            "embedding: contiguous gradient, int64 ids, one row of dout per id");
  const int type = dt(dout), gtype = dt(grad);
  On on(py::none{});
  launch([&] {
    return dh_embedding_bwd(dout.data_ptr(), ids.data_ptr<int64_t>(), ids.numel(), grad.size(1), grad.size(0), vocab_start, type,
                            grad.data_ptr(), gtype, on.get());
  });
}

Tensor rows_of(const Tensor &t, int64_t cols) {      // [..., cols] as rows of unit inner stride
  Tensor x = t.reshape({-1, cols});
  return x.stride(1) == 1 ? x : x.contiguous();
}

// -> (statistics [4, rows]: loss, row max, exp sum, target logit; softmax or None, target mask [rows], local target [rows])
std::tuple<Tensor, OptTensor, Tensor, Tensor> cross_entropy_fwd(const Tensor &logits, const Tensor &target, int64_t vocab_start,
                                                                double label_smoothing, bool keep_softmax) {
  need_gpu({&logits, &target});
  PY_ASSERT(logits.stride(-1) == 1 && target.scalar_type() == at::kLong && target.sizes() == logits.sizes().slice(0, logits.dim() - 1),
            "cross_entropy: logits of unit inner stride, one int64 target per row");
  const int64_t cols = logits.size(-1);
  const Tensor x = rows_of(logits, cols), tgt = target.contiguous();
  const int64_t rows = x.size(0);
  const int type = dt(x);
  On on(py::none{});
  Tensor stats = at::empty({4, rows > 0 ? rows : 1}, logits.options().dtype(at::kFloat));
  OptTensor softmax;
  if (keep_softmax) softmax = at::empty({rows, cols}, logits.options());
  Tensor mask = at::empty({rows}, logits.options().dtype(at::kBool)), local = at::empty({rows}, target.options());
  float *st = stats.data_ptr<float>();
  const int64_t pitch = stats.size(1);
  launch([&] {
    return dh_cross_entropy_fwd(x.data_ptr(), tgt.data_ptr<int64_t>(), rows, cols, x.stride(0), vocab_start, (float)label_smoothing, type,
                                st, st + pitch, st + 2 * pitch, st + 3 * pitch, mptr(softmax), cols, (uint8_t *)mask.data_ptr(),
                                local.data_ptr<int64_t>(), on.get());
  });
  return {stats, softmax, mask, local};
}

// grad (made here if not given) from the logits and their row statistics
Tensor cross_entropy_bwd(const Tensor &logits, const Tensor &row_max, const Tensor &sum_exp, const Tensor &target, const Tensor &dout,
                         int64_t vocab_start, double label_smoothing, const OptTensor &grad_out) {
  need_gpu({&logits, &row_max, &sum_exp, &target, &dout});
  const int64_t cols = logits.size(-1);
  const Tensor x = rows_of(logits, cols), tgt = target.contiguous(), d = dout.to(at::kFloat).contiguous();
  PY_ASSERT(d.numel() == tgt.numel() && x.size(0) == tgt.numel() && row_max.is_contiguous() && sum_exp.is_contiguous(),
            "cross_entropy: one gradient and one pair of statistics per row");
  const int type = dt(x);
  On on(py::none{});
  const Tensor g = grad_out.has_value() ? grad_out->view({-1, cols}) : at::empty({x.size(0), cols}, logits.options());
  PY_ASSERT(g.scalar_type() == x.scalar_type() && g.stride(1) == 1, "cross_entropy: gradient of the logits' type, unit inner stride");
  launch([&] {
    return dh_cross_entropy_bwd(x.data_ptr(), x.stride(0), 1, row_max.data_ptr<float>(), sum_exp.data_ptr<float>(),
                                tgt.data_ptr<int64_t>(), d.data_ptr<float>(), x.size(0), cols, vocab_start, (float)label_smoothing, type,
                                g.data_ptr(), g.stride(0), on.get());
  });
  return g.view(logits.sizes());
}

// -> (out fp32 [2]: loss, mask sum; mask in fp32)
std::tuple<Tensor, Tensor> masked_mean_fwd(const Tensor &losses, const Tensor &mask, double scale) {
  need_gpu({&losses, &mask});
  const Tensor x = losses.to(at::kFloat).contiguous(), m = mask.reshape({-1}).to(at::kFloat).contiguous();
  PY_ASSERT(x.numel() == m.numel() && x.numel() > 0, "masked mean: one mask value per loss");
  On on(py::none{});
  Tensor out = at::empty({2}, x.options());
  launch([&] {
    return dh_masked_mean_fwd(x.data_ptr<float>(), m.data_ptr<float>(), x.numel(), (float)scale, out.data_ptr<float>(), on.get());
  });
  return {out, m};
}

Tensor masked_mean_bwd(const Tensor &mask, const Tensor &mask_sum, double scale) {
  On on(py::none{});
  Tensor g = at::empty({mask.numel()}, mask.options());
  launch([&] {
    return dh_masked_mean_bwd(mask.data_ptr<float>(), mask_sum.data_ptr<float>(), mask.numel(), (float)scale, g.data_ptr<float>(), on.get());
  });
  return g;
}

// Zeros in every tensor of the list (contiguous ones, neighbours in the list or not): one launch.
void zero_all(const std::vector<Tensor> &ts, const OptStream &stream) {
  On on(stream);
  std::vector<void *> ptrs;
  std::vector<int64_t> bytes;
  for (const Tensor &t : ts) {
    if (t.is_cuda() && t.is_contiguous() && t.nbytes() % 4 == 0 && (uintptr_t)t.data_ptr() % 16 == 0) {
      ptrs.push_back(t.data_ptr());
      bytes.push_back((int64_t)t.nbytes());
    } else {
      t.zero_();
    }
  }
  if (!ptrs.empty()) launch([&] { return dh_zero_many(ptrs.data(), bytes.data(), (int)ptrs.size(), on.get()); });
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.doc() = "host path of the dhellam_amd operators over libdhellam_hip.so";
  m.attr("SCRATCH_GEMM") = (int)kGemm;
  m.attr("GEMM_WORKSPACE_BYTES") = kGemmWorkspace;
  m.def("scratch_keys", &scratch_keys);
  m.def("stream_ptr", &stream_ptr);
  m.def("norm_fwd", &norm_fwd);
  m.def("norm_bwd", &norm_bwd);
  m.def("swiglu_fwd", &swiglu_fwd);
  m.def("swiglu_bwd", &swiglu_bwd);
  m.def("residual_add", &residual_add);
  m.def("rope", &rope);
  m.def("dense_gemm", &dense_gemm);
  m.def("linear", &linear);
  m.def("matmul", &matmul);
  m.def("dgrad", &dgrad);
  m.def("transpose_2d", &transpose_2d);
  m.def("attn_fwd", &attn_fwd);
  m.def("attn_bwd", &attn_bwd);
  m.def("attn_fwd_packed", &attn_fwd_packed);
  m.def("attn_bwd_packed", &attn_bwd_packed);
  m.def("ring_fwd", &ring_fwd);
  m.def("ring_bwd", &ring_bwd);
  m.def("ring_lse", &ring_lse);
  m.def("attn_merge", &attn_merge);
  m.def("attn_merge_new", &attn_merge_new);
  m.def("moe_route", &moe_route);
  m.def("moe_sort", &moe_sort);
  m.def("moe_gather", &moe_gather);
  m.def("moe_scatter", &moe_scatter);
  m.def("moe_unpermute_bwd", &moe_unpermute_bwd);
  m.def("expert_ffn_fwd", &expert_ffn_fwd);
  m.def("expert_ffn_bwd", &expert_ffn_bwd);
  m.def("grouped_gemm", &grouped_gemm);
  m.def("grouped_gemm_tn", &grouped_gemm_tn);
  m.def("wgrad", &wgrad);
  m.def("wgrad_grouped", &wgrad_grouped);
  m.def("dgrad_grouped", &dgrad_grouped);
  m.def("embedding_fwd", &embedding_fwd);
  m.def("embedding_bwd", &embedding_bwd);
  m.def("cross_entropy_fwd", &cross_entropy_fwd);
  m.def("cross_entropy_bwd", &cross_entropy_bwd);
  m.def("masked_mean_fwd", &masked_mean_fwd);
  m.def("masked_mean_bwd", &masked_mean_bwd);
  m.def("zero_all", &zero_all);
}
