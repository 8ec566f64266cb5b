// Native call path of the Python entry points (extension module triton_grouped_gemm_amd._host).
//
// A call through torch's custom-operator layer, the wrapper's checks and ctypes costs 9-20 us of host time, more than
// the kernel of a small problem takes.  The functions here take the ordinary eager call -- plain tensors on the current GPU
// in the form the kernels want, no gradient to record, no dispatch or function mode active -- allocate the result and cross
// the C ABI in one step (4-5 us, of which the kernel launch is 2.5).  Anything else returns None, and the Python
// wrapper goes its own way: it checks, converts, raises the documented errors and goes through the operator.  So nothing is
// decided here that the wrappers do not decide too, and no state is kept.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/record_function.h>
#include <c10/core/Event.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <chrono>
#include <optional>

#include "../../include/tgg_amd.h"

namespace {

constexpr int64_t kMaxGroups = 1024, kMaxGroupsOther = 512, kMaxExperts = 1024;

// A plain torch.Tensor (or Parameter) on the current GPU, without functorch or Python layers around it and without a
// forward-mode tangent (the wrappers' autograd functions have no jvp and say so); null otherwise.
// device: the current GPU, looked up (-1 before) once a tensor on some GPU has been seen.
const at::Tensor* plain(PyObject* o, c10::DeviceIndex& device) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided) return nullptr;
  if (device < 0) device = c10::hip::current_device();
  if (t.device().index() != device) return nullptr;
  static const c10::DispatchKeySet layered({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                            c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                            c10::DispatchKey::Conjugate, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor,
                                            c10::DispatchKey::Batched});
  return t.key_set().has_any(layered) || t._fw_grad(/*level=*/0).defined() ? nullptr : &t;
}

bool modes_active() {
  static const c10::DispatchKeySet watched({c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::Functionalize,
                                            c10::DispatchKey::Python, c10::DispatchKey::Tracer});
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
         c10::impl::tls_local_dispatch_key_set().included_.has_any(watched);
}

// Whether the dispatcher has an implementation or a rule of someone else's for the operator on GPU tensors (the operator's
// own ones serve all devices): a call then goes through it.
bool replaced(const c10::OperatorName& op) {
  const auto handle = c10::Dispatcher::singleton().findOp(op);
  return handle && (handle->hasKernelForDispatchKey(c10::DispatchKey::CUDA) || handle->hasKernelForDispatchKey(c10::DispatchKey::AutocastCUDA) ||
                    handle->hasKernelForDispatchKey(c10::DispatchKey::AutogradCUDA));
}

bool records(const at::Tensor& t) { return t.requires_grad() && c10::GradMode::is_enabled(); }

void* stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

int code16(const at::Tensor& t) {
  return t.scalar_type() == at::kBFloat16 ? TGG_BF16 : (t.scalar_type() == at::kHalf ? TGG_F16 : -1);
}
int code8(const at::Tensor& t) {
  return t.scalar_type() == at::kFloat8_e4m3fn ? TGG_E4M3 : (t.scalar_type() == at::kFloat8_e5m2 ? TGG_E5M2 : -1);
}
int code_act(const at::Tensor& t) { return t.scalar_type() == at::kFloat ? 4 : code16(t) >= 0 ? code16(t) : code8(t); }

// Integer sizes as the kernels read them: 1-D, contiguous, int32 or int64, `groups` long.
bool sizes_ok(const at::Tensor& s, int64_t groups) {
  return s.dim() == 1 && s.size(0) == groups && (s.scalar_type() == at::kInt || s.scalar_type() == at::kLong) && s.is_contiguous();
}
int is64(const at::Tensor& s) { return s.scalar_type() == at::kLong; }

PyObject* done(const char* name, int rc, const at::Tensor& result) {
  if (rc != 0) {
    PyErr_Format(PyExc_RuntimeError, "%s failed (code %d): %s", name, rc, tgg_last_error());
    return nullptr;
  }
  return THPVariable_Wrap(result);
}

// The interpreter lock is given up in the scope of one of these, and taken again also where an exception leaves it: the
// allocation and the launch can both block (a device allocation; a stream with a full queue) and must not stop the other
// host threads.  Giving it up and taking it back does not show in the time of a call (5.2 us of host time either way).
class Unlocked {
 public:
  Unlocked() : state_(PyEval_SaveThread()) {}
  ~Unlocked() { PyEval_RestoreThread(state_); }
  Unlocked(const Unlocked&) = delete;
  Unlocked& operator=(const Unlocked&) = delete;

 private:
  PyThreadState* const state_;
};

#define TGG_ARGS(n) \
  if (nargs != (n)) { PyErr_SetString(PyExc_TypeError, "wrong number of arguments"); return nullptr; } \
  if (modes_active()) Py_RETURN_NONE; \
  c10::DeviceIndex device = -1
#define TGG_TENSOR(name, i) \
  const at::Tensor* const name##_p = plain(args[i], device); \
  if (!name##_p) Py_RETURN_NONE; \
  const at::Tensor& name = *name##_p
#define TGG_INT(name, i) \
  const long name = PyLong_AsLong(args[i]); \
  if (name == -1 && PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
#define TGG_TRUTH(name, i) \
  if (!PyBool_Check(args[i])) Py_RETURN_NONE; \
  const bool name = args[i] == Py_True

// (A, B, sizes, trans_b, num_cu) -> C
PyObject* m_grouped_gemm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TGG_ARGS(5);
  TGG_TENSOR(a, 0);
  TGG_TENSOR(b, 1);
  TGG_TENSOR(sizes, 2);
  TGG_TRUTH(trans_b, 3);
  TGG_INT(num_cu, 4);
  if (a.dim() != 2 || b.dim() != 3 || records(a) || records(b)) Py_RETURN_NONE;
  const int64_t m = a.size(0), k = a.size(1), g = b.size(0), n = b.size(trans_b ? 1 : 2);
  const int dt = code16(a);
  if (dt < 0 || b.scalar_type() != a.scalar_type() || b.size(trans_b ? 2 : 1) != k || (n & 7) || (k & 7) || g > kMaxGroups ||
      !sizes_ok(sizes, g) || !a.is_contiguous() || !b.is_contiguous())
    Py_RETURN_NONE;
  static const c10::OperatorName op("moe::m_grouped_gemm", "");
  if (replaced(op)) Py_RETURN_NONE;
  RECORD_FUNCTION(op.name, std::vector<c10::IValue>({a, b, sizes, trans_b, (int64_t)num_cu}));  // under the operator's name
  at::Tensor c;
  int rc;
  {
    const Unlocked unlocked;
    c = at::empty({m, n}, a.options());
    rc = tgg_m_grouped_gemm(a.data_ptr(), b.data_ptr(), c.data_ptr(), sizes.data_ptr(), is64(sizes), (int)g, m, (int)n, (int)k,
                            trans_b, dt, (int)num_cu, stream());
  }
  return done("tgg_m_grouped_gemm", rc, c);
  END_HANDLE_TH_ERRORS
}

// (lhs, rhs, out, masked_m, expected_m, trans_b) -> out
PyObject* m_grouped_gemm_masked(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TGG_ARGS(6);
  TGG_TENSOR(a, 0);
  TGG_TENSOR(b, 1);
  TGG_TENSOR(out, 2);
  TGG_TENSOR(sizes, 3);
  TGG_INT(stride, 4);
  TGG_TRUTH(trans_b, 5);
  if (a.dim() != 2 || b.dim() != 3 || out.dim() != 2 || out.requires_grad()) Py_RETURN_NONE;
  const int64_t m = a.size(0), k = a.size(1), g = b.size(0), n = b.size(trans_b ? 1 : 2);
  const int dt = code16(a);
  if (dt < 0 || b.scalar_type() != a.scalar_type() || out.scalar_type() != a.scalar_type() || b.size(trans_b ? 2 : 1) != k ||
      (n & 7) || (k & 7) || m % 128 || out.size(0) != m || out.size(1) != n || stride < 0 || g * stride > m ||
      g > kMaxGroupsOther || !sizes_ok(sizes, g) || !a.is_contiguous() || !b.is_contiguous() || !out.is_contiguous())
    Py_RETURN_NONE;
  int rc;
  {
    const Unlocked unlocked;
    rc = tgg_m_grouped_gemm_masked(a.data_ptr(), b.data_ptr(), out.data_ptr(), sizes.data_ptr(), is64(sizes), (int)g, stride, m,
                                   (int)n, (int)k, trans_b, dt, -1, stream());
  }
  return done("tgg_m_grouped_gemm_masked", rc, out);
  END_HANDLE_TH_ERRORS
}

// (A, B, sizes, num_cu, queue) -> C
PyObject* k_grouped_gemm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TGG_ARGS(5);
  TGG_TENSOR(a, 0);
  TGG_TENSOR(b, 1);
  TGG_TENSOR(sizes, 2);
  TGG_INT(num_cu, 3);
  TGG_TENSOR(queue, 4);
  if (a.dim() != 2 || b.dim() != 2 || sizes.dim() != 1) Py_RETURN_NONE;
  const int64_t kt = a.size(0), m = a.size(1), n = b.size(1), g = sizes.size(0);
  const int dt = code16(a);
  if (dt < 0 || b.scalar_type() != a.scalar_type() || b.size(0) != kt || (m & 7) || (n & 7) || g < 1 || g > kMaxGroups ||
      !sizes_ok(sizes, g) || !a.is_contiguous() || !b.is_contiguous() || ((uintptr_t)a.data_ptr() & 15) || ((uintptr_t)b.data_ptr() & 15))
    Py_RETURN_NONE;
  at::Tensor c;
  int rc;
  {
    const Unlocked unlocked;
    c = at::empty({g, m, n}, a.options());
    at::Tensor workspace;  // of launches that are cut along K; the allocator keeps it for the stream's next ones
    int64_t bytes = 0;
    rc = tgg_k_grouped_split_bytes((int)g, (int)m, (int)n, kt, 0, (int)num_cu, &bytes);
    if (bytes > 0) {
      try {
        workspace = at::empty({bytes}, a.options().dtype(at::kByte));
      } catch (const c10::OutOfMemoryError&) {  // it runs without one as well, only longer
        bytes = 0;
      }
    }
    if (rc == 0)
      rc = tgg_k_grouped_gemm_split(a.data_ptr(), b.data_ptr(), c.data_ptr(), sizes.data_ptr(), is64(sizes), (int)g, (int)m, (int)n, kt, dt,
                                    (int)num_cu, (int32_t*)queue.data_ptr(), bytes > 0 ? workspace.data_ptr() : nullptr, bytes, stream());
  }
  return done("tgg_k_grouped_gemm_split", rc, c);
  END_HANDLE_TH_ERRORS
}

// (A, A_scale, B, B_scale, sizes, out_is_fp16) -> C
PyObject* m_grouped_gemm_fp8_channel(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TGG_ARGS(6);
  TGG_TENSOR(a, 0);
  TGG_TENSOR(sa, 1);
  TGG_TENSOR(b, 2);
  TGG_TENSOR(sb, 3);
  TGG_TENSOR(sizes, 4);
  TGG_TRUTH(fp16, 5);
  if (a.dim() != 2 || b.dim() != 3 || records(a) || records(sa) || records(b) || records(sb)) Py_RETURN_NONE;
  const int64_t m = a.size(0), k = a.size(1), g = b.size(0), n = b.size(1);
  const int fa = code8(a), fb = code8(b);
  if (fa < 0 || fb < 0 || b.size(2) != k || sa.numel() != m || sb.numel() != g * n || sa.scalar_type() != at::kFloat ||
      sb.scalar_type() != at::kFloat || !sa.is_contiguous() || !sb.is_contiguous() || g > kMaxGroupsOther ||
      !sizes_ok(sizes, g) || !a.is_contiguous() || !b.is_contiguous())
    Py_RETURN_NONE;
  static const c10::OperatorName op("myfp8::gmm_fp8_act_per_channel_w_per_expert", "");
  if (replaced(op)) Py_RETURN_NONE;
  RECORD_FUNCTION(op.name, std::vector<c10::IValue>({a, sa, b, sb, sizes}));
  at::Tensor c;
  int rc;
  {
    const Unlocked unlocked;
    c = at::empty({m, n}, a.options().dtype(fp16 ? at::kHalf : at::kBFloat16));
    rc = tgg_m_grouped_gemm_fp8_channel(a.data_ptr(), (const float*)sa.data_ptr(), b.data_ptr(), (const float*)sb.data_ptr(), c.data_ptr(),
                                        sizes.data_ptr(), is64(sizes), (int)g, m, (int)n, (int)k, fa, fb, fp16 ? TGG_F16 : TGG_BF16,
                                        -1, stream());
  }
  return done("tgg_m_grouped_gemm_fp8_channel", rc, c);
  END_HANDLE_TH_ERRORS
}

// Gives (first, second) as a Python pair.
PyObject* pair(const at::Tensor& first, const at::Tensor& second) {
  PyObject* const t = PyTuple_New(2);
  if (!t) return nullptr;
  PyTuple_SET_ITEM(t, 0, THPVariable_Wrap(first));
  PyTuple_SET_ITEM(t, 1, THPVariable_Wrap(second));
  return t;
}

// The sort's workspace; undefined when it needs none.
at::Tensor sort_workspace(int64_t tokens, int64_t topk, int64_t experts, const at::Tensor& like, int64_t& bytes) {
  bytes = 0;
  if (tgg_moe_sort_workspace_bytes(tokens, (int)topk, (int)experts, &bytes) != 0 || bytes == 0) return at::Tensor();
  return at::empty({bytes}, like.options().dtype(at::kByte));
}

// (indices, num_out_tokens, num_experts, counts_i64) -> (row_id_map, counts)
PyObject* permute_map(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TGG_ARGS(4);
  TGG_TENSOR(idx, 0);
  TGG_INT(keep, 1);
  TGG_INT(experts, 2);
  TGG_TRUTH(wide, 3);
  if (idx.dim() != 2 || idx.scalar_type() != at::kInt || !idx.is_contiguous() || experts < 1 || experts > kMaxExperts) Py_RETURN_NONE;
  const int64_t tokens = idx.size(0), topk = idx.size(1);
  at::Tensor map, counts;
  int rc;
  {
    const Unlocked unlocked;
    map = at::empty({tokens * topk}, idx.options());
    counts = at::empty({experts}, idx.options().dtype(wide ? at::kLong : at::kInt));
    int64_t bytes;
    const at::Tensor ws = sort_workspace(tokens, topk, experts, idx, bytes);
    rc = tgg_moe_permute_map((const int32_t*)idx.data_ptr(), tokens, (int)topk, (int)experts, keep, (int32_t*)map.data_ptr(),
                             counts.data_ptr(), wide, ws.defined() ? ws.data_ptr() : nullptr, bytes, stream());
  }
  return rc != 0 ? done("tgg_moe_permute_map", rc, map) : pair(map, counts);
  END_HANDLE_TH_ERRORS
}

// (input, indices, num_out_tokens, num_experts) -> (permuted, row_id_map); records nothing
PyObject* permute(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TGG_ARGS(4);
  TGG_TENSOR(x, 0);
  TGG_TENSOR(idx, 1);
  TGG_INT(keep, 2);
  TGG_INT(experts, 3);
  if (x.dim() != 2 || idx.dim() != 2 || idx.scalar_type() != at::kInt || !x.is_contiguous() || !idx.is_contiguous() || x.numel() == 0 ||
      x.size(0) != idx.size(0) || code_act(x) < 0 || experts < 1 || experts > kMaxExperts)
    Py_RETURN_NONE;
  const int64_t tokens = idx.size(0), topk = idx.size(1), hidden = x.size(1), rows = keep > 0 ? keep : tokens * topk;
  at::Tensor map, out;
  int rc;
  {
    const Unlocked unlocked;
    map = at::empty({tokens * topk}, idx.options());
    out = at::empty({rows, hidden}, x.options());
    int64_t bytes;
    const at::Tensor ws = sort_workspace(tokens, topk, experts, idx, bytes);
    rc = tgg_moe_permute(x.data_ptr(), out.data_ptr(), (const int32_t*)idx.data_ptr(), tokens, (int)topk, (int)experts, keep, (int)hidden,
                         code_act(x), (int32_t*)map.data_ptr(), nullptr, 0, ws.defined() ? ws.data_ptr() : nullptr, bytes, stream());
  }
  return rc != 0 ? done("tgg_moe_permute", rc, map) : pair(out, map);
  END_HANDLE_TH_ERRORS
}

// (input, row_id_map, probs or None) -> out; records nothing
PyObject* unpermute(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TGG_ARGS(3);
  TGG_TENSOR(x, 0);
  TGG_TENSOR(map, 1);
  if (x.dim() != 2 || !x.is_contiguous() || x.numel() == 0 || code_act(x) < 0 || map.scalar_type() != at::kInt || !map.is_contiguous()) Py_RETURN_NONE;
  int64_t tokens = x.size(0), topk = 1;
  const float* weights = nullptr;
  if (args[2] != Py_None) {
    TGG_TENSOR(probs, 2);
    if (probs.dim() != 2 || probs.scalar_type() != at::kFloat || !probs.is_contiguous() || map.size(0) != probs.numel()) Py_RETURN_NONE;
    tokens = probs.size(0);
    topk = probs.size(1);
    weights = (const float*)probs.data_ptr();
  } else if (map.numel() < tokens) {  // fewer entries than rows of x: the wrapper raises
    Py_RETURN_NONE;
  }
  at::Tensor out;
  int rc;
  {
    const Unlocked unlocked;
    out = at::empty({tokens, x.size(1)}, x.options());
    rc = tgg_moe_unpermute(x.data_ptr(), out.data_ptr(), (const int32_t*)map.data_ptr(), weights, tokens, (int)topk, (int)x.size(1),
                           code_act(x), stream());
  }
  return done("tgg_moe_unpermute", rc, out);
  END_HANDLE_TH_ERRORS
}

// The padded total of a contiguous layout against the rows of A (the reference reads it back too,
// gemm/deep_gemm_ops.py:49-51).  It is asked for in front of the GEMM and waited for behind the GEMM's launch, so the GPU has the GEMM to work on
// meanwhile; the GEMM never touches rows at or beyond M, whatever the sizes say.  Two ways:
//   brief: a kernel sums the sizes and writes the total to page-locked memory, and the host watches that word.  For GEMMs that are over before a copy
//          and an event are: 16 experts, 896 rows, N = 2048, K = 1024 26 -> 19 us a call; 4 of 1664, N = 896, K = 512 23 -> 15.5.  The memory
//          is the call's own until the word has been written.
//   else:  the sizes are copied, and an event behind the copy is waited for, which takes longer but puts no kernel in front of the
//          GEMM (66-85 us a call either way; with the kernel a call of 954 us takes 958).
class PaddedTotal {
 public:
  PaddedTotal(const at::Tensor& sizes, int64_t block_m, bool brief) : block_m_(block_m) {
    if (brief) {
      word_ = at::empty({2}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
      word()[1] = 0;
      rc_ = tgg_padded_total(sizes.data_ptr(), is64(sizes), (int)sizes.size(0), block_m, word(), stream());
      return;
    }
    sizes_ = sizes.to(at::TensorOptions(sizes.options()).device(at::kCPU), /*non_blocking=*/true);
    // torch's streams and events carry the device type CUDA
    event_.emplace(c10::DeviceType::CUDA);
    event_->record(c10::Stream(c10::Stream::UNSAFE, sizes.device(), c10::hip::getCurrentHIPStream().id()));
  }
  int rc() const { return rc_; }
  int64_t wait() {
    if (event_) return read_back();
    // a word that is long in coming (the stream has other work) is not watched but waited for; what the GPU could not run throws there
    const auto patience = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
    while (!written()) {
      if (std::chrono::steady_clock::now() < patience) continue;
      c10::hip::getCurrentHIPStream().synchronize();
      TORCH_CHECK(written(), "the padded total was not written");
    }
    return word()[0];
  }
  ~PaddedTotal() {  // also where something throws before wait(): the GPU is not to write to memory that has been given back
    if (event_ || rc_ != 0 || written()) return;
    try {
      c10::hip::getCurrentHIPStream().synchronize();
    } catch (...) {
    }
  }
  PaddedTotal(const PaddedTotal&) = delete;
  PaddedTotal& operator=(const PaddedTotal&) = delete;

 private:
  int64_t* word() { return word_.data_ptr<int64_t>(); }
  bool written() { return __atomic_load_n(word() + 1, __ATOMIC_ACQUIRE) != 0; }
  int64_t read_back() {
    event_->synchronize();
    int64_t total = 0;
    for (int64_t g = 0; g < sizes_.size(0); ++g) {
      const int64_t v = sizes_.scalar_type() == at::kLong ? (int32_t)sizes_.const_data_ptr<int64_t>()[g] : sizes_.const_data_ptr<int32_t>()[g];
      const int64_t up = v + block_m_ - 1;
      total += (up >= 0 ? up / block_m_ : -((block_m_ - 1 - up) / block_m_)) * block_m_;
    }
    return total;
  }
  const int64_t block_m_;
  at::Tensor word_, sizes_;
  std::optional<c10::Event> event_;
  int rc_ = 0;
};

// Whether a GEMM is over within some 30 us: its products, and the weights of the groups that can have rows.  (No groups: no sizes to sum either, the
// total of 0 is the other way's, with its errors.)
bool brief_gemm(int64_t m, int64_t n, int64_t k, int64_t groups, int64_t block_m, int64_t element_bytes) {
  if (groups < 1) return false;
  const int64_t used = std::min(groups, (m + block_m - 1) / block_m);
  return 2.0 * m * n * k * element_bytes <= 4e10 && (double)used * n * k * element_bytes <= 1.5e8;
}

// Runs `gemm`, which returns the C ABI's code, with the total looked at behind it, or in front of it where the result is the
// caller's tensor, which then stays as it is if the total is wrong.
template <class Gemm>
PyObject* padded_gemm(const char* name, const at::Tensor& sizes, int64_t block_m, int64_t m, bool brief, const at::Tensor& c, bool callers, Gemm gemm) {
  int rc = 0;
  int64_t total = m;
  {
    const Unlocked unlocked;
    PaddedTotal padded(sizes, block_m, brief);
    rc = padded.rc();
    if (rc == 0 && callers) total = padded.wait();
    if (rc == 0 && total == m) rc = gemm();
    if (rc == 0 && !callers) total = padded.wait();
  }
  if (total != m) {
    PyErr_Format(PyExc_ValueError, "A must include padded expert rows: expected M=%lld, got M=%lld", (long long)total, (long long)m);
    return nullptr;
  }
  return done(name, rc, c);
}

bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }

// (a, b, sizes, out or None, block_m) -> out
PyObject* m_grouped_bf16_contiguous(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TGG_ARGS(5);
  TGG_TENSOR(a, 0);
  TGG_TENSOR(b, 1);
  TGG_TENSOR(sizes, 2);
  TGG_INT(block_m, 4);
  if (a.dim() != 2 || b.dim() != 3 || capturing()) Py_RETURN_NONE;
  const int64_t m = a.size(0), k = a.size(1), g = b.size(0), n = b.size(1);
  if (a.scalar_type() != at::kBFloat16 || b.scalar_type() != at::kBFloat16 || b.size(2) != k || (n & 7) || (k & 7) || block_m < 1 ||
      g > kMaxGroupsOther || !sizes_ok(sizes, g) || !a.is_contiguous() || !b.is_contiguous())
    Py_RETURN_NONE;
  at::Tensor c;
  const bool callers = args[3] != Py_None;
  if (callers) {
    TGG_TENSOR(out, 3);
    if (out.scalar_type() != at::kBFloat16 || !out.is_contiguous() || out.numel() != m * n || out.requires_grad()) Py_RETURN_NONE;
    c = out;
  }
  return padded_gemm("tgg_m_grouped_gemm_padded", sizes, block_m, m, brief_gemm(m, n, k, g, block_m, 2), c, callers, [&] {
    if (!callers) c = at::empty({m, n}, a.options());
    return tgg_m_grouped_gemm_padded(a.data_ptr(), b.data_ptr(), c.data_ptr(), sizes.data_ptr(), is64(sizes), (int)g, m, (int)n, (int)k,
                                     (int)block_m, TGG_BF16, -1, stream());
  });
  END_HANDLE_TH_ERRORS
}

// (a codes, a scales, b codes, b scales, sizes, out or None, block_m) -> out
PyObject* m_grouped_fp8_contiguous(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TGG_ARGS(7);
  TGG_TENSOR(a, 0);
  TGG_TENSOR(sa_in, 1);
  TGG_TENSOR(b, 2);
  TGG_TENSOR(sb, 3);
  TGG_TENSOR(sizes, 4);
  TGG_INT(block_m, 6);
  if (a.dim() != 2 || b.dim() != 3 || sa_in.dim() != 2 || sb.dim() != 3 || capturing()) Py_RETURN_NONE;
  const int64_t m = a.size(0), k = a.size(1), g = b.size(0), n = b.size(1), kb = (k + 127) / 128, nb = (n + 127) / 128;
  if (a.scalar_type() != at::kFloat8_e4m3fn || b.scalar_type() != at::kFloat8_e4m3fn || b.size(2) != k || (k & 15) || block_m < 128 ||
      block_m % 128 || sa_in.size(0) != m || sa_in.size(1) != kb || sb.size(0) != g || sb.size(1) != nb || sb.size(2) != kb ||
      sa_in.scalar_type() != at::kFloat || sb.scalar_type() != at::kFloat || !sb.is_contiguous() || g > kMaxGroupsOther ||
      !sizes_ok(sizes, g) || !a.is_contiguous() || !b.is_contiguous() || m == 0)
    Py_RETURN_NONE;
  const bool mn_major = kb == 1 ? sa_in.is_contiguous() : sa_in.stride(0) == 1 && sa_in.stride(1) == m;
  if (!mn_major && !sa_in.is_contiguous()) Py_RETURN_NONE;
  at::Tensor c;
  const bool callers = args[5] != Py_None;
  if (callers) {
    TGG_TENSOR(out, 5);
    if (out.scalar_type() != at::kBFloat16 || !out.is_contiguous() || out.numel() != m * n || out.requires_grad()) Py_RETURN_NONE;
    c = out;
  }
  return padded_gemm("tgg_m_grouped_gemm_fp8_block", sizes, block_m, m, brief_gemm(m, n, k, g, block_m, 1), c, callers, [&] {
    if (!callers) c = at::empty({m, n}, a.options().dtype(at::kBFloat16));
    at::Tensor sa = sa_in;
    if (!mn_major) {  // the kernel streams one K block of all rows at a time
      sa = at::empty({kb, m}, sa_in.options());
      if (int rc = tgg_scales_to_mn_major((const float*)sa_in.data_ptr(), (float*)sa.data_ptr(), m, (int)kb, stream())) return rc;
    }
    return tgg_m_grouped_gemm_fp8_block(a.data_ptr(), (const float*)sa.data_ptr(), b.data_ptr(), (const float*)sb.data_ptr(), c.data_ptr(),
                                        sizes.data_ptr(), is64(sizes), (int)g, m, (int)n, (int)k, (int)block_m, 1, -1, stream());
  });
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"m_grouped_bf16_contiguous", (PyCFunction)(void*)m_grouped_bf16_contiguous, METH_FASTCALL, nullptr},
    {"m_grouped_fp8_contiguous", (PyCFunction)(void*)m_grouped_fp8_contiguous, METH_FASTCALL, nullptr},
    {"m_grouped_gemm", (PyCFunction)(void*)m_grouped_gemm, METH_FASTCALL, nullptr},
    {"m_grouped_gemm_masked", (PyCFunction)(void*)m_grouped_gemm_masked, METH_FASTCALL, nullptr},
    {"k_grouped_gemm", (PyCFunction)(void*)k_grouped_gemm, METH_FASTCALL, nullptr},
    {"m_grouped_gemm_fp8_channel", (PyCFunction)(void*)m_grouped_gemm_fp8_channel, METH_FASTCALL, nullptr},
    {"permute_map", (PyCFunction)(void*)permute_map, METH_FASTCALL, nullptr},
    {"permute", (PyCFunction)(void*)permute, METH_FASTCALL, nullptr},
    {"unpermute", (PyCFunction)(void*)unpermute, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
