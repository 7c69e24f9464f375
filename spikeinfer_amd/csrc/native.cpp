// Python entry of the launch-bound operators: the argument checks, output
// allocation and launch of one call in C++.
//
// The operators' Python wrappers spend 9 to 15 us a call reading tensor metadata
// and building ctypes arguments, more than their kernels take on small inputs.
// Each function here does the same for the usual form of its arguments -- plain
// tensors on one GPU, already in the dtypes and layouts the C ABI takes -- and
// returns None, with nothing launched, for every other form: the Python wrapper
// then goes on as it would without this module, converting, or raising the error
// the caller should see.  An error that the library reports once it has come to
// launching is raised here: the kernel may be queued, and an operator that updates
// in place must not run twice.  Whatever else can fail comes before the launch.
// Nothing is kept between calls.
//
// Calls reach the kernels through the C ABI (include/spikeinfer_amd.h) at the
// addresses bind() is given, so one library is loaded, by _lib.py.  The
// interpreter lock is released around them, as ctypes does.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/utils/object_ptr.h>

#include <cmath>
#include <cstring>

#include "../../include/spikeinfer_amd.h"

namespace {

// The kind of tensors taken: the GPU's, or the CPU's where the functions bound are
// a test's stand-ins on the host.
c10::DeviceType taken_on = at::kCUDA;

decltype(&spk_decode_attn) decode_attn_fn;
decltype(&spk_decode_attn_workspace_bytes) workspace_fn;
decltype(&spk_lif_pack_write_sites) lif_sites_fn;
decltype(&spk_lif_multistep) lif_fn;
decltype(&spk_prefill_attn) prefill_fn;
decltype(&spk_embed_rmsnorm) embed_fn;
decltype(&spk_add_rmsnorm) add_norm_fn;
decltype(&spk_rmsnorm_mean_t) mean_fn;
decltype(&spk_lif_gate_mul) gate_mul_fn;
decltype(&spk_linear_decode) linear_fn;
decltype(&spk_mlp_gate_lif) mlp_gate_fn;
decltype(&spk_qkv_rope_lif_pack_kv) qkv_fn;
decltype(&spk_last_error) last_error_fn;

// A call this module does not take (never seen by the caller).
struct NotTaken {};
// A call that failed with its Python exception set.
struct Failed {};
void need(bool ok) {
  if (!ok) throw NotTaken{};
}

// A plain tensor (no subclass, which may have its own semantics) on a GPU, with
// memory of its own (torch.vmap's and torch.func's wrappers have none).
const at::Tensor &tensor(PyObject *o) {
  need(THPVariable_CheckExact(o));
  const at::Tensor &t = THPVariable_Unpack(o);
  need(t.device().type() == taken_on && t.layout() == at::kStrided && !t.is_conj() && !t.is_neg() && t.has_storage());
  return t;
}

int64_t integer(PyObject *o) {
  need(PyLong_CheckExact(o));
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw NotTaken{};
  }
  return v;
}
int int32(PyObject *o) {
  const int64_t v = integer(o);
  need(v >= -0x7fffffff && v <= 0x7fffffff);
  return static_cast<int>(v);
}

float real(PyObject *o) {
  need(PyFloat_CheckExact(o));
  return static_cast<float>(PyFloat_AS_DOUBLE(o));
}

int float_code(at::ScalarType t) {
  if (t == at::kFloat) return SPK_F32;
  if (t == at::kHalf) return SPK_F16;
  if (t == at::kBFloat16) return SPK_BF16;
  throw NotTaken{};
}

at::ScalarType dtype_of(PyObject *o) {
  need(THPDtype_Check(o));
  return reinterpret_cast<THPDtype *>(o)->scalar_type;
}

void *stream_of(const at::Tensor &t) {
  return taken_on == at::kCUDA ? c10::hip::getCurrentHIPStream(t.device().index()).stream() : nullptr;
}

at::Tensor empty(at::IntArrayRef sizes, at::ScalarType dtype, const at::Tensor &like) {
  return at::empty(sizes, at::TensorOptions().dtype(dtype).device(like.device()));
}

struct Strides {
  int64_t s[4];
  explicit Strides(const at::Tensor &t) {
    for (int i = 0; i < 4; ++i) s[i] = t.stride(i);
  }
};

bool packed4(const at::Tensor &t) {
  return t.scalar_type() == at::kInt && t.dim() == 4 && t.stride(3) == 1;
}

// The interpreter lock, given up while an object of this type lives.
struct Unlocked {
  PyThreadState *const state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

template <class T> struct Same { typedef T type; };

// Calls fn(args...) without the interpreter lock; the arguments, and whatever may
// throw in working them out, are the caller's, before the lock is given up.
// SPK_EINVAL and SPK_EUNSUPPORTED come before anything is launched: the call is
// not taken, and the wrapper repeats it and raises its error.  SPK_EHIP is read
// after a launch (and may be an earlier call's error): raised as _lib.check does.
template <class... P> void launch(const char *what, int (*fn)(P...), typename Same<P>::type... args) {
  int rc;
  {
    const Unlocked unlocked;
    rc = fn(args...);
  }
  need(rc != SPK_EINVAL && rc != SPK_EUNSUPPORTED);
  if (rc == SPK_OK) return;
  PyErr_Format(PyExc_RuntimeError, "%s: %s", what, last_error_fn());
  throw Failed{};
}

// What a call returns, made before its launch: the tensor given by the caller, or
// the new one.
THPObjectPtr result(PyObject *given, const at::Tensor &made) {
  return THPObjectPtr(given == Py_None ? THPVariable_Wrap(made) : Py_NewRef(given));
}
THPObjectPtr pair(const at::Tensor &a, const at::Tensor &b) {
  THPObjectPtr r(PyTuple_New(2));
  need(r.get() != nullptr);
  PyTuple_SET_ITEM(r.get(), 0, THPVariable_Wrap(a));
  PyTuple_SET_ITEM(r.get(), 1, THPVariable_Wrap(b));
  return r;
}

// Calls f, turning NotTaken and C++ errors (an allocation that fails) into None.
template <class F> PyObject *guarded(Py_ssize_t given, Py_ssize_t wanted, F f) {
  try {
    need(given == wanted && !c10::impl::dispatch_mode_enabled());
    return f();
  } catch (const Failed &) {
    return nullptr;
  } catch (const NotTaken &) {
  } catch (const std::exception &) {
  }
  PyErr_Clear();
  Py_RETURN_NONE;
}

// decode_attn(q, k, v, tables, lens, head_dim, block_size, Hq, Hkv, out|None, dtype, workspace|None)
PyObject *decode_attn(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded(n, 12, [&]() -> PyObject * {
    const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &bt = tensor(a[3]), &lens = tensor(a[4]);
    const int D = int32(a[5]), bs = int32(a[6]), Hq = int32(a[7]), Hkv = int32(a[8]);
    need(packed4(q) && packed4(k) && packed4(v) && D > 0 && D <= 128);
    const int64_t T = q.size(0), N = q.size(1), W = (D + 31) / 32;
    need(N > 0 && N < (1 << 24) && T < (1 << 16) && q.size(2) == Hq && q.size(3) == W);
    need(k.sizes() == v.sizes() && k.size(0) == T && k.size(1) == Hkv && k.size(3) == W);
    need(bt.scalar_type() == at::kInt && bt.dim() == 2 && bt.size(0) >= N && bt.size(1) < (1 << 28));
    need(lens.scalar_type() == at::kInt && lens.is_contiguous() && lens.numel() >= N);
    need(k.device() == q.device() && v.device() == q.device() && bt.device() == q.device() &&
         lens.device() == q.device());
    at::Tensor out;
    if (a[9] == Py_None) {
      const at::ScalarType dt = dtype_of(a[10]);
      float_code(dt);
      out = empty({T, N, Hq, D}, dt, q);
    } else {
      out = tensor(a[9]);
      need(out.dim() == 4 && out.size(0) == T && out.size(1) == N && out.size(2) == Hq && out.size(3) == D &&
           out.device() == q.device());
    }
    const int code = float_code(out.scalar_type());
    const int mb = static_cast<int>(bt.size(1));
    const size_t bytes = workspace_fn(T, N, Hq, Hkv, D, bs, mb);
    at::Tensor ws;
    if (bytes) {
      if (a[11] == Py_None) {
        ws = empty({static_cast<int64_t>(bytes)}, at::kByte, q);
      } else {
        ws = tensor(a[11]);
        need(static_cast<size_t>(ws.nbytes()) >= bytes);
      }
    }
    const Strides qs(q), ks(k), vs(v), os(out);
    void *const stream = stream_of(q);
    THPObjectPtr done = result(a[9], out);
    launch("paged_spike_attn_decode", decode_attn_fn, static_cast<const int32_t *>(q.data_ptr()), qs.s,
           static_cast<const int32_t *>(k.data_ptr()), ks.s, static_cast<const int32_t *>(v.data_ptr()), vs.s,
           k.size(2), static_cast<const int32_t *>(bt.data_ptr()), bt.stride(0), bt.stride(1),
           static_cast<const int32_t *>(lens.data_ptr()), out.data_ptr(), code, os.s, static_cast<int>(T),
           static_cast<int>(N), Hq, Hkv, D, bs, mb, static_cast<float>(1.0 / std::sqrt(static_cast<double>(D))),
           bytes ? ws.data_ptr() : nullptr, bytes, stream);
    return done.release();
  });
}

// lif_sites([(x, beta, threshold, out, scatter), ...], slot_mapping|None) -> True
PyObject *lif_sites(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded(n, 2, [&]() -> PyObject * {
    need(PyList_CheckExact(a[0]));
    const Py_ssize_t count = PyList_GET_SIZE(a[0]);
    need(count >= 1 && count <= 4);
    const at::Tensor *slots = nullptr;
    if (a[1] != Py_None) {
      slots = &tensor(a[1]);
      need(slots->scalar_type() == at::kLong && slots->is_contiguous());
    }
    SpkLifSite sites[4];
    std::memset(sites, 0, sizeof sites);
    const at::Tensor *first = nullptr;
    int x_code = 0;
    for (Py_ssize_t i = 0; i < count; ++i) {
      PyObject *s = PyList_GET_ITEM(a[0], i);
      need(PyTuple_CheckExact(s) && PyTuple_GET_SIZE(s) == 5);
      const at::Tensor &x = tensor(PyTuple_GET_ITEM(s, 0)), &beta = tensor(PyTuple_GET_ITEM(s, 1)),
                       &th = tensor(PyTuple_GET_ITEM(s, 2)), &out = tensor(PyTuple_GET_ITEM(s, 3));
      need(PyBool_Check(PyTuple_GET_ITEM(s, 4)));
      const bool scatter = PyTuple_GET_ITEM(s, 4) == Py_True;
      need(x.dim() == 4 && packed4(out));
      const int64_t T = x.size(0), n_tok = x.size(1), H = x.size(2), D = x.size(3);
      need(D > 0 && H > 0 && D < (1 << 20) && H < (1 << 20) && T > 0 && T < (1 << 20) && out.size(3) == (D + 31) / 32);
      if (!first) {
        first = &x;
        x_code = float_code(x.scalar_type());
      }
      need(x.scalar_type() == first->scalar_type() && T == first->size(0) && x.device() == first->device() &&
           out.device() == x.device() && beta.device() == x.device() && th.device() == x.device());
      need(beta.dim() == 1 && th.dim() == 1 && beta.size(0) == D && th.size(0) == D && beta.is_contiguous() &&
           th.is_contiguous() && beta.scalar_type() == th.scalar_type());
      if (scatter) {
        need(slots && slots->device() == x.device() && slots->numel() >= n_tok && out.size(0) == T && out.size(1) == H);
      } else {
        need(out.size(0) == T && out.size(1) == n_tok && out.size(2) == H);
      }
      SpkLifSite &st = sites[i];
      st.x = x.data_ptr();
      for (int j = 0; j < 4; ++j) st.x_strides[j] = x.stride(j);
      st.beta = beta.data_ptr();
      st.threshold = th.data_ptr();
      st.param_dtype = float_code(beta.scalar_type());
      st.scatter = scatter ? 1 : 0;
      st.out = static_cast<int32_t *>(out.data_ptr());
      for (int j = 0; j < 3; ++j) st.out_strides[j] = out.stride(j);
      st.num_slots = scatter ? out.size(2) : 0;
      st.n_tok = n_tok;
      st.H = static_cast<int>(H);
      st.D = static_cast<int>(D);
    }
    void *const stream = stream_of(*first);
    const int T = static_cast<int>(first->size(0));
    launch("lif_pack_write_sites", lif_sites_fn, sites, static_cast<int>(count), x_code, T,
           slots ? static_cast<const int64_t *>(slots->data_ptr()) : nullptr, stream);
    Py_RETURN_TRUE;
  });
}

// lif(x, beta, threshold, return_membrane) -> spikes in x's dtype, or (spikes, membrane)
PyObject *lif(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded(n, 4, [&]() -> PyObject * {
    const at::Tensor &x = tensor(a[0]), &beta = tensor(a[1]), &th = tensor(a[2]);
    need(x.dim() >= 2 && x.is_contiguous());
    const bool membrane = a[3] == Py_True;
    const int64_t T = x.size(0), N = x.size(-1);
    need(T > 0 && T < (1 << 20) && N > 0 && N < (1 << 30) && x.numel() > 0);
    need(beta.dim() == 1 && th.dim() == 1 && beta.size(0) == N && th.size(0) == N && beta.is_contiguous() &&
         th.is_contiguous() && beta.scalar_type() == th.scalar_type() && beta.device() == x.device() &&
         th.device() == x.device());
    const int64_t M = x.numel() / (T * N);
    const int xc = float_code(x.scalar_type()), pc = float_code(beta.scalar_type());
    const at::Tensor spikes = empty(x.sizes(), x.scalar_type(), x);
    at::Tensor u;
    if (membrane) u = empty(x.sizes().slice(1), at::kFloat, x);
    const int64_t strides[3] = {M * N, N, 1};
    void *const stream = stream_of(x);
    THPObjectPtr done = membrane ? pair(spikes, u) : result(Py_None, spikes);
    launch("lif_multistep", lif_fn, x.data_ptr(), xc, strides, beta.data_ptr(), th.data_ptr(), pc, nullptr,
           spikes.data_ptr(), xc, membrane ? static_cast<float *>(u.data_ptr()) : nullptr, static_cast<int>(T), M,
           static_cast<int>(N), stream);
    return done.release();
  });
}

// prefill(q, k, v, [(q_row, out_row, q_len, ctx, table|None), ...], out, head_dim, block_size) -> True
PyObject *prefill(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded(n, 7, [&]() -> PyObject * {
    const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &out = tensor(a[4]);
    const int D = int32(a[5]), bs = int32(a[6]);
    need(packed4(q) && packed4(k) && packed4(v) && D > 0 && D <= 128 && PyList_CheckExact(a[3]));
    const int64_t T = q.size(0), Hq = q.size(2), W = (D + 31) / 32;
    need(q.size(3) == W && k.size(3) == W && k.size(0) == T && T < (1 << 16) && Hq < (1 << 16) &&
         k.size(1) < (1 << 16));
    need(k.sizes() == v.sizes() && k.strides() == v.strides());
    need(out.dim() == 4 && out.size(0) == T && out.size(2) == Hq && out.size(3) == D && out.stride(3) == 1);
    need(k.device() == q.device() && v.device() == q.device() && out.device() == q.device());
    constexpr Py_ssize_t kMost = 64;
    const Py_ssize_t count = PyList_GET_SIZE(a[3]);
    need(count >= 1 && count <= kMost);
    SpkPrefillChunk chunks[kMost];
    int64_t shift = 0;
    for (Py_ssize_t i = 0; i < count; ++i) {
      PyObject *c = PyList_GET_ITEM(a[3], i);
      need(PyTuple_CheckExact(c) && PyTuple_GET_SIZE(c) == 5);
      const int64_t q_row = integer(PyTuple_GET_ITEM(c, 0)), out_row = integer(PyTuple_GET_ITEM(c, 1));
      SpkPrefillChunk &s = chunks[i];
      s = SpkPrefillChunk{};
      s.start = q_row;
      s.q_len = int32(PyTuple_GET_ITEM(c, 2));
      s.ctx = int32(PyTuple_GET_ITEM(c, 3));
      // (differences of what lies in a tensor's range: a sum could pass 64 bits)
      need(s.q_len > 0 && q_row >= 0 && q_row <= q.size(1) - s.q_len && out_row >= 0 &&
           out_row <= out.size(1) - s.q_len);
      if (i == 0) shift = out_row - q_row;
      need(shift == out_row - q_row);
      PyObject *table = PyTuple_GET_ITEM(c, 4);
      if (table != Py_None) {
        const at::Tensor &t = tensor(table);
        need(t.scalar_type() == at::kInt && t.dim() == 1 && t.device() == q.device() && t.numel() > 0 &&
             t.numel() < (1 << 30));
        s.table = static_cast<const int32_t *>(t.data_ptr());
        s.table_stride = t.stride(0);
        s.n_table = static_cast<int>(t.numel());
      }
    }
    const Strides qs(q), ks(k), os(out);
    const int code = float_code(out.scalar_type());
    char *const dst = static_cast<char *>(out.data_ptr()) + shift * out.stride(1) * out.element_size();
    void *const stream = stream_of(q);
    launch("paged_spike_attn_prefill", prefill_fn, static_cast<const int32_t *>(q.data_ptr()), qs.s,
           static_cast<const int32_t *>(k.data_ptr()), static_cast<const int32_t *>(v.data_ptr()), ks.s, k.size(2),
           chunks, static_cast<int>(count), dst, code, os.s, static_cast<int>(T), static_cast<int>(Hq),
           static_cast<int>(k.size(1)), D, bs, static_cast<float>(1.0 / std::sqrt(static_cast<double>(D))), stream);
    Py_RETURN_TRUE;
  });
}

// A contiguous tensor of `like`'s dtype and device.
const at::Tensor &alike(PyObject *o, const at::Tensor &like) {
  const at::Tensor &t = tensor(o);
  need(t.is_contiguous() && t.scalar_type() == like.scalar_type() && t.device() == like.device());
  return t;
}
// A contiguous vector of n values on `like`'s device.
const at::Tensor &vector(PyObject *o, int64_t n, const at::Tensor &like) {
  const at::Tensor &t = tensor(o);
  need(t.is_contiguous() && t.numel() == n && t.device() == like.device());
  return t;
}

// embed_rmsnorm(ids, embed, weight, eps, T) -> (h, x)
PyObject *embed_rmsnorm(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded(n, 5, [&]() -> PyObject * {
    const at::Tensor &ids = tensor(a[0]), &embed = tensor(a[1]);
    const at::Tensor &w = alike(a[2], embed);
    const float eps = real(a[3]);
    const int T = int32(a[4]);
    need(ids.scalar_type() == at::kLong && ids.dim() == 1 && ids.is_contiguous() && ids.device() == embed.device() &&
         ids.numel() > 0 && embed.dim() == 2 && embed.is_contiguous() && w.numel() == embed.size(1) && T > 0);
    const int code = float_code(embed.scalar_type());
    const int64_t rows = ids.numel(), hidden = embed.size(1);
    need(hidden < (1 << 30));
    const at::Tensor h = empty({T, rows, hidden}, embed.scalar_type(), embed), x = at::empty_like(h);
    void *const stream = stream_of(embed);
    THPObjectPtr done = pair(h, x);
    launch("embed_rmsnorm", embed_fn, static_cast<const int64_t *>(ids.data_ptr()), embed.data_ptr(), embed.size(0),
           w.data_ptr(), h.data_ptr(), x.data_ptr(), code, T, rows, static_cast<int>(hidden), eps, stream);
    return done.release();
  });
}

// add_rmsnorm(h, delta|None, weight, eps, out|None) -> out
PyObject *add_rmsnorm(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded(n, 5, [&]() -> PyObject * {
    const at::Tensor &h = tensor(a[0]);
    need(h.is_contiguous() && h.dim() >= 1 && h.numel() > 0);
    const int code = float_code(h.scalar_type());
    const at::Tensor *delta = a[1] == Py_None ? nullptr : &alike(a[1], h);
    need(!delta || delta->sizes() == h.sizes());
    const at::Tensor &w = alike(a[2], h);
    const int64_t hidden = h.size(-1);
    need(w.numel() == hidden && hidden < (1 << 30));
    const float eps = real(a[3]);
    at::Tensor out;
    if (a[4] == Py_None) out = at::empty_like(h);
    else out = alike(a[4], h);
    need(out.numel() == h.numel());
    void *const stream = stream_of(h);
    THPObjectPtr done = result(a[4], out);
    launch("add_rmsnorm", add_norm_fn, h.data_ptr(),
           delta ? delta->data_ptr() : nullptr, w.data_ptr(), out.data_ptr(), code, h.numel() / hidden,
           static_cast<int>(hidden), eps, stream);
    return done.release();
  });
}

// rmsnorm_mean_t(h, weight, eps, delta|None) -> out
PyObject *rmsnorm_mean_t(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded(n, 4, [&]() -> PyObject * {
    const at::Tensor &h = tensor(a[0]);
    need(h.is_contiguous() && h.dim() == 3 && h.numel() > 0);
    const int code = float_code(h.scalar_type());
    const at::Tensor &w = alike(a[1], h);
    const float eps = real(a[2]);
    const at::Tensor *delta = a[3] == Py_None ? nullptr : &alike(a[3], h);
    need((!delta || delta->sizes() == h.sizes()) && w.numel() == h.size(2) && h.size(0) <= 8 && h.size(2) < (1 << 30));
    const at::Tensor out = empty({h.size(1), h.size(2)}, h.scalar_type(), h);
    void *const stream = stream_of(h);
    THPObjectPtr done = result(Py_None, out);
    launch("rmsnorm_mean_t", mean_fn, h.data_ptr(),
           delta ? delta->data_ptr() : nullptr, w.data_ptr(), out.data_ptr(), code, static_cast<int>(h.size(0)),
           h.size(1), static_cast<int>(h.size(2)), eps, stream);
    return done.release();
  });
}

// lif_gate_mul(gate_up, beta, threshold) -> out
PyObject *lif_gate_mul(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded(n, 3, [&]() -> PyObject * {
    const at::Tensor &x = tensor(a[0]);
    need(x.dim() == 3 && x.numel() > 0 && x.stride(2) == 1 && x.size(2) % 2 == 0 && x.size(0) < (1 << 20) &&
         x.size(2) < (1 << 30));
    const int64_t I = x.size(2) / 2;
    const at::Tensor &beta = vector(a[1], I, x), &th = vector(a[2], I, x);
    need(beta.scalar_type() == th.scalar_type());
    const int code = float_code(x.scalar_type()), pc = float_code(beta.scalar_type());
    const at::Tensor out = empty({x.size(0), x.size(1), I}, x.scalar_type(), x);
    const int64_t strides[2] = {x.stride(0), x.stride(1)};
    void *const stream = stream_of(x);
    THPObjectPtr done = result(Py_None, out);
    launch("lif_gate_mul", gate_mul_fn, x.data_ptr(), code, strides, beta.data_ptr(), th.data_ptr(), pc, out.data_ptr(),
           static_cast<int>(x.size(0)), x.size(1), static_cast<int>(I), stream);
    return done.release();
  });
}

// linear_decode(x, w_packed, bias|None, out|None) -> y
PyObject *linear_decode(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded(n, 4, [&]() -> PyObject * {
    const at::Tensor &x = tensor(a[0]);
    need(x.scalar_type() == at::kBFloat16 && x.is_contiguous() && x.dim() >= 1 && x.numel() > 0);
    const at::Tensor &w = alike(a[1], x);
    need(w.dim() == 2 && w.size(1) == x.size(-1) && w.size(0) < (1 << 30) && w.size(1) < (1 << 30));
    const at::Tensor *bias = a[2] == Py_None ? nullptr : &alike(a[2], x);
    const int64_t N = w.size(0), K = w.size(1), M = x.numel() / K;
    need((!bias || bias->numel() == N) && M < (1 << 30));
    at::Tensor y;
    if (a[3] == Py_None) {
      c10::SmallVector<int64_t, 6> shape(x.sizes().begin(), x.sizes().end());
      shape.back() = N;
      y = empty(shape, x.scalar_type(), x);
    } else {
      y = alike(a[3], x);
      need(y.dim() >= 1 && y.size(-1) == N && y.numel() == M * N);
    }
    void *const stream = stream_of(x);
    THPObjectPtr done = result(a[3], y);
    launch("linear_decode", linear_fn, x.data_ptr(), w.data_ptr(),
           bias ? bias->data_ptr() : nullptr, y.data_ptr(), static_cast<int>(M),
           static_cast<int>(N), static_cast<int>(K), SPK_BF16, stream);
    return done.release();
  });
}

// mlp_gate_lif(x, w_packed, beta, threshold) -> y
PyObject *mlp_gate_lif(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded(n, 4, [&]() -> PyObject * {
    const at::Tensor &x = tensor(a[0]);
    need(x.scalar_type() == at::kBFloat16 && x.is_contiguous() && x.dim() == 3 && x.numel() > 0);
    const at::Tensor &w = alike(a[1], x);
    const at::Tensor &beta = tensor(a[2]);
    const int64_t I = beta.numel(), hidden = x.size(2);
    need(beta.scalar_type() == at::kFloat && beta.is_contiguous() && beta.device() == x.device());
    const at::Tensor &th = vector(a[3], I, x);
    need(th.scalar_type() == at::kFloat && I < (1 << 28) && hidden < (1 << 28) && w.numel() == 2 * I * hidden &&
         x.size(0) < (1 << 20) && x.size(1) < (1 << 28));
    const at::Tensor y = empty({x.size(0), x.size(1), I}, x.scalar_type(), x);
    void *const stream = stream_of(x);
    THPObjectPtr done = result(Py_None, y);
    launch("mlp_gate_lif", mlp_gate_fn, x.data_ptr(), w.data_ptr(), beta.data_ptr(), th.data_ptr(), SPK_F32,
           y.data_ptr(), static_cast<int>(x.size(0)), static_cast<int>(x.size(1)), static_cast<int>(hidden),
           static_cast<int>(I), SPK_BF16, stream);
    return done.release();
  });
}

// qkv_rope_lif_pack(qkv, cos, sin, beta, threshold, k_cache, v_cache, slots, Hq, Hkv, D, q_packed|None, n_q,
//                   positions, k_packed|None, v_packed|None) -> True; no dense outputs
PyObject *qkv_rope_lif_pack(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded(n, 16, [&]() -> PyObject * {
    const at::Tensor &x = tensor(a[0]);
    need(x.dim() == 3 && x.stride(2) == 1 && x.numel() > 0 && x.size(0) < (1 << 20));
    const int code = float_code(x.scalar_type());
    const at::Tensor &cos = alike(a[1], x), &sin = alike(a[2], x);
    const at::Tensor &k = tensor(a[5]), &v = tensor(a[6]);
    const int Hq = int32(a[8]), Hkv = int32(a[9]), D = int32(a[10]);
    need(Hq > 0 && Hkv > 0 && D >= 32 && D % 32 == 0 && D <= 1024 && Hq < (1 << 16) && Hkv < (1 << 16));
    const at::Tensor &beta = vector(a[3], 3 * D, x), &th = vector(a[4], 3 * D, x);
    need(beta.scalar_type() == th.scalar_type());
    const int64_t T = x.size(0), n_tok = x.size(1);
    need(x.size(2) == static_cast<int64_t>(Hq + 2 * Hkv) * D && packed4(k) && packed4(v) && k.sizes() == v.sizes() &&
         k.strides() == v.strides() && k.size(0) == T && k.size(1) == Hkv && k.size(3) == D / 32 &&
         k.device() == x.device() && v.device() == x.device());
    need(cos.dim() == 2 && sin.dim() == 2 && cos.sizes() == sin.sizes() && cos.size(1) == D && cos.size(0) >= 1);
    const at::Tensor &slots = tensor(a[7]), &pos = tensor(a[13]);
    need(slots.scalar_type() == at::kLong && slots.is_contiguous() && slots.numel() >= n_tok &&
         slots.device() == x.device() && pos.scalar_type() == at::kLong && pos.is_contiguous() &&
         pos.numel() >= n_tok && pos.device() == x.device());
    const int64_t n_q = integer(a[12]);
    need(n_q >= 0 && n_q <= n_tok);
    const at::Tensor *q = a[11] == Py_None ? nullptr : &tensor(a[11]);
    int64_t qs[3] = {0, 0, 0};
    if (q) {
      need(packed4(*q) && q->size(0) == T && q->size(1) >= n_q && q->size(2) == Hq && q->size(3) == D / 32 &&
           q->device() == x.device());
      for (int i = 0; i < 3; ++i) qs[i] = q->stride(i);
    }
    need(q || n_q == 0);
    const at::Tensor *own[2] = {nullptr, nullptr};
    need((a[14] == Py_None) == (a[15] == Py_None));
    for (int i = 0; i < 2 && a[14] != Py_None; ++i) {
      own[i] = &tensor(a[14 + i]);
      need(packed4(*own[i]) && own[i]->is_contiguous() && own[i]->size(0) == T && own[i]->size(1) == n_tok &&
           own[i]->size(2) == Hkv && own[i]->size(3) == D / 32 && own[i]->device() == x.device());
    }
    const int64_t xs[2] = {x.stride(0), x.stride(1)}, cs[3] = {k.stride(0), k.stride(1), k.stride(2)};
    const int pc = float_code(beta.scalar_type());
    void *const stream = stream_of(x);
    auto words = [](const at::Tensor *t) { return t ? static_cast<int32_t *>(t->data_ptr()) : nullptr; };
    launch("qkv_rope_lif_pack", qkv_fn, x.data_ptr(), code, xs, cos.data_ptr(), sin.data_ptr(),
           static_cast<const int64_t *>(pos.data_ptr()), cos.size(0), beta.data_ptr(), th.data_ptr(), pc, words(q), qs,
           n_q, words(&k), words(&v), cs, static_cast<const int64_t *>(slots.data_ptr()), k.size(2), words(own[0]),
           words(own[1]), nullptr, nullptr, nullptr, static_cast<int>(T), n_tok, Hq, Hkv, D, stream);
    Py_RETURN_TRUE;
  });
}

template <class F> void set(F &f, void *p) { f = reinterpret_cast<F>(p); }

// bind(device, addresses): "cuda" or "cpu", and the C ABI's functions in the order of
// the declarations above.
PyObject *bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
  constexpr int kFns = 13;
  if (n != kFns + 1 || !PyUnicode_Check(a[0])) {
    PyErr_Format(PyExc_TypeError, "bind takes a device type and %d addresses", kFns);
    return nullptr;
  }
  taken_on = PyUnicode_CompareWithASCIIString(a[0], "cpu") == 0 ? at::kCPU : at::kCUDA;
  ++a;
  void *p[kFns];
  for (int i = 0; i < kFns; ++i) {
    p[i] = PyLong_AsVoidPtr(a[i]);
    if (!p[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
      return nullptr;
    }
  }
  set(decode_attn_fn, p[0]);
  set(workspace_fn, p[1]);
  set(lif_sites_fn, p[2]);
  set(lif_fn, p[3]);
  set(prefill_fn, p[4]);
  set(embed_fn, p[5]);
  set(add_norm_fn, p[6]);
  set(mean_fn, p[7]);
  set(gate_mul_fn, p[8]);
  set(linear_fn, p[9]);
  set(mlp_gate_fn, p[10]);
  set(qkv_fn, p[11]);
  set(last_error_fn, p[12]);
  Py_RETURN_NONE;
}

#define SPK_METHOD(name) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    SPK_METHOD(bind),          SPK_METHOD(decode_attn),       SPK_METHOD(lif_sites),    SPK_METHOD(lif),
    SPK_METHOD(prefill),       SPK_METHOD(embed_rmsnorm),     SPK_METHOD(add_rmsnorm),  SPK_METHOD(rmsnorm_mean_t),
    SPK_METHOD(lif_gate_mul),  SPK_METHOD(linear_decode),     SPK_METHOD(mlp_gate_lif), SPK_METHOD(qkv_rope_lif_pack),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// The module carries what it was compiled for: the addresses that bind() takes are
// called by this version of the C ABI, and tensors are read by this torch's layout.
PyMODINIT_FUNC PyInit__native() {
  THPObjectPtr m(PyModule_Create(&module));
  if (!m || PyModule_AddIntConstant(m.get(), "abi_version", SPK_ABI_VERSION) ||
      PyModule_AddStringConstant(m.get(), "built_for", SPK_TORCH_VERSION))
    return nullptr;
  return m.release();
}
