// binding.cpp -- the plain calls of the package without Python between the
// caller and the C ABI: codec, fold and cast over ordinary GPU tensors, the
// optimizer step's checks and descriptor tables, and the gradient clip.
//
// Every function takes the Python objects as the caller has them and either
// does the whole call or returns None before any effect.  None means "not a
// plain call": another type of tensor, a transform or mode in force, a
// layout, dtype or device the kernels do not take as it is, or a refusal of
// the library.  The Python code behind it then runs as if this file did not
// exist, with its copies, checks and messages.
//
// What it buys on the host, against Python and ctypes, in us a call (tensors of
// a few KB, the GPU not waited for): quantize 15.2 -> 4.9, dequantize 10.3 ->
// 4.3, roundtrip 12.0 -> 4.2, cast 9.2 -> 4.4, fold 7.5 -> 3.4; the clipped step
// of 38 tensors 104 -> 19, the folded one of 1,100 2,242 -> 156; the clip of 38
// 55 -> 14, of 1,100 782 -> 59.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include "../../include/ely.h"

namespace {

using at::Tensor;

// An ordinary GPU or CPU tensor: nothing but these keys (no Python subclass
// behaviour, transform wrapper, functionalization, negative or zero bit).
const c10::DispatchKeySet kPlainKeys({c10::DispatchKey::CUDA, c10::DispatchKey::CPU, c10::DispatchKey::AutogradCUDA,
                                      c10::DispatchKey::AutogradCPU, c10::DispatchKey::ADInplaceOrView,
                                      c10::DispatchKey::AutocastCUDA, c10::DispatchKey::AutocastCPU});

// No key and no backend of `ks` outside `allowed` (the set's own difference
// keeps backends).
bool within(c10::DispatchKeySet ks, c10::DispatchKeySet allowed) { return (ks.raw_repr() & ~allowed.raw_repr()) == 0; }

bool plain_tensor(const Tensor& t) { return t.defined() && within(t.key_set(), kPlainKeys) && t.layout() == at::kStrided; }

// No torch function or dispatch mode, transform or trace in force.
bool plain_state() {
    if (at::impl::torch_function_mode_enabled()) return false;
    return within(c10::impl::tls_local_dispatch_key_set().included_, c10::default_included_set | c10::autocast_dispatch_keyset);
}

// The tensor of a Python object that is exactly a torch.Tensor or Parameter.
const Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const Tensor& t = THPVariable_Unpack(o);
    return plain_tensor(t) ? &t : nullptr;
}

int dtype_code(const Tensor& t) {
    const auto s = t.scalar_type();
    return s == at::kFloat ? ELY_F32 : s == at::kBFloat16 ? ELY_BF16 : -1;
}

// ... and it is contiguous fp32 or bf16 on a GPU.
const Tensor* kernel_tensor(PyObject* o) {
    const Tensor* t = plain(o);
    return t && t->is_cuda() && dtype_code(*t) >= 0 && t->is_contiguous() ? t : nullptr;
}

void* stream_of(c10::DeviceIndex dev) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev).stream(); }

// Scratch buffers, one per device and stream: calls on one stream are
// ordered, so reuse is safe; when one grows, the old buffer returns to
// torch's allocator, which reuses it only after work already queued on that
// stream.  The map is never destroyed: the GPU runtime ends before static
// objects do.  Nothing is allocated or freed under the mutex: the allocator
// may run Python (a memory trace) and so let another thread go on to wait
// for the mutex with the interpreter lock held.
std::mutex g_ws_mu;
std::map<std::pair<int, void*>, Tensor>& workspaces() {
    static auto* m = new std::map<std::pair<int, void*>, Tensor>();
    return *m;
}

Tensor workspace(c10::DeviceIndex dev, int64_t nbytes) {
    nbytes = std::max<int64_t>(nbytes, 256);
    const std::pair<int, void*> key(dev, stream_of(dev));
    {
        std::lock_guard<std::mutex> lk(g_ws_mu);
        const auto it = workspaces().find(key);
        if (it != workspaces().end() && it->second.numel() >= nbytes) return it->second;
    }
    const Tensor buf = at::empty({std::max<int64_t>(nbytes, 1 << 20)},
                                 at::TensorOptions().dtype(at::kByte).device(c10::Device(at::kCUDA, dev)));
    Tensor old;  // outlives the lock
    std::lock_guard<std::mutex> lk(g_ws_mu);
    Tensor& kept = workspaces()[key];
    if (!kept.defined() || kept.numel() < buf.numel()) {
        old = std::move(kept);
        kept = buf;
    }
    return buf;
}

// The library call without the interpreter lock: it may wait for a slot of
// the table ring.
template <class F>
int unlocked(F f) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    return rc;
}

int fmt_code(PyObject* o) {
    if (!PyUnicode_Check(o)) return -1;
    if (PyUnicode_CompareWithASCIIString(o, "e4m3") == 0) return ELY_E4M3;
    if (PyUnicode_CompareWithASCIIString(o, "e5m2") == 0) return ELY_E5M2;
    return -1;
}

at::ScalarType fp8_type(int fmt) { return fmt == ELY_E4M3 ? at::kFloat8_e4m3fn : at::kFloat8_e5m2; }

// x's rows and columns (per_tensor: one row); false for shapes left to Python.
bool rows_of(const Tensor& x, bool per_tensor, int64_t& rows, int64_t& cols) {
    if (x.dim() == 0 || x.numel() == 0) return false;
    cols = per_tensor ? x.numel() : x.size(-1);
    rows = x.numel() / cols;
    return true;
}

std::vector<int64_t> k_shape(const Tensor& x, bool per_tensor) {
    std::vector<int64_t> s(x.sizes().begin(), x.sizes().end());
    if (per_tensor) std::fill(s.begin(), s.end(), 1);
    s.back() = 1;
    return s;
}

// workspace_(dev): PyObject* (device index, nbytes) -> the uint8 buffer.
PyObject* py_workspace(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 2) return PyErr_Format(PyExc_TypeError, "workspace takes a device index and a size");
    const long dev = PyLong_AsLong(a[0]);
    const long long nbytes = PyLong_AsLongLong(a[1]);
    if (PyErr_Occurred()) return nullptr;
    return THPVariable_Wrap(workspace((c10::DeviceIndex)dev, nbytes));
    END_HANDLE_TH_ERRORS
}

// quantize(x, fmt, per_tensor) -> (q, k) or None.
PyObject* py_quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3) Py_RETURN_NONE;
    const Tensor* x = kernel_tensor(a[0]);
    const int fmt = fmt_code(a[1]);
    const bool per_tensor = a[2] == Py_True;
    int64_t rows, cols;
    if (!x || fmt < 0 || (!per_tensor && a[2] != Py_False) || !plain_state() || !rows_of(*x, per_tensor, rows, cols)) Py_RETURN_NONE;
    const auto dev = x->device();
    const int dt = dtype_code(*x);
    Tensor q = at::empty(x->sizes(), at::TensorOptions().dtype(fp8_type(fmt)).device(dev));
    Tensor k = at::empty(k_shape(*x, per_tensor), at::TensorOptions().dtype(at::kInt).device(dev));
    Tensor ws = workspace(dev.index(), ely_fp8_workspace_bytes(rows, cols, dt));
    const void* xp = x->const_data_ptr();
    uint8_t* qp = static_cast<uint8_t*>(q.mutable_data_ptr());
    int32_t* kp = static_cast<int32_t*>(k.mutable_data_ptr());
    void* wp = ws.mutable_data_ptr();
    const int64_t wn = ws.numel();
    void* s = stream_of(dev.index());
    if (unlocked([&] { return ely_fp8_quantize(xp, dt, rows, cols, fmt, qp, kp, wp, wn, s); }) != ELY_OK) Py_RETURN_NONE;
    PyObject* out = PyTuple_New(2);
    if (!out) return nullptr;
    PyTuple_SET_ITEM(out, 0, THPVariable_Wrap(std::move(q)));
    PyTuple_SET_ITEM(out, 1, THPVariable_Wrap(std::move(k)));
    return out;
    END_HANDLE_TH_ERRORS
}

// roundtrip(x, fmt, per_tensor) -> out or None.
PyObject* py_roundtrip(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3) Py_RETURN_NONE;
    const Tensor* x = kernel_tensor(a[0]);
    const int fmt = fmt_code(a[1]);
    const bool per_tensor = a[2] == Py_True;
    int64_t rows, cols;
    if (!x || fmt < 0 || (!per_tensor && a[2] != Py_False) || !plain_state() || !rows_of(*x, per_tensor, rows, cols)) Py_RETURN_NONE;
    const auto dev = x->device();
    const int dt = dtype_code(*x);
    Tensor out = at::empty(x->sizes(), at::TensorOptions().dtype(x->scalar_type()).device(dev));
    Tensor ws = workspace(dev.index(), ely_fp8_workspace_bytes(rows, cols, dt));
    const void* xp = x->const_data_ptr();
    void* op = out.mutable_data_ptr();
    void* wp = ws.mutable_data_ptr();
    const int64_t wn = ws.numel();
    void* s = stream_of(dev.index());
    if (unlocked([&] { return ely_fp8_roundtrip(xp, dt, rows, cols, fmt, op, nullptr, nullptr, wp, wn, s); }) != ELY_OK)
        Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// dequantize(q, k, bf16) -> out (bf16, else fp32) or None.
PyObject* py_dequantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3) Py_RETURN_NONE;
    const Tensor* q = plain(a[0]);
    const Tensor* k = plain(a[1]);
    if (!q || !k || !q->is_cuda() || k->device() != q->device() || !q->is_contiguous() || !k->is_contiguous() ||
        k->scalar_type() != at::kInt || !plain_state())
        Py_RETURN_NONE;
    const int fmt = q->scalar_type() == at::kFloat8_e4m3fn ? ELY_E4M3 : q->scalar_type() == at::kFloat8_e5m2 ? ELY_E5M2 : -1;
    int64_t rows, cols;
    if (fmt < 0 || !rows_of(*q, false, rows, cols)) Py_RETURN_NONE;
    if (k->numel() == 1 && rows != 1) {  // a per-tensor exponent: one row of every element
        cols = q->numel();
        rows = 1;
    }
    if (k->numel() != rows) Py_RETURN_NONE;
    const bool bf16 = a[2] == Py_True;
    const auto dev = q->device();
    Tensor out = at::empty(q->sizes(), at::TensorOptions().dtype(bf16 ? at::kBFloat16 : at::kFloat).device(dev));
    const uint8_t* qp = static_cast<const uint8_t*>(q->const_data_ptr());
    const int32_t* kp = static_cast<const int32_t*>(k->const_data_ptr());
    void* op = out.mutable_data_ptr();
    void* s = stream_of(dev.index());
    if (unlocked([&] { return ely_fp8_dequantize(qp, kp, rows, cols, fmt, op, bf16 ? ELY_BF16 : ELY_F32, s); }) != ELY_OK)
        Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// cast_bf16(x) (fp32 -> bf16) and widen_bf16(x) (bf16 -> fp32): a new tensor or None.
template <bool WIDEN>
PyObject* py_convert(PyObject*, PyObject* o) {
    HANDLE_TH_ERRORS
    const Tensor* x = kernel_tensor(o);
    if (!x || x->scalar_type() != (WIDEN ? at::kBFloat16 : at::kFloat) || !plain_state()) Py_RETURN_NONE;
    const auto dev = x->device();
    Tensor out = at::empty(x->sizes(), at::TensorOptions().dtype(WIDEN ? at::kFloat : at::kBFloat16).device(dev));
    const void* xp = x->const_data_ptr();
    void* op = out.mutable_data_ptr();
    const int64_t ne = x->numel();
    void* s = stream_of(dev.index());
    const int rc = unlocked([&] {
        return WIDEN ? ely_widen_bf16(static_cast<const uint16_t*>(xp), static_cast<float*>(op), ne, s)
                     : ely_cast_bf16(static_cast<const float*>(xp), static_cast<uint16_t*>(op), ne, s);
    });
    if (rc != ELY_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// fold_add(acc, g): True when acc += g was issued, else None.
PyObject* py_fold_add(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 2) Py_RETURN_NONE;
    const Tensor* acc = kernel_tensor(a[0]);
    const Tensor* g = kernel_tensor(a[1]);
    if (!acc || !g || g->numel() != acc->numel() || g->device() != acc->device() || !plain_state()) Py_RETURN_NONE;
    void* ap = acc->mutable_data_ptr();
    const void* gp = g->const_data_ptr();
    const int dt = dtype_code(*g);
    const bool wide = acc->scalar_type() == at::kFloat;
    const int64_t ne = acc->numel();
    void* s = stream_of(acc->device().index());
    const int rc = unlocked([&] {
        return wide ? ely_fold_add(static_cast<float*>(ap), gp, dt, ne, s) : ely_fold_add_bf16(static_cast<uint16_t*>(ap), gp, dt, ne, s);
    });
    if (rc != ELY_OK) Py_RETURN_NONE;
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// A tensor that the call only reads, and one that it writes: of a lazy copy
// the latter is given memory of its own first, as Tensor.data_ptr() does.
ely_tensor entry(const Tensor& t) {
    return ely_tensor{const_cast<void*>(t.const_data_ptr()), t.numel(), dtype_code(t), 0};
}
ely_tensor written(const Tensor& t) { return ely_tensor{t.mutable_data_ptr(), t.numel(), dtype_code(t), 0}; }

// References to the objects whose memory a call's tables name, held until its
// launches are queued: the caller's lists and the state may change meanwhile, in
// consts() or in another thread while the interpreter lock is released.
class Held {
public:
    Held() = default;
    Held(const Held&) = delete;
    Held& operator=(const Held&) = delete;
    ~Held() {
        for (PyObject* o : objects_) Py_DECREF(o);
    }
    void reserve(size_t n) { objects_.reserve(n); }
    PyObject* add(PyObject* o) {
        objects_.push_back(o);
        Py_INCREF(o);
        return o;
    }

private:
    std::vector<PyObject*> objects_;
};

// Fails of adamw_step and clip that the library reported: (status, which call).
PyObject* status(int rc, int which) { return Py_BuildValue("(ii)", rc, which); }

// adamw_step(params, grads, accs, state, steps, copies, device, order, wd,
// max_norm, norm, consts) -> (status, which call) of the step over every
// parameter with a gradient, or None.  All lists are aligned with params;
// accs and copies may be None; state maps a parameter's index to its entry;
// steps is the flat fp32 step counters; max_norm None means no clipping, else
// norm is the 16-byte result buffer; consts(t) gives the 8 constants of step t.
PyObject* py_adamw_step(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 12) Py_RETURN_NONE;
    PyObject *params = a[0], *grads = a[1], *accs = a[2], *state = a[3], *copies = a[5];
    if (!PyList_CheckExact(params) || !PyList_CheckExact(grads) || !PyDict_CheckExact(state) || !plain_state()) Py_RETURN_NONE;
    const bool fold = accs != Py_None, copy = copies != Py_None;
    const Py_ssize_t n = PyList_GET_SIZE(params);
    if (PyList_GET_SIZE(grads) != n || (fold && (!PyList_CheckExact(accs) || PyList_GET_SIZE(accs) != n)) ||
        (copy && (!PyList_CheckExact(copies) || PyList_GET_SIZE(copies) != n)) || n > INT32_MAX)
        Py_RETURN_NONE;
    const Tensor* steps = plain(a[4]);
    if (!steps || !steps->is_cpu() || steps->scalar_type() != at::kFloat || !steps->is_contiguous() || steps->numel() < n)
        Py_RETURN_NONE;
    const long dev = PyLong_AsLong(a[6]), order = PyLong_AsLong(a[7]), wd = PyLong_AsLong(a[8]);
    const bool clip = a[9] != Py_None;
    const double max_norm = clip ? PyFloat_AsDouble(a[9]) : 0.0;
    if (PyErr_Occurred()) return nullptr;
    const Tensor* norm = clip ? plain(a[10]) : nullptr;
    if (clip && (!norm || !norm->is_cuda() || norm->get_device() != dev || norm->nbytes() < sizeof(ely_norm_result))) Py_RETURN_NONE;

    static PyObject* k_m = PyUnicode_InternFromString("exp_avg");
    static PyObject* k_v = PyUnicode_InternFromString("exp_avg_sq");
    Held held;
    held.reserve((size_t)n * 6);
    std::vector<ely_tensor> P, G, A, M, V, C;
    std::vector<Py_ssize_t> idx;
    for (auto* v : {&P, &G, &M, &V, &C}) v->reserve(n);
    if (fold) A.reserve(n);
    idx.reserve(n);
    int64_t n_bf16 = 0;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* go = PyList_GET_ITEM(grads, i);
        if (go == Py_None) continue;
        const Tensor *p = kernel_tensor(held.add(PyList_GET_ITEM(params, i))), *g = kernel_tensor(held.add(go));
        if (!p || !g || p->scalar_type() != at::kFloat || p->get_device() != dev || g->get_device() != dev || g->sizes() != p->sizes())
            Py_RETURN_NONE;
        if (fold) {
            const Tensor* ac = kernel_tensor(held.add(PyList_GET_ITEM(accs, i)));
            if (!ac || ac->scalar_type() != at::kFloat || ac->get_device() != dev || ac->sizes() != p->sizes()) Py_RETURN_NONE;
            A.push_back(entry(*ac));
        }
        PyObject* key = PyLong_FromSsize_t(i);
        if (!key) return nullptr;
        PyObject* st = PyDict_GetItemWithError(state, key);  // borrowed
        Py_DECREF(key);
        if (!st && PyErr_Occurred()) return nullptr;
        if (!st || !PyDict_CheckExact(st)) Py_RETURN_NONE;
        PyObject *mo = PyDict_GetItem(st, k_m), *vo = PyDict_GetItem(st, k_v);
        const Tensor *m = mo ? kernel_tensor(held.add(mo)) : nullptr, *v = vo ? kernel_tensor(held.add(vo)) : nullptr;
        if (!m || !v || m->scalar_type() != at::kFloat || v->scalar_type() != at::kFloat) Py_RETURN_NONE;
        PyObject* co = copy ? PyList_GET_ITEM(copies, i) : Py_None;
        if (co == Py_None) {
            C.push_back(ely_tensor{nullptr, 0, ELY_BF16, 0});
        } else {
            const Tensor* c = kernel_tensor(held.add(co));
            if (!c) Py_RETURN_NONE;
            C.push_back(written(*c));
        }
        P.push_back(written(*p));
        G.push_back(entry(*g));
        M.push_back(written(*m));
        V.push_back(written(*v));
        idx.push_back(i);
        n_bf16 += g->scalar_type() == at::kBFloat16;
    }
    if (idx.empty() || c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().device_index() != dev)
        Py_RETURN_NONE;  // nothing to step, or another device is current

    // the plain call stands: from here on it has effects
    float* sp = static_cast<float*>(steps->mutable_data_ptr());
    std::vector<std::pair<float, ely_adamw_consts>> by_step;  // almost always one
    std::vector<ely_adamw_consts> consts(idx.size());
    for (Py_ssize_t i : idx) sp[i] += 1.0f;
    for (size_t j = 0; j < idx.size(); ++j) {
        const float t = sp[idx[j]];
        size_t h = 0;
        while (h < by_step.size() && by_step[h].first != t) ++h;
        if (h == by_step.size()) {
            PyObject* tf = PyFloat_FromDouble(t);
            PyObject* row = tf ? PyObject_CallOneArg(a[11], tf) : nullptr;
            Py_XDECREF(tf);
            if (!row) return nullptr;
            ely_adamw_consts c;
            std::memset(&c, 0, sizeof c);
            float* f = reinterpret_cast<float*>(&c);
            const bool ok = PyList_CheckExact(row) && PyList_GET_SIZE(row) * sizeof(float) <= sizeof c;
            for (Py_ssize_t k = 0; ok && k < PyList_GET_SIZE(row); ++k) f[k] = (float)PyFloat_AsDouble(PyList_GET_ITEM(row, k));
            Py_DECREF(row);
            if (!ok) return PyErr_Format(PyExc_TypeError, "the constants of a step are a list of at most 8 floats");
            if (PyErr_Occurred()) return nullptr;
            by_step.emplace_back(t, c);
        }
        consts[j] = by_step[h].second;
    }

    void* s = stream_of((c10::DeviceIndex)dev);
    const float* coef = nullptr;
    const int32_t ns = (int32_t)idx.size();
    if (clip) {
        ely_norm_result* res = static_cast<ely_norm_result*>(norm->mutable_data_ptr());
        Tensor ws = workspace((c10::DeviceIndex)dev, ely_grad_norm_workspace_bytes(G.data(), ns));
        void* wp = ws.mutable_data_ptr();
        const int64_t wn = ws.numel();
        const int rc = unlocked([&] {
            return fold ? ely_grad_norm_fold(A.data(), G.data(), ns, (float)max_norm, res, wp, wn, s)
                        : ely_grad_norm(G.data(), ns, (float)max_norm, res, wp, wn, s);
        });
        if (rc != ELY_OK) return status(rc, 0);
        coef = &res->coef;
    }
    // one launch per gradient dtype, bf16 first
    auto launch = [&](const std::vector<ely_tensor>& p, const std::vector<ely_tensor>& ac, const std::vector<ely_tensor>& g,
                      const std::vector<ely_tensor>& m, const std::vector<ely_tensor>& v, const std::vector<ely_tensor>& c,
                      const std::vector<ely_adamw_consts>& k) {
        const int32_t nl = (int32_t)p.size();
        Tensor ws = workspace((c10::DeviceIndex)dev, ely_adamw_workspace_bytes(nl));
        void* wp = ws.mutable_data_ptr();
        const int64_t wn = ws.numel();
        return unlocked([&] {
            return fold ? ely_adamw_fold_step(p.data(), ac.data(), g.data(), m.data(), v.data(), c.data(), nl, k.data(), (int32_t)order,
                                              (int32_t)wd, coef, wp, wn, s)
                        : ely_adamw_step(p.data(), g.data(), m.data(), v.data(), c.data(), nl, k.data(), (int32_t)order, (int32_t)wd,
                                         coef, wp, wn, s);
        });
    };
    if (n_bf16 == 0 || n_bf16 == ns) return status(launch(P, A, G, M, V, C, consts), 1);
    for (int32_t want : {ELY_BF16, ELY_F32}) {
        auto pick = [&](const std::vector<ely_tensor>& from) {
            std::vector<ely_tensor> out;
            for (size_t j = 0; j < from.size(); ++j)
                if (G[j].dtype == want) out.push_back(from[j]);
            return out;
        };
        std::vector<ely_adamw_consts> k;
        for (size_t j = 0; j < consts.size(); ++j)
            if (G[j].dtype == want) k.push_back(consts[j]);
        const int rc = launch(pick(P), pick(A), pick(G), pick(M), pick(V), pick(C), k);
        if (rc != ELY_OK) return status(rc, 1);
    }
    return status(ELY_OK, 1);
    END_HANDLE_TH_ERRORS
}

// clip(params, max_norm) -> the total norm (0-d fp32) after scaling every
// gradient of the list in place, or None.
PyObject* py_clip(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 2 || !(PyList_CheckExact(a[0]) || PyTuple_CheckExact(a[0])) || !plain_state()) Py_RETURN_NONE;
    const double max_norm = PyFloat_AsDouble(a[1]);
    if (PyErr_Occurred()) {
        PyErr_Clear();  // Python's own float() says what is wrong with it
        Py_RETURN_NONE;
    }
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(a[0]);
    // the gradients themselves: .grad may be cleared while the interpreter lock is released
    std::vector<Tensor> held;
    std::vector<ely_tensor> G;
    held.reserve(n);
    G.reserve(n);
    c10::DeviceIndex dev = -1;
    for (Py_ssize_t i = 0; i < n; ++i) {
        const Tensor* p = plain(PySequence_Fast_GET_ITEM(a[0], i));
        if (!p || !p->is_leaf()) Py_RETURN_NONE;
        const Tensor& g = p->grad();
        if (!g.defined()) continue;
        if (!plain_tensor(g) || !g.is_cuda() || !g.is_contiguous() || dtype_code(g) < 0) Py_RETURN_NONE;
        if (dev < 0) dev = (c10::DeviceIndex)g.get_device();
        if (g.get_device() != dev) Py_RETURN_NONE;
        G.push_back(written(g));
        held.push_back(g);
    }
    if (G.empty() || G.size() > INT32_MAX || c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().device_index() != dev) Py_RETURN_NONE;
    const int32_t ns = (int32_t)G.size();
    static_assert(sizeof(ely_norm_result) == 16, "the norm result is four words: sumsq, norm, coef");
    Tensor res = at::empty({4}, at::TensorOptions().dtype(at::kFloat).device(c10::Device(at::kCUDA, dev)));
    ely_norm_result* rp = static_cast<ely_norm_result*>(res.mutable_data_ptr());
    Tensor ws = workspace(dev, ely_grad_norm_workspace_bytes(G.data(), ns));
    void* wp = ws.mutable_data_ptr();
    const int64_t wn = ws.numel();
    void* s = stream_of(dev);
    if (unlocked([&] { return ely_grad_norm_clip(G.data(), ns, (float)max_norm, rp, wp, wn, s); }) != ELY_OK) Py_RETURN_NONE;
    // a tensor of its own over the result's memory: as a view of it, detach_() would be refused
    Tensor total = at::empty({0}, res.options());
    total.set_(res.storage(), 2, {}, {});
    return THPVariable_Wrap(std::move(total));
    END_HANDLE_TH_ERRORS
}

// abi_version(): of the library that these calls run in.
PyObject* py_abi_version(PyObject*, PyObject*) { return PyLong_FromLong(ely_abi_version()); }

#define FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f)), METH_FASTCALL
PyMethodDef kMethods[] = {
    {"abi_version", py_abi_version, METH_NOARGS, "abi_version()"},
    {"workspace", FAST(py_workspace), "workspace(device index, nbytes)"},
    {"quantize", FAST(py_quantize), "quantize(x, fmt, per_tensor)"},
    {"roundtrip", FAST(py_roundtrip), "roundtrip(x, fmt, per_tensor)"},
    {"dequantize", FAST(py_dequantize), "dequantize(q, k, bf16)"},
    {"cast_bf16", py_convert<false>, METH_O, "cast_bf16(x)"},
    {"widen_bf16", py_convert<true>, METH_O, "widen_bf16(x)"},
    {"fold_add", FAST(py_fold_add), "fold_add(acc, g)"},
    {"adamw_step", FAST(py_adamw_step), "the step over plain tensors"},
    {"clip", FAST(py_clip), "clip(params, max_norm)"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "plain calls over the C ABI", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&kModule); }
