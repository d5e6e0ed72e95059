// Host path of the table entries: the part of coffin_amd/backend.py that runs on every call.
//
// At one row a projection kernel takes 2.5 .. 10 us and the Python adapter in front of it (argument
// checks, weight lookup, output allocation, foreign-function call) took 7.3 us, so eager decode was
// bound by the host.  Each function here does one entry's whole call for the common case -- exact bf16
// torch tensors on the current device, a weight that the kernels take -- in about 3 us, most of it
// the runtime's own launch, and answers `None` for everything else: the caller then takes the Python
// adapter, which converts and raises the errors.  A weight's first use resolves it through the module.  Nothing is decided differently
// here; the switches and the scratch blocks are the Python module's, read on every call.
//
//   2560 -> 1024, one row, through GEMV.__call__: 7.4 us per call with the Python adapter (kernel 2.6).
//
// The interpreter lock is released around launches (they may wait for room in the queue).
#include <torch/csrc/autograd/VariableTypeUtils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/TensorImpl.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <structmember.h>

#include <unordered_map>

#include "../../include/coffin_mi355.h"

namespace {

// ------------------------------------------------------------------- the Python module's state
PyObject *g_vars = nullptr;   // coffin_amd.backend.__dict__ (borrowed: the module outlives every call)
PyObject *g_check = nullptr;  // coffin_amd._native.check
long long g_handed_uses[2];   // projections that took handed rows: int4 weights, int8 weights

struct Names {
    PyObject *wq, *packed, *scale, *records, *kind, *src, *src2, *a, *b, *n, *k, *kd, *gs, *dev, *family, *index, *device;
    PyObject *prefill_min, *mfma_min, *ragged_min, *batch_mfma, *w8a8_verify, *w4a16, *handover, *handover_min, *handover_max, *seen, *handed;
    PyObject *workspace, *handover_arena, *take, *resolve;
} N;

PyObject *var(PyObject *name) { return PyDict_GetItem(g_vars, name); }  // borrowed

bool truth(PyObject *name) {
    PyObject *v = var(name);
    return v && PyObject_IsTrue(v) == 1;
}

long long number(PyObject *name) {
    PyObject *v = var(name);
    return v ? PyLong_AsLongLong(v) : 0;
}

// ------------------------------------------------------------------------------- weights
// What a launch needs of a quantized weight, copied from the adapter's record.  Trusted while the
// tensors it was made from are the ones the weight object holds (weak references, as in the record).
struct Weight {
    PyObject *src, *src2;  // weak references
    const void *a;
    const float *b;
    int kind, n, k, kd, gs, family;  // family: -1 (the process's setting), 0 dot, 1 mfma
    c10::DeviceIndex dev;
};

std::unordered_map<PyObject *, Weight> g_weights;  // by weight object; entries hold weak references only
constexpr size_t WEIGHTS_MAX = 1 << 16;

bool get_ll(PyObject *o, PyObject *name, long long *out) {
    PyObject *v = PyObject_GetAttr(o, name);
    if (!v) return false;
    *out = PyLong_AsLongLong(v);
    Py_DECREF(v);
    return !(*out == -1 && PyErr_Occurred());
}

bool get_ptr(PyObject *o, PyObject *name, const void **out) {
    PyObject *v = PyObject_GetAttr(o, name);
    if (!v) return false;
    *out = PyLong_AsVoidPtr(v);
    Py_DECREF(v);
    return !PyErr_Occurred();
}

bool holds(PyObject *w, const Weight &e) {
    PyObject *first = PyObject_GetAttr(w, e.kind == 8 ? N.wq : N.packed);
    PyObject *second = first ? PyObject_GetAttr(w, N.scale) : nullptr;
    if (!second) PyErr_Clear();
    // (a dead reference reads as None, which is also what a released weight may hold)
    const bool same = second && first != Py_None && second != Py_None && PyWeakref_GetObject(e.src) == first &&
                      PyWeakref_GetObject(e.src2) == second;
    Py_XDECREF(first);
    Py_XDECREF(second);
    return same;
}

void drop(const Weight &e) {
    Py_DECREF(e.src);
    Py_DECREF(e.src2);
}

// Makes `e` from an adapter's record; false: the record is about other tensors than `w` holds (a dead weight's under the
// same id; not asked of one just made), or an error was set.  The tensors are looked at first: a stale record costs no
// more than that.
bool from_record(PyObject *rec, PyObject *w, bool made, Weight *e) {
    long long kind, n, k, kd, gs, index = -1;
    const void *b = nullptr;
    PyObject *dev = nullptr, *family = nullptr;
    if (!get_ll(rec, N.kind, &kind)) return false;
    e->kind = (int)kind;
    e->src = PyObject_GetAttr(rec, N.src);
    e->src2 = e->src ? PyObject_GetAttr(rec, N.src2) : nullptr;
    bool ok = e->src2 && PyWeakref_Check(e->src) && PyWeakref_Check(e->src2) && (made || holds(w, *e));
    ok = ok && get_ll(rec, N.n, &n) && get_ll(rec, N.k, &k) && get_ll(rec, N.kd, &kd) && get_ll(rec, N.gs, &gs) &&
         get_ptr(rec, N.a, &e->a) && get_ptr(rec, N.b, &b) && (dev = PyObject_GetAttr(rec, N.dev)) &&
         get_ll(dev, N.index, &index) && (family = PyObject_GetAttr(rec, N.family));
    if (ok) {
        e->b = static_cast<const float *>(b);
        e->n = (int)n, e->k = (int)k, e->kd = (int)kd, e->gs = (int)gs;
        e->dev = (c10::DeviceIndex)index;
        e->family = family == Py_None ? -1 : PyUnicode_CompareWithASCIIString(family, "mfma") == 0;
    } else {
        Py_XDECREF(e->src);
        Py_XDECREF(e->src2);
    }
    Py_XDECREF(dev);
    Py_XDECREF(family);
    return ok;
}

// The entry of `w` in `out`: 1, or 0 where the adapter has to answer (a plain tensor, a weight that the kernels do not
// take), or -1 with the Python error set.  Reading an attribute of a weight may run Python code (a property), and with it
// other calls and threads that change the table, so nothing points into the table across such a read.
// resolve_k >= 0: a weight of that width that nobody has used yet is resolved here, by the module's own function.
int find_weight(PyObject *w, Weight *out, int64_t resolve_k, c10::DeviceIndex here) {
    auto it = g_weights.find(w);
    if (it != g_weights.end()) {
        const Weight e = it->second;
        Py_INCREF(e.src);
        Py_INCREF(e.src2);
        const bool same = holds(w, e);
        if (!same && (it = g_weights.find(w)) != g_weights.end() && it->second.src == e.src && it->second.src2 == e.src2) {
            g_weights.erase(it);
            drop(e);  // the table's references
        }
        drop(e);
        if (same) {
            *out = e;
            return 1;
        }
    }
    if (THPVariable_CheckExact(w)) return 0;
    // The adapter's record, by the weight's id.
    PyObject *records = var(N.records), *id = PyLong_FromVoidPtr(w);
    PyObject *rec = records && PyDict_Check(records) && id ? PyDict_GetItem(records, id) : nullptr;
    Py_XINCREF(rec);
    Py_XDECREF(id);
    Weight e{};
    bool ok = rec && from_record(rec, w, false, &e);
    if (PyErr_Occurred()) PyErr_Clear();
    if (!ok && resolve_k >= 0) {
        Py_XDECREF(rec);
        PyObject *width = PyLong_FromLongLong(resolve_k), *device = PyLong_FromLong(here), *resolve = var(N.resolve);
        rec = width && device && resolve ? PyObject_CallFunctionObjArgs(resolve, w, width, device, nullptr) : nullptr;
        Py_XDECREF(width);
        Py_XDECREF(device);
        if (!rec) return -1;
        ok = rec != Py_None && from_record(rec, w, true, &e);
        if (PyErr_Occurred()) PyErr_Clear();
    }
    Py_XDECREF(rec);
    if (!ok) return 0;
    if (g_weights.size() >= WEIGHTS_MAX) {
        std::unordered_map<PyObject *, Weight> all;
        all.swap(g_weights);
        for (auto &w_e : all) drop(w_e.second);
    }
    const auto [at, fresh] = g_weights.try_emplace(w, e);
    if (!fresh) {  // a property's Python code, or another thread during it, has entered the weight
        const Weight before = at->second;
        at->second = e;
        drop(before);
    }
    *out = e;
    return 1;
}

// ------------------------------------------------------------------------------- tensors
// A torch tensor (no subclass) with memory on the current device, or null.
const at::Tensor *plain(PyObject *o, c10::DeviceIndex here) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = reinterpret_cast<THPVariable *>(o)->cdata;
    return t.defined() && t.is_cuda() && t.layout() == c10::kStrided && t.device().index() == here ? &t : nullptr;
}

bool is_bf16(const at::Tensor &t) { return t.scalar_type() == at::kBFloat16; }

at::Tensor new_bf16(c10::IntArrayRef size, c10::DeviceIndex dev) {
    return at::Tensor(at::detail::empty_cuda(size, at::kBFloat16, c10::Device(c10::DeviceType::CUDA, dev), std::nullopt));
}

// Rows of `width` contiguous elements at one pitch, from [width] or [rows, width].
struct Rows {
    int64_t rows, width, pitch;
};

bool rows_of(const at::Tensor &t, Rows *r) {
    if (t.dim() == 1) {
        *r = {1, t.size(0), t.size(0)};
        return t.stride(0) == 1 || t.size(0) <= 1;
    }
    if (t.dim() != 2 || (t.size(1) > 1 && t.stride(1) != 1)) return false;
    *r = {t.size(0), t.size(1), t.size(0) > 1 ? t.stride(0) : std::max(t.stride(0), t.size(1))};
    return r->rows <= INT32_MAX && r->width <= INT32_MAX;
}

struct Unlocked {
    PyThreadState *state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};

// Status of a C-ABI call: true if it succeeded, else the Python error is set.
bool succeeded(int rc, const char *what) {
    if (rc == CMI_OK) return true;
    PyObject *r = PyObject_CallFunction(g_check, "is", rc, what);
    Py_XDECREF(r);
    if (r) PyErr_Format(PyExc_RuntimeError, "%s: status %d", what, rc);
    return false;
}

// ------------------------------------------------------------------------------- scratch
// The module's grow-only blocks (backend._Arena: never freed, never moved), remembered here by address.
struct Scratch {
    PyObject **name;
    unsigned char *base[64] = {};
    size_t bytes[64] = {};

    // Address of `need` bytes, or null with the Python error set.
    unsigned char *take(size_t need, PyObject *tensor, c10::DeviceIndex dev) {
        if (need <= bytes[dev & 63]) return base[dev & 63];
        PyObject *arena = var(*name), *device = PyObject_GetAttr(tensor, N.device);
        PyObject *size = PyLong_FromSize_t(need);
        PyObject *at = arena && device && size ? PyObject_CallMethodObjArgs(arena, N.take, size, device, nullptr) : nullptr;
        Py_XDECREF(device);
        Py_XDECREF(size);
        if (!at) return nullptr;
        base[dev & 63] = static_cast<unsigned char *>(PyLong_AsVoidPtr(at));
        bytes[dev & 63] = need;
        Py_DECREF(at);
        return base[dev & 63];
    }
};
Scratch g_workspace{&N.workspace}, g_handover{&N.handover_arena};

// ------------------------------------------------- quantised rows handed to the next projection
// backend._HANDED: the latest producer output and where its quantised rows are (see there).
struct Handed {
    PyObject_HEAD
    PyObject *tensor;
    long long version, ptr, rows, k, ld, xq, xs, capture;
};

void handed_free(PyObject *self) {
    Py_XDECREF(reinterpret_cast<Handed *>(self)->tensor);
    Py_TYPE(self)->tp_free(self);
}

PyObject *handed_dev(PyObject *self, void *) {
    return PyObject_GetAttr(reinterpret_cast<Handed *>(self)->tensor, N.device);
}

PyMemberDef handed_members[] = {
    {"tensor", T_OBJECT, offsetof(Handed, tensor), READONLY, nullptr},
    {"version", T_LONGLONG, offsetof(Handed, version), READONLY, nullptr},
    {"ptr", T_LONGLONG, offsetof(Handed, ptr), READONLY, nullptr},
    {"rows", T_LONGLONG, offsetof(Handed, rows), READONLY, nullptr},
    {"k", T_LONGLONG, offsetof(Handed, k), READONLY, nullptr},
    {"ld", T_LONGLONG, offsetof(Handed, ld), READONLY, nullptr},
    {"xq", T_LONGLONG, offsetof(Handed, xq), READONLY, nullptr},
    {"xs", T_LONGLONG, offsetof(Handed, xs), READONLY, nullptr},
    {"capture", T_LONGLONG, offsetof(Handed, capture), READONLY, nullptr},
    {nullptr, 0, 0, 0, nullptr}};

PyGetSetDef handed_getset[] = {{"dev", handed_dev, nullptr, nullptr, nullptr}, {nullptr, nullptr, nullptr, nullptr, nullptr}};

PyTypeObject HandedType = {PyVarObject_HEAD_INIT(nullptr, 0)};

void drop_handed() {
    if (var(N.handed) != Py_None) PyDict_SetItem(g_vars, N.handed, Py_None);
}

long long address(const void *p) { return (long long)reinterpret_cast<intptr_t>(p); }
size_t round256(size_t v) { return (v + 255) / 256 * 256; }

// Room for the quantised rows of a producer; false where it should not leave any.
bool hand_target(int64_t rows, int64_t k, PyObject *tensor, c10::DeviceIndex dev, int8_t **xq, float **xs) {
    if (rows < number(N.handover_min) || rows * k > number(N.handover_max) || !truth(N.handover) || !truth(N.seen)) return false;
    unsigned char *base = g_handover.take(round256((size_t)rows * k) + round256(4 * (size_t)rows), tensor, dev);
    if (!base) {
        PyErr_Clear();  // it would have to grow inside a capture: this call goes without
        return false;
    }
    *xq = reinterpret_cast<int8_t *>(base);
    *xs = reinterpret_cast<float *>(base + round256((size_t)rows * k));
    return true;
}

void hand_over(PyObject *obj, const at::Tensor &t, int64_t rows, int64_t k, int64_t ld, int8_t *xq, float *xs, void *stream) {
    if (t.is_inference()) return;  // no version counter: writes to it would go unseen
    Handed *h = PyObject_New(Handed, &HandedType);
    if (!h) {
        PyErr_Clear();
        return;
    }
    Py_INCREF(obj);
    h->tensor = obj;
    h->version = t._version();
    h->ptr = address(t.const_data_ptr());
    h->rows = rows, h->k = k, h->ld = ld;
    h->xq = address(xq), h->xs = address(xs);
    h->capture = cmi_stream_capture_id(stream);
    PyDict_SetItem(g_vars, N.handed, reinterpret_cast<PyObject *>(h));
    Py_DECREF(h);
}

// Whether `h` is about exactly this activation (backend._handed_rows).
bool handed_matches(const Handed *h, const at::Tensor &x, int64_t rows, int64_t k, void *stream) {
    const at::Tensor &t = reinterpret_cast<THPVariable *>(h->tensor)->cdata;
    if (address(x.const_data_ptr()) != h->ptr || rows != h->rows || k != h->k || x.device() != t.device()) return false;
    if (x.is_inference() || (long long)x._version() != h->version) return false;
    if (x.stride(-1) != 1 || (x.dim() == 2 && rows > 1 && x.stride(0) != h->ld)) return false;
    return cmi_stream_capture_id(stream) == h->capture;
}

// --------------------------------------------------------------------------------- entries
constexpr int PREFILL = 1, MFMA = 2;

// Column ranges of a projection's output: what `split` returns, views of it (its memory, its version counter, `_base`).
// Made directly: through the dispatcher three parts of a CPU tensor take 2.5 us, this way 1.3.
PyObject *parts_of(const at::Tensor &y, PyObject *sizes) {
    PyObject *seq = PySequence_Fast(sizes, "sizes");
    if (!seq) return nullptr;
    const Py_ssize_t count = PySequence_Fast_GET_SIZE(seq);
    PyObject *out = PyTuple_New(count);
    const auto meta = at::GradMode::is_enabled() ? torch::autograd::CreationMeta::MULTI_OUTPUT_NODE
                                                 : torch::autograd::CreationMeta::NO_GRAD_MODE;
    int64_t at = 0;
    for (Py_ssize_t i = 0; out && i < count; ++i) {
        const int64_t n = PyLong_AsLongLong(PySequence_Fast_GET_ITEM(seq, i));
        if (n < 0 || at + n > y.size(-1)) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "sizes do not match the projection's outputs");
            Py_CLEAR(out);
            break;
        }
        at::Tensor piece = at::detail::make_tensor<c10::TensorImpl>(c10::TensorImpl::VIEW, c10::Storage(y.storage()), y.key_set(), y.dtype());
        c10::TensorImpl *impl = piece.unsafeGetTensorImpl();
        if (y.dim() == 1) {
            const int64_t size[1] = {n};
            impl->set_sizes_and_strides(size, y.strides(), y.storage_offset() + at);
        } else {
            const int64_t size[2] = {y.size(0), n};
            impl->set_sizes_and_strides(size, y.strides(), y.storage_offset() + at);
        }
        PyObject *o = THPVariable_Wrap(torch::autograd::as_view(y, piece, true, true, nullptr, nullptr, meta));
        if (!o) {
            Py_CLEAR(out);
            break;
        }
        PyTuple_SET_ITEM(out, i, o);
        at += n;
    }
    Py_DECREF(seq);
    if (out && at != y.size(-1)) {
        PyErr_SetString(PyExc_RuntimeError, "sizes do not match the projection's outputs");
        Py_CLEAR(out);
    }
    return out;
}

// project(w, x, flags[, sizes]): backend._project for a known weight and contiguous bf16 rows.
PyObject *project(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs < 3) Py_RETURN_NONE;
    const c10::DeviceIndex here = c10::hip::current_device();
    const at::Tensor *xp = plain(args[1], here);
    if (!xp || !is_bf16(*xp)) Py_RETURN_NONE;
    const at::Tensor &x = *xp;
    const int64_t nd = x.dim();
    if ((nd != 1 && nd != 2) || !x.is_contiguous()) Py_RETURN_NONE;
    const int64_t rows = nd == 1 ? 1 : x.size(0);
    if (rows < 1 || rows > INT32_MAX) Py_RETURN_NONE;
    Weight e;
    const int found = find_weight(args[0], &e, x.size(-1), here);
    if (found < 0) return nullptr;
    if (!found || e.dev != here || x.size(-1) != e.k) Py_RETURN_NONE;
    const long flags = PyLong_AsLong(args[2]);
    const bool quantised = e.kind == 4 || ((flags & PREFILL) && rows >= number(N.prefill_min));
    if (e.kind == 4 ? truth(N.w4a16) : ((flags & MFMA) && !(flags & PREFILL) && truth(N.w8a8_verify))) Py_RETURN_NONE;

    void *stream = c10::hip::getCurrentHIPStream(here).stream();
    const int M = (int)rows, Nn = e.n, K = e.k;
    const int8_t *xq = nullptr;
    const float *xs = nullptr;
    size_t need = 0;
    unsigned char *work = nullptr;
    if (quantised) {
        PyObject *handed = var(N.handed);
        if (handed && handed != Py_None && e.kd == K) {
            if (Py_TYPE(handed) != &HandedType) Py_RETURN_NONE;  // left by the Python adapter, which can read it
            const Handed *h = reinterpret_cast<Handed *>(handed);
            // a W8A8 shape that splits K needs the quantiser's launch, which clears its counters
            if (handed_matches(h, x, rows, K, stream) && (e.kind == 4 || !cmi_linear_w8a8_splits(M, Nn, K))) {
                xq = reinterpret_cast<const int8_t *>(static_cast<intptr_t>(h->xq));
                xs = reinterpret_cast<const float *>(static_cast<intptr_t>(h->xs));
                ++g_handed_uses[e.kind == 8];
            }
        }
        if (!xq) {
            need = e.kind == 4 ? cmi_linear_workspace_bytes(M, e.kd) : cmi_linear_w8a8_workspace_bytes(M, Nn, K);
            work = g_workspace.take(need, args[1], here);
            if (!work) return nullptr;
            if (!truth(N.seen)) PyDict_SetItem(g_vars, N.seen, Py_True);
        }
    }
    const int64_t size[2] = {rows, Nn};
    at::Tensor y = new_bf16(nd == 1 ? c10::IntArrayRef(size + 1, 1) : c10::IntArrayRef(size, 2), here);
    void *yp = y.mutable_data_ptr();
    const void *xd = x.const_data_ptr();
    const bool whole = e.family >= 0 ? e.family == 1 : truth(N.batch_mfma);
    const bool fast = !quantised && K % 128 == 0 && (whole || ((flags & MFMA) && rows >= number(N.mfma_min)));
    // rows that end inside a line of 128
    const bool ragged = !quantised && !whole && K % 128 != 0 && K % 16 == 0 && K >= 128 && (flags & MFMA) && rows >= number(N.ragged_min);
    int rc;
    const char *what;
    {
        Unlocked unlocked;
        if (e.kind == 4) {
            const uint8_t *w4 = static_cast<const uint8_t *>(e.a);
            if (xq) {
                what = "projection of quantised rows";
                rc = M <= 16 ? cmi_gemv_w4a8(w4, e.b, xq, xs, yp, nullptr, M, Nn, K, e.gs, stream)
                             : cmi_gemm_w4a8(w4, e.b, xq, xs, yp, nullptr, M, Nn, K, e.gs, stream);
            } else {
                what = "linear_w4a8_bf16";
                rc = cmi_linear_w4a8_bf16(w4, e.b, xd, yp, M, Nn, K, e.gs, work, need, stream);
            }
        } else {
            const int8_t *wq = static_cast<const int8_t *>(e.a);
            if (xq) {
                what = "projection of quantised rows";
                rc = cmi_gemm_w8a8(xq, wq, xs, e.b, yp, nullptr, M, Nn, K, Nn, stream);
            } else if (quantised) {
                what = "linear_w8a8_bf16";
                rc = cmi_linear_w8a8_bf16(xd, wq, e.b, yp, M, Nn, K, Nn, work, need, stream);
            } else {
                what = "linear_w8a16";
                rc = ragged ? cmi_linear_w8a16_rows(wq, e.b, xd, yp, M, Nn, K, stream) : cmi_linear_w8a16(wq, e.b, xd, yp, M, Nn, K, fast ? CMI_FAMILY_MFMA : CMI_FAMILY_DOT, stream);
            }
        }
    }
    if (!succeeded(rc, what)) return nullptr;
    if (nargs > 3) return parts_of(y, args[3]);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// rms_norm(x, w, eps): backend.rms_norm for bf16 rows and a bf16 gain.
PyObject *rms_norm(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 3) Py_RETURN_NONE;
    const c10::DeviceIndex here = c10::hip::current_device();
    const at::Tensor *x = plain(args[0], here), *w = plain(args[1], here);
    Rows r;
    if (!x || !w || !is_bf16(*x) || !is_bf16(*w) || x->dim() != 2 || !rows_of(*x, &r) || r.rows < 1 || r.width < 1) Py_RETURN_NONE;
    if (w->numel() != r.width || !w->is_contiguous()) Py_RETURN_NONE;
    const double eps = PyFloat_AsDouble(args[2]);
    if (eps == -1.0 && PyErr_Occurred()) return nullptr;
    drop_handed();
    void *stream = c10::hip::getCurrentHIPStream(here).stream();
    const int64_t size[2] = {r.rows, r.width};
    at::Tensor y = new_bf16(size, here);
    int8_t *xq = nullptr;
    float *xs = nullptr;
    const bool hand = hand_target(r.rows, r.width, args[0], here, &xq, &xs);
    int rc;
    {
        const void *xd = x->const_data_ptr(), *wd = w->const_data_ptr();
        void *yd = y.mutable_data_ptr();
        Unlocked unlocked;
        rc = cmi_rms_norm_i8(xd, wd, yd, xq, xs, (int)r.rows, (int)r.width, r.pitch, r.width, (float)eps, stream);
    }
    if (!succeeded(rc, "rms_norm")) return nullptr;
    PyObject *out = THPVariable_Wrap(y);
    if (out && hand) hand_over(out, y, r.rows, r.width, r.width, xq, xs, stream);
    return out;
    END_HANDLE_TH_ERRORS
}

// add_rms_norm(x, add, w, out, eps): backend.add_rms_norm; answers `out`.
PyObject *add_rms_norm(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 5) Py_RETURN_NONE;
    const c10::DeviceIndex here = c10::hip::current_device();
    const at::Tensor *x = plain(args[0], here), *add = plain(args[1], here), *w = plain(args[2], here), *out = plain(args[3], here);
    Rows r, ra, ro;
    if (!x || !add || !w || !out || !is_bf16(*x) || !is_bf16(*add) || !is_bf16(*w) || !is_bf16(*out)) Py_RETURN_NONE;
    if (x->dim() != 2 || add->sizes() != x->sizes() || out->sizes() != x->sizes()) Py_RETURN_NONE;
    if (!rows_of(*x, &r) || !rows_of(*add, &ra) || !rows_of(*out, &ro) || r.rows < 1 || r.width < 1) Py_RETURN_NONE;
    if (w->numel() != r.width || !w->is_contiguous()) Py_RETURN_NONE;
    const double eps = PyFloat_AsDouble(args[4]);
    if (eps == -1.0 && PyErr_Occurred()) return nullptr;
    drop_handed();
    void *stream = c10::hip::getCurrentHIPStream(here).stream();
    int8_t *xq = nullptr;
    float *xs = nullptr;
    const bool hand = hand_target(r.rows, r.width, args[0], here, &xq, &xs);
    int rc;
    {
        void *xd = x->mutable_data_ptr(), *od = out->mutable_data_ptr();
        const void *ad = add->const_data_ptr(), *wd = w->const_data_ptr();
        Unlocked unlocked;
        rc = cmi_add_rms_norm_i8(xd, ad, wd, od, xq, xs, (int)r.rows, (int)r.width, r.pitch, ra.pitch, ro.pitch, (float)eps, stream);
    }
    if (!succeeded(rc, "add_rms_norm")) return nullptr;
    if (hand) hand_over(args[3], *out, r.rows, r.width, ro.pitch, xq, xs, stream);
    Py_INCREF(args[3]);
    return args[3];
    END_HANDLE_TH_ERRORS
}

// int8 rows and their scales in a caller's buffers.
bool quantised_buffers(const at::Tensor *q, const at::Tensor *s, int64_t rows, int64_t k) {
    return q && s && q->scalar_type() == at::kChar && s->scalar_type() == at::kFloat && q->is_contiguous() &&
           s->is_contiguous() && s->numel() == rows && q->dim() == 2 && q->size(0) == rows && q->size(1) == k;
}

// silu_mul(gate, up, out[, out_q, out_s]): backend.silu_mul / silu_mul_quant; answers `out`.
PyObject *silu_mul(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 3 && nargs != 5) Py_RETURN_NONE;
    const c10::DeviceIndex here = c10::hip::current_device();
    const at::Tensor *gate = plain(args[0], here), *up = plain(args[1], here), *out = plain(args[2], here);
    Rows g, u, o;
    if (!gate || !up || !out || !is_bf16(*gate) || !is_bf16(*up) || !is_bf16(*out)) Py_RETURN_NONE;
    if (up->sizes() != gate->sizes() || out->sizes() != gate->sizes()) Py_RETURN_NONE;
    if (!rows_of(*gate, &g) || !rows_of(*up, &u) || !rows_of(*out, &o) || g.rows < 1 || g.width < 1) Py_RETURN_NONE;
    int8_t *xq = nullptr;
    float *xs = nullptr;
    bool hand = false;
    if (nargs == 5) {
        const at::Tensor *q = plain(args[3], here), *s = plain(args[4], here);
        if (gate->dim() != 2 || !quantised_buffers(q, s, g.rows, g.width)) Py_RETURN_NONE;
        xq = static_cast<int8_t *>(q->mutable_data_ptr());
        xs = static_cast<float *>(s->mutable_data_ptr());
    }
    drop_handed();
    if (nargs == 3) hand = hand_target(g.rows, g.width, args[0], here, &xq, &xs);
    void *stream = c10::hip::getCurrentHIPStream(here).stream();
    int rc;
    {
        const void *gd = gate->const_data_ptr(), *ud = up->const_data_ptr();
        void *od = out->mutable_data_ptr();
        Unlocked unlocked;
        rc = cmi_silu_mul_quant(gd, ud, od, xq, xs, (int)g.rows, (int)g.width, g.pitch, u.pitch, o.pitch, stream);
    }
    if (!succeeded(rc, "silu_mul_quant")) return nullptr;
    if (hand) hand_over(args[2], *out, g.rows, g.width, o.pitch, xq, xs, stream);
    Py_INCREF(args[2]);
    return args[2];
    END_HANDLE_TH_ERRORS
}

// kv_quant(x, out_q, out_s): backend.kv_quant for contiguous bf16 rows; answers `out_q`.
PyObject *kv_quant(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 3) Py_RETURN_NONE;
    const c10::DeviceIndex here = c10::hip::current_device();
    const at::Tensor *x = plain(args[0], here), *q = plain(args[1], here), *s = plain(args[2], here);
    if (!x || !is_bf16(*x) || x->dim() != 2 || !x->is_contiguous() || x->size(0) < 1 || x->size(0) > INT32_MAX || x->size(1) < 1 ||
        x->size(1) > INT32_MAX || !quantised_buffers(q, s, x->size(0), x->size(1)))
        Py_RETURN_NONE;
    PyObject *handed = var(N.handed);
    if (handed && handed != Py_None) {
        if (Py_TYPE(handed) != &HandedType) Py_RETURN_NONE;
        const at::Tensor &t = reinterpret_cast<THPVariable *>(reinterpret_cast<Handed *>(handed)->tensor)->cdata;
        if (t.storage().data() == q->storage().data() || t.storage().data() == s->storage().data()) drop_handed();
    }
    void *stream = c10::hip::getCurrentHIPStream(here).stream();
    int rc;
    {
        const int M = (int)x->size(0), K = (int)x->size(1);
        const void *xd = x->const_data_ptr();
        int8_t *qd = static_cast<int8_t *>(q->mutable_data_ptr());
        float *sd = static_cast<float *>(s->mutable_data_ptr());
        Unlocked unlocked;
        rc = cmi_quant_act_i8(xd, qd, sd, M, K, stream);
    }
    if (!succeeded(rc, "quant_act_i8")) return nullptr;
    Py_INCREF(args[1]);
    return args[1];
    END_HANDLE_TH_ERRORS
}

// embed_rows(w, ids): backend.embed_rows for a known weight and contiguous int64 ids.
PyObject *embed_rows(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 2) Py_RETURN_NONE;
    const c10::DeviceIndex here = c10::hip::current_device();
    const at::Tensor *ids = plain(args[1], here);
    if (!ids || ids->scalar_type() != at::kLong || !ids->is_contiguous() || ids->numel() < 1 || ids->numel() > INT32_MAX) Py_RETURN_NONE;
    Weight e;
    if (find_weight(args[0], &e, -1, here) != 1 || e.dev != here) Py_RETURN_NONE;
    void *stream = c10::hip::getCurrentHIPStream(here).stream();
    const int64_t size[2] = {ids->numel(), e.k};
    at::Tensor y = new_bf16(size, here);
    int rc;
    {
        const int T = (int)size[0];
        const int64_t *id = static_cast<const int64_t *>(ids->const_data_ptr());
        void *yd = y.mutable_data_ptr();
        Unlocked unlocked;
        rc = e.kind == 4 ? cmi_embed_rows_w4(static_cast<const uint8_t *>(e.a), e.b, id, yd, T, e.n, e.k, e.gs, stream)
                         : cmi_embed_rows_i8(static_cast<const int8_t *>(e.a), e.b, id, yd, T, e.n, e.k, stream);
    }
    if (!succeeded(rc, "embed_rows")) return nullptr;
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// handed_uses(): how many projections took rows a producer had quantised, (int4 weights, int8 weights).
PyObject *handed_uses(PyObject *, PyObject *const *, Py_ssize_t) {
    return Py_BuildValue("LL", g_handed_uses[0], g_handed_uses[1]);
}

// bind(vars, check): the module whose state this is (once).
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    if (nargs != 2 || !PyDict_Check(args[0])) {
        PyErr_SetString(PyExc_TypeError, "bind(module dict, check)");
        return nullptr;
    }
    for (int i = 0; i < 2; ++i) Py_INCREF(args[i]);
    g_vars = args[0];
    g_check = args[1];
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
    {"handed_uses", (PyCFunction)(void (*)(void))handed_uses, METH_FASTCALL, nullptr},
    {"project", (PyCFunction)(void (*)(void))project, METH_FASTCALL, nullptr},
    {"rms_norm", (PyCFunction)(void (*)(void))rms_norm, METH_FASTCALL, nullptr},
    {"add_rms_norm", (PyCFunction)(void (*)(void))add_rms_norm, METH_FASTCALL, nullptr},
    {"silu_mul", (PyCFunction)(void (*)(void))silu_mul, METH_FASTCALL, nullptr},
    {"kv_quant", (PyCFunction)(void (*)(void))kv_quant, METH_FASTCALL, nullptr},
    {"embed_rows", (PyCFunction)(void (*)(void))embed_rows, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    HandedType.tp_name = "coffin_amd._host.Handed";
    HandedType.tp_basicsize = sizeof(Handed);
    HandedType.tp_dealloc = handed_free;
    HandedType.tp_flags = Py_TPFLAGS_DEFAULT;
    HandedType.tp_members = handed_members;
    HandedType.tp_getset = handed_getset;
    if (PyType_Ready(&HandedType) < 0) return nullptr;
    struct {
        PyObject **slot;
        const char *text;
    } const all[] = {{&N.wq, "wq"}, {&N.packed, "packed"}, {&N.scale, "scale"}, {&N.records, "_RECORDS"}, {&N.kind, "kind"},
                     {&N.src, "src"}, {&N.src2, "src2"}, {&N.a, "a"}, {&N.b, "b"}, {&N.n, "n"}, {&N.k, "k"}, {&N.kd, "kd"},
                     {&N.gs, "gs"}, {&N.dev, "dev"}, {&N.family, "family"}, {&N.index, "index"}, {&N.device, "device"},
                     {&N.prefill_min, "PREFILL_MIN_ROWS"}, {&N.mfma_min, "MFMA_MIN_ROWS"}, {&N.ragged_min, "RAGGED_MFMA_MIN_ROWS"}, {&N.batch_mfma, "BATCH_MFMA"}, {&N.w8a8_verify, "W8A8_VERIFY"}, {&N.w4a16, "W4A16"},
                     {&N.handover, "HANDOVER"}, {&N.handover_min, "HANDOVER_MIN_ROWS"}, {&N.handover_max, "HANDOVER_MAX_BYTES"},
                     {&N.seen, "_QUANT_CONSUMER_SEEN"}, {&N.handed, "_HANDED"},
                     {&N.workspace, "_WORKSPACE"}, {&N.handover_arena, "_HANDOVER_ARENA"}, {&N.take, "take"}, {&N.resolve, "_resolve"}};
    for (const auto &e : all)
        if (!(*e.slot = PyUnicode_InternFromString(e.text))) return nullptr;
    return PyModule_Create(&module);
}
