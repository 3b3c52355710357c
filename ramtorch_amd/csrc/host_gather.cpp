// Host-side helper of AdamW.step, for sets of any size: walks one
// param group and writes the rt_tensor_desc rows of every "plain" tensor (param, gradient
// and both states contiguous on one GPU, supported dtypes) straight into a caller-owned
// buffer, advancing state["step"] as adamw.py:177 does.  It does, per tensor, what the Python
// loop of AdamW.step does (the checks of adamw.py:112-119 and the lazy-state test of
// adamw.py:125), only without ~2 us of interpreter and binding overhead per tensor; whatever
// is not plain is handed back to that Python loop untouched.
//
// A CPython extension that reads torch tensors through torch's C++ API.  It moves no tensor
// data and launches nothing: the update itself runs behind the C ABI of
// include/ramtorch_sr_adamw.h.  Optional: AdamW.step works without it.
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>
#include <ATen/core/Tensor.h>

#include <cstdint>
#include <algorithm>
#include <cstring>
#include <thread>
#include <utility>
#include <vector>

#include "../../include/ramtorch_sr_adamw.h"

static_assert(sizeof(rt_tensor_desc) == 136, "rt_tensor_desc layout");

namespace {

PyObject* k_ema = nullptr;
PyObject* k_ema_squared = nullptr;
PyObject* k_step = nullptr;
Py_hash_t h_ema = 0, h_ema_squared = 0, h_step = 0;
PyTypeObject* t_tensor = nullptr;     // torch.Tensor
PyTypeObject* t_parameter = nullptr;  // torch.nn.Parameter

enum Status : uint8_t {
    kWritten = 0,  // row written, state["step"] advanced
    kNoGrad = 1,   // grad is None: skipped, step not advanced (adamw.py:114)
    kPython = 2,   // not plain (or not initialised yet): the Python loop handles it
};

inline bool exact_tensor(PyObject* o) {
    PyTypeObject* t = Py_TYPE(o);
    return t == t_tensor || t == t_parameter;
}

inline const c10::TensorImpl* impl_of(PyObject* o) { return THPVariable_Unpack(o).unsafeGetTensorImpl(); }

// dtype code of a param / state (bf16, f32, f16, f64) or -1
inline int pmv_code(const c10::TensorImpl* t) {
    switch (c10::typeMetaToScalarType(t->dtype())) {
        case at::kBFloat16: return RT_DT_BF16;
        case at::kFloat: return RT_DT_F32;
        case at::kHalf: return RT_DT_F16;
        case at::kDouble: return RT_DT_F64;
        default: return -1;
    }
}

// dtype code of a gradient (bf16, f32, f16) or -1
inline int grad_code(const c10::TensorImpl* t) {
    const int code = pmv_code(t);
    return code == RT_DT_F64 ? -1 : code;
}

// dev >= 0: on that GPU; dev < 0: in host memory (exercised by the CPU-only tests of this
// helper; the optimizer only ever passes a GPU index)
inline bool dense_on(const c10::TensorImpl* t, int dev) {
    if (t->layout() != at::kStrided || !t->is_contiguous()) return false;
    return dev >= 0 ? (t->is_cuda() && t->get_device() == dev) : t->is_cpu();
}

// Function transforms' tensors have no storage; a Python subclass and a nested tensor have sizes of their own kind.
inline bool ordinary(const c10::TensorImpl* t) {
    const uint64_t odd = c10::DispatchKeySet(c10::DispatchKey::Python).raw_repr() |
                         c10::DispatchKeySet(c10::DispatchKey::NestedTensor).raw_repr();
    return (t->key_set().raw_repr() & odd) == 0 && t->has_storage();
}

inline void* data_of(const c10::TensorImpl* t) { return const_cast<c10::TensorImpl*>(t)->mutable_data(); }

// A state dict's entry (borrowed) or NULL.  With the hash at hand a lookup costs half of PyDict_GetItem, which also
// saves and restores the interpreter's error state.
inline PyObject* entry(PyObject* dict, PyObject* key, Py_hash_t hash) {
#if PY_VERSION_HEX < 0x030D0000
    PyObject* o = _PyDict_GetItem_KnownHash(dict, key, hash);
    if (!o && PyErr_Occurred()) PyErr_Clear();   // a foreign key's comparison failed: not there
    return o;
#else
    (void)hash;
    return PyDict_GetItem(dict, key);
#endif
}

// The walk below is a chain of dependent loads per tensor (list item -> Python wrapper ->
// TensorImpl -> autograd meta -> gradient -> storage, and the same through the state dict), and
// with tens of thousands of tensors none of it is in cache: the chain's latency is the cost.
// Warm runs ahead of the main loop as a software pipeline: level k of the chain is prefetched
// for tensor i + (5 - k) * kLead while tensor i is processed, so each level finds the
// previous one already in cache.  It hands what it has read to the main loop and decides nothing.  Nothing runs in between
// that could change it: of what it holds, the main loop only replaces a state's step.
constexpr size_t kLead = 6;
constexpr size_t kRing = 64;  // > 5 * kLead, a power of two

inline void touch(const void* p, int lines = 1) {
    const char* c = static_cast<const char*>(p);
    for (int k = 0; k < lines; ++k) __builtin_prefetch(c + 64 * k, 0, 3);
}

struct Warm {
    PyObject* params;
    PyObject* states;
    PyObject* grads;   // list or NULL
    size_t n;
    // What the walk has found out about tensor i, at i % kRing: the main loop uses it too.
    const c10::TensorImpl* impl[kRing][4];   // p, gradient, ema, ema_squared; NULL: none, or not an exact Tensor / Parameter
    PyObject* obj[kRing][3];                 // the state's ema, ema_squared, step (borrowed) or NULL

    template <int LEVEL>
    void level(size_t i) {
        if (i >= n) return;
        const size_t r = i % kRing;
        PyObject* po = PyList_GET_ITEM(params, i);
        PyObject* so = PyList_GET_ITEM(states, i);
        if constexpr (LEVEL == 0) {   // wrappers and dict headers
            touch(po);
            touch(so);
            if (grads) touch(PyList_GET_ITEM(grads, i));
        } else if constexpr (LEVEL == 1) {   // TensorImpl of the param; key table of the dict
            impl[r][0] = exact_tensor(po) ? impl_of(po) : nullptr;
            if (impl[r][0]) touch(impl[r][0], 4);
            if (PyDict_CheckExact(so)) touch(reinterpret_cast<PyDictObject*>(so)->ma_keys, 4);
        } else if constexpr (LEVEL == 2) {   // autograd meta + storage of the param; state objects
            if (impl[r][0]) {
                if (!grads) touch(impl[r][0]->autograd_meta(), 2);
                touch(impl[r][0]->unsafe_storage().unsafeGetStorageImpl());
            }
            obj[r][0] = obj[r][1] = obj[r][2] = nullptr;
            if (PyDict_CheckExact(so)) {
                obj[r][0] = entry(so, k_ema, h_ema);
                obj[r][1] = entry(so, k_ema_squared, h_ema_squared);
                obj[r][2] = entry(so, k_step, h_step);
                for (int j = 0; j < 3; ++j)
                    if (obj[r][j]) touch(obj[r][j]);
            }
        } else if constexpr (LEVEL == 3) {   // TensorImpl of the gradient and of both states
            impl[r][1] = nullptr;
            if (grads) {
                PyObject* go = PyList_GET_ITEM(grads, i);
                if (exact_tensor(go)) impl[r][1] = impl_of(go);
            } else if (impl[r][0]) {
                const at::Tensor& g = THPVariable_Unpack(po).grad();
                if (g.defined()) impl[r][1] = g.unsafeGetTensorImpl();
            }
            for (int j = 0; j < 2; ++j)
                impl[r][2 + j] = obj[r][j] && exact_tensor(obj[r][j]) ? impl_of(obj[r][j]) : nullptr;
            for (int j = 1; j < 4; ++j)
                if (impl[r][j]) touch(impl[r][j], 4);
        } else {   // their storages
            for (int j = 1; j < 4; ++j)
                if (impl[r][j]) touch(impl[r][j]->unsafe_storage().unsafeGetStorageImpl());
        }
    }

    // called before tensor i is processed; afterwards its entries are complete
    void ahead_of(size_t i) {
        if (i == 0) {  // fill the pipeline
            for (size_t j = 0; j < 5 * kLead; ++j) level<0>(j);
            for (size_t j = 0; j < 4 * kLead; ++j) level<1>(j);
            for (size_t j = 0; j < 3 * kLead; ++j) level<2>(j);
            for (size_t j = 0; j < 2 * kLead; ++j) level<3>(j);
            for (size_t j = 0; j < 1 * kLead; ++j) level<4>(j);
        }
        level<0>(i + 5 * kLead);
        level<1>(i + 4 * kLead);
        level<2>(i + 3 * kLead);
        level<3>(i + 2 * kLead);
        level<4>(i + 1 * kLead);
    }
};

// Whether the update can take the row means of such a tensor itself (the rule of the library's row-wise kernel).
inline bool sums_rows_itself(const rt_tensor_desc& d) {
    constexpr uint64_t kMin = 512, kMax = 32768;   // elements of a row
    const auto narrow = [](uint8_t dt) { return dt == RT_DT_BF16 || dt == RT_DT_F16; };
    return d.row_len % 8 == 0 && d.row_len >= kMin && d.row_len <= kMax && narrow(d.p_dtype) && narrow(d.g_dtype) &&
           narrow(d.m_dtype) && narrow(d.v_dtype) && (d.m_dtype == RT_DT_F16) == (d.v_dtype == RT_DT_F16);
}

// (new step, its number as a Python int): tensors at the same step share the object
using Steps = std::vector<std::pair<long long, PyObject*>>;

struct Walk {
    PyObject *params, *states, *grads, *recorded;   // the last two may be NULL
    Py_ssize_t n, cap;
    int dev;
    long centralize;
    unsigned long scalars_base, id_base;
    rt_tensor_desc* rows;
    uint8_t* status;       // kPython everywhere when the walk begins
    Py_ssize_t written, left;   // results
    uint64_t means;
};

// The walk of gather_group.  False: a Python error is set.  It may throw as well, where torch does not give away a
// tensor's sizes or memory; either way `status` says which step counts have moved, and those tensors' rows by how much.
bool walk_group(Walk& a, Steps& steps) {
    PyObject *const params = a.params, *const states = a.states, *const grads = a.grads, *const recorded = a.recorded;
    const Py_ssize_t n = a.n, cap = a.cap;
    const int dev = a.dev;
    const long centralize = a.centralize;
    const unsigned long scalars_base = a.scalars_base, id_base = a.id_base;
    rt_tensor_desc* const rows = a.rows;
    uint8_t* const status = a.status;
    Py_ssize_t w = 0, left = 0;
    uint64_t means = 0;
    Warm warm;
    warm.params = params;
    warm.states = states;
    warm.grads = grads;
    warm.n = (size_t)n;
    for (Py_ssize_t i = 0; i < n; ++i) {
        warm.ahead_of(i);
        ++left;
        PyObject* po = PyList_GET_ITEM(params, i);
        PyObject* so = PyList_GET_ITEM(states, i);
        const c10::TensorImpl* const* im = warm.impl[(size_t)i % kRing];
        const c10::TensorImpl *p = im[0], *g = im[1], *m = im[2], *v = im[3];
        if (!p || !PyDict_CheckExact(so) || (recorded && PyList_GET_ITEM(recorded, i) != po)) continue;
        if (!g) {
            if (grads && PyList_GET_ITEM(grads, i) != Py_None) continue;
            status[i] = kNoGrad;
            --left;
            continue;
        }
        if (w >= cap) continue;
        PyObject* st = entry(so, k_step, h_step);   // (not the one found ahead: the same dict may have had its turn since)
        if (!m || !v || !st || !PyLong_CheckExact(st)) continue;
        const int pc = pmv_code(p), mc = pmv_code(m), vc = pmv_code(v), gc = grad_code(g);
        if (pc < 0 || mc < 0 || vc < 0 || gc < 0) continue;
        if (!ordinary(g) || !dense_on(p, dev) || !dense_on(g, dev) || !dense_on(m, dev) || !dense_on(v, dev))
            continue;
        const int64_t numel = p->numel();
        if (g->numel() != numel || m->numel() != numel || v->numel() != numel) continue;
        int overflow = 0;
        const long long step = PyLong_AsLongLongAndOverflow(st, &overflow);
        if (overflow || step < 0) continue;
        const long long new_step = step + 1;  // adamw.py:177
        size_t si = steps.size();
        for (size_t k = steps.size(); k-- > 0;)
            if (steps[k].first == new_step) {
                si = k;
                break;
            }
        if (si == steps.size()) {
            PyObject* ns = PyLong_FromLongLong(new_step);
            if (!ns) return false;
            steps.emplace_back(new_step, ns);
        }
        if (PyDict_SetItem(so, k_step, steps[si].second) != 0) return false;
        // (what putting the count back takes; with the addresses read before the dict is written the walk measured
        // 124 ns a tensor instead of 105)
        rows[w].scalars_idx = (uint32_t)(scalars_base + si);
        status[i] = kWritten;

        rt_tensor_desc d{};
        d.p = data_of(p);
        d.g = data_of(g);
        d.m = data_of(m);
        d.v = data_of(v);
        d.numel = (uint64_t)numel;
        d.tensor_id = (uint32_t)(id_base + (unsigned long)i);
        d.step = (uint32_t)((unsigned long long)new_step & 0xFFFFFFFFull);
        d.scalars_idx = (uint32_t)(scalars_base + si);
        d.p_dtype = (uint8_t)pc;
        d.g_dtype = (uint8_t)gc;
        d.m_dtype = (uint8_t)mc;
        d.v_dtype = (uint8_t)vc;
        --left;
        if (centralize && numel > 0) {
            const uint64_t count = g->dim() >= 2 ? (uint64_t)g->size(0) : 1;
            d.row_len = (uint64_t)numel / count;
            if (centralize != 2 || !sums_rows_itself(d)) {
                d.row_mean = reinterpret_cast<float*>(means + 1);
                means += count;
            }
        }
        rows[w++] = d;
    }
    a.written = w;
    a.left = left;
    a.means = means;
    return true;
}

// gather_group(params, states, dev, desc_addr, desc_cap, status_addr, scalars_base, tensor_id_base
//              [, grads, centralize[, recorded]])
//   -> (rows_written, [distinct new step values, in order of first use]
//       [, tensors left to the caller, row means needed])
// params: list of tensors; states: list of the per-param state dicts (same order);
// desc_addr / desc_cap: address and capacity (rows) of an rt_tensor_desc buffer;
// status_addr: address of a uint8 buffer with len(params) entries.
// Row r of a written tensor gets scalars_idx = scalars_base + (index of its step in the returned list).
// grads: None (every parameter's own .grad), or a list of the gradients to use, None for no gradient.
// centralize: 0, 1 or 2.  Rows get their row_len (adamw.py:179-184: the mean is over every dim but the first, over all
// of them for 0-d / 1-d); with 2 the update takes the means itself where it can; every other row gets its
// place among the means, counted in floats from 1, in row_mean (see place_row_means).
// recorded: the parameters that `states` was made for, in the same order.  A parameter that is another object than the one
// recorded in its place has other states: it is left to the caller.
// A call that fails has changed no step count.
PyObject* gather_group(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 8 && nargs != 10 && nargs != 11) {
        PyErr_SetString(PyExc_TypeError, "gather_group takes 8, 10 or 11 arguments");
        return nullptr;
    }
    PyObject* params = args[0];
    PyObject* states = args[1];
    if (!PyList_CheckExact(params) || !PyList_CheckExact(states)) {
        PyErr_SetString(PyExc_TypeError, "params and states must be lists");
        return nullptr;
    }
    const long dev = PyLong_AsLong(args[2]);
    auto* rows = reinterpret_cast<rt_tensor_desc*>(PyLong_AsUnsignedLongLong(args[3]));
    const Py_ssize_t cap = PyLong_AsSsize_t(args[4]);
    auto* status = reinterpret_cast<uint8_t*>(PyLong_AsUnsignedLongLong(args[5]));
    const unsigned long scalars_base = PyLong_AsUnsignedLong(args[6]);
    const unsigned long id_base = PyLong_AsUnsignedLong(args[7]);
    PyObject* grads = nargs >= 10 && args[8] != Py_None ? args[8] : nullptr;
    const long centralize = nargs >= 10 ? PyLong_AsLong(args[9]) : 0;
    PyObject* recorded = nargs == 11 ? args[10] : nullptr;
    if (PyErr_Occurred()) return nullptr;
    const Py_ssize_t n = PyList_GET_SIZE(params);
    const auto list_of_n = [n](PyObject* o) { return !o || (PyList_CheckExact(o) && PyList_GET_SIZE(o) == n); };
    if (PyList_GET_SIZE(states) != n || !rows || !status || !list_of_n(grads) || !list_of_n(recorded)) {
        PyErr_SetString(PyExc_ValueError, "params / states length mismatch, NULL buffer, or grads / recorded is not a list of that length");
        return nullptr;
    }
    Walk a{params, states, grads, recorded, n, cap, (int)dev, centralize, scalars_base, id_base, rows, status, 0, 0, 0};
    Steps steps;
    std::memset(status, kPython, (size_t)n);
    bool ok = false;
    try {
        ok = walk_group(a, steps);
    } catch (const std::exception& e) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    PyObject* out = nullptr;
    if (ok) {
        PyObject* lst = PyList_New((Py_ssize_t)steps.size());
        for (size_t k = 0; lst && k < steps.size(); ++k) {
            Py_INCREF(steps[k].second);
            PyList_SET_ITEM(lst, (Py_ssize_t)k, steps[k].second);
        }
        if (lst) out = nargs >= 10 ? Py_BuildValue("(nNnK)", a.written, lst, a.left, (unsigned long long)a.means) : Py_BuildValue("(nN)", a.written, lst);
    }
    if (!out) {   // put the step counts back; the error stays set
        PyObject *type, *value, *trace;
        PyErr_Fetch(&type, &value, &trace);
        for (Py_ssize_t k = 0, r = 0; k < n; ++k) {
            if (status[k] != kWritten) continue;
            PyObject* old = PyLong_FromLongLong(steps[rows[r++].scalars_idx - scalars_base].first - 1);
            if (!old || PyDict_SetItem(PyList_GET_ITEM(states, k), k_step, old) != 0) PyErr_Clear();
            Py_XDECREF(old);
        }
        PyErr_Restore(type, value, trace);
    }
    for (auto& s : steps) Py_DECREF(s.second);
    return out;
}

// place_row_means(desc_addr, rows, base_addr): turns the places gather_group left in row_mean into addresses
// in the buffer of means at base_addr.
PyObject* place_row_means(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 3) {
        PyErr_SetString(PyExc_TypeError, "place_row_means takes 3 arguments");
        return nullptr;
    }
    auto* rows = reinterpret_cast<rt_tensor_desc*>(PyLong_AsUnsignedLongLong(args[0]));
    const Py_ssize_t n = PyLong_AsSsize_t(args[1]);
    auto* base = reinterpret_cast<float*>(PyLong_AsUnsignedLongLong(args[2]));
    if (PyErr_Occurred()) return nullptr;
    for (Py_ssize_t r = 0; r < n; ++r)
        if (rows[r].row_mean) rows[r].row_mean = base + (reinterpret_cast<uint64_t>(rows[r].row_mean) - 1);
    Py_RETURN_NONE;
}

// same_objects(flat, lists) -> bool: whether `lists`, one behind the other, hold the very objects of `flat`.
PyObject* same_objects(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 2 || !PyList_CheckExact(args[0]) || !PyList_CheckExact(args[1])) {
        PyErr_SetString(PyExc_TypeError, "same_objects takes a list and a list of lists");
        return nullptr;
    }
    const Py_ssize_t n = PyList_GET_SIZE(args[0]);
    Py_ssize_t at = 0;
    for (Py_ssize_t k = 0; k < PyList_GET_SIZE(args[1]); ++k) {
        PyObject* lst = PyList_GET_ITEM(args[1], k);
        if (!PyList_Check(lst) || PyList_GET_SIZE(lst) > n - at) Py_RETURN_FALSE;
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(lst); ++i)
            if (PyList_GET_ITEM(lst, i) != PyList_GET_ITEM(args[0], at + i)) Py_RETURN_FALSE;
        at += PyList_GET_SIZE(lst);
    }
    return PyBool_FromLong(at == n);
}

// verify_layout(params, expect_addr, n) -> bool
// The cheap per-step check of a frozen layout: params is the flat list of parameters the layout was
// recorded for, expect_addr the address of n triples of uint64 (data pointer of the parameter, data
// pointer of its gradient or 0 for "no gradient", RT_DT_* code of the gradient).  True when every
// parameter is still an exact Tensor / Parameter at the recorded address whose gradient is where it
// was (or still absent), dense, contiguous, of the recorded dtype and of the parameter's size.
// Reads what gather_group reads of a parameter and its gradient, with the same software prefetch,
// and nothing of the states; it changes nothing.
// One contiguous range of the check.  Only reads: object headers, tensor records, storages.
bool verify_range(PyObject* params, const uint64_t* expect, Py_ssize_t lo, Py_ssize_t hi) {
    constexpr Py_ssize_t kAhead = 8;
    constexpr Py_ssize_t kSlots = 4 * kAhead;
    const c10::TensorImpl* pimpl[kSlots] = {};
    auto stage = [&](int level, Py_ssize_t i) {
        if (i < lo || i >= hi) return;
        const Py_ssize_t r = i % kSlots;
        PyObject* po = PyList_GET_ITEM(params, i);
        switch (level) {
            case 0: touch(po); break;
            case 1:
                pimpl[r] = exact_tensor(po) ? THPVariable_Unpack(po).unsafeGetTensorImpl() : nullptr;
                if (pimpl[r]) touch(pimpl[r], 4);
                break;
            case 2:
                if (pimpl[r]) {
                    touch(pimpl[r]->autograd_meta(), 2);
                    touch(pimpl[r]->unsafe_storage().unsafeGetStorageImpl());
                }
                break;
            default:
                if (pimpl[r]) {
                    const at::Tensor& g = THPVariable_Unpack(po).grad();
                    if (g.defined()) touch(g.unsafeGetTensorImpl(), 4);
                }
        }
    };
    for (int level = 0; level < 4; ++level)
        for (Py_ssize_t j = 0; j < (4 - level) * kAhead; ++j) stage(level, lo + j);
    for (Py_ssize_t i = lo; i < hi; ++i) {
        for (int level = 0; level < 4; ++level) stage(level, i + (4 - level) * kAhead);
        PyObject* po = PyList_GET_ITEM(params, i);
        if (!exact_tensor(po)) return false;
        const at::Tensor& p = THPVariable_Unpack(po);
        if (!p.has_storage() || reinterpret_cast<uint64_t>(p.data_ptr()) != expect[3 * i]) return false;
        const at::Tensor& g = p.grad();
        const uint64_t want = expect[3 * i + 1];
        if (!g.defined()) {
            if (want != 0) return false;
            continue;
        }
        if (want == 0 || !ordinary(g.unsafeGetTensorImpl()) || g.layout() != at::kStrided || !g.is_contiguous() || g.numel() != p.numel() ||
            reinterpret_cast<uint64_t>(g.data_ptr()) != want || (uint64_t)grad_code(g.unsafeGetTensorImpl()) != expect[3 * i + 2])
            return false;
    }
    return true;
}

PyObject* verify_layout(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 3) {
        PyErr_SetString(PyExc_TypeError, "verify_layout takes 3 arguments");
        return nullptr;
    }
    PyObject* params = args[0];
    if (!PyList_CheckExact(params)) {
        PyErr_SetString(PyExc_TypeError, "params must be a list");
        return nullptr;
    }
    const auto* expect = reinterpret_cast<const uint64_t*>(PyLong_AsUnsignedLongLong(args[1]));
    const Py_ssize_t n = PyLong_AsSsize_t(args[2]);
    if (PyErr_Occurred()) return nullptr;
    if (PyList_GET_SIZE(params) != n || (n > 0 && !expect)) Py_RETURN_FALSE;
    // The walk is bound by the latency of dependent loads, so long lists are split over a few
    // threads.  The calling thread keeps the interpreter lock throughout: nothing can change the
    // objects while the helpers read them, and the helpers call nothing of the interpreter.
    const Py_ssize_t kPerThread = 2048;
    const int threads = (int)std::min<Py_ssize_t>(8, std::max<Py_ssize_t>(1, n / kPerThread));
    if (threads <= 1) {
        if (verify_range(params, expect, 0, n)) Py_RETURN_TRUE;
        Py_RETURN_FALSE;
    }
    std::vector<char> ok(threads, 0);
    std::vector<std::thread> pool;
    const Py_ssize_t per = (n + threads - 1) / threads;
    for (int t = 1; t < threads; ++t)
        pool.emplace_back([&, t] { ok[t] = verify_range(params, expect, t * per, std::min(n, (t + 1) * per)); });
    ok[0] = verify_range(params, expect, 0, std::min(n, per));
    for (auto& th : pool) th.join();
    for (char c : ok)
        if (!c) Py_RETURN_FALSE;
    Py_RETURN_TRUE;
}

// dict_versions(dicts, out_addr, n) / verify_versions(dicts, expect_addr, n) -> bool
// A recorded layout keeps the addresses of the two state tensors of every parameter and does not
// read the state dicts again while it is in use, so nothing else may change them either.  CPython
// stamps every dict with a version that changes whenever the dict is modified (ma_version_tag);
// dict_versions writes the stamps of n dicts as uint64 to out_addr, verify_versions compares them:
// a state tensor that was replaced, removed or added shows as a changed stamp, for one load per
// dict.  (Interpreters without the stamp, 3.12 and later: dict_versions fails and no layout is recorded.)
PyObject* dict_versions(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
#if PY_VERSION_HEX >= 0x030C0000
    PyErr_SetString(PyExc_NotImplementedError, "this interpreter's dicts carry no version stamp");
    return nullptr;
#else
    if (nargs != 3 || !PyList_CheckExact(args[0])) {
        PyErr_SetString(PyExc_TypeError, "dict_versions(list, address, n)");
        return nullptr;
    }
    auto* out = reinterpret_cast<uint64_t*>(PyLong_AsUnsignedLongLong(args[1]));
    const Py_ssize_t n = PyLong_AsSsize_t(args[2]);
    if (PyErr_Occurred()) return nullptr;
    if (PyList_GET_SIZE(args[0]) != n || (n > 0 && !out)) {
        PyErr_SetString(PyExc_ValueError, "list length and n differ");
        return nullptr;
    }
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* d = PyList_GET_ITEM(args[0], i);
        if (!PyDict_Check(d)) {
            PyErr_SetString(PyExc_TypeError, "not a dict");
            return nullptr;
        }
        out[i] = reinterpret_cast<PyDictObject*>(d)->ma_version_tag;
    }
    Py_RETURN_NONE;
#endif
}

PyObject* verify_versions(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
#if PY_VERSION_HEX >= 0x030C0000
    Py_RETURN_FALSE;
#else
    if (nargs != 3 || !PyList_CheckExact(args[0])) {
        PyErr_SetString(PyExc_TypeError, "verify_versions(list, address, n)");
        return nullptr;
    }
    const auto* expect = reinterpret_cast<const uint64_t*>(PyLong_AsUnsignedLongLong(args[1]));
    const Py_ssize_t n = PyLong_AsSsize_t(args[2]);
    if (PyErr_Occurred()) return nullptr;
    if (PyList_GET_SIZE(args[0]) != n || (n > 0 && !expect)) Py_RETURN_FALSE;
    constexpr Py_ssize_t kAhead = 16;
    for (Py_ssize_t i = 0; i < n; ++i) {
        if (i + kAhead < n) touch(PyList_GET_ITEM(args[0], i + kAhead));
        PyObject* d = PyList_GET_ITEM(args[0], i);
        if (!PyDict_Check(d) || reinterpret_cast<PyDictObject*>(d)->ma_version_tag != expect[i]) Py_RETURN_FALSE;
    }
    Py_RETURN_TRUE;
#endif
}

// set_types(torch.Tensor, torch.nn.Parameter): only objects of exactly these types take the fast path.
PyObject* set_types(PyObject*, PyObject* args) {
    PyObject *a = nullptr, *b = nullptr;
    if (!PyArg_ParseTuple(args, "OO", &a, &b)) return nullptr;
    if (!PyType_Check(a) || !PyType_Check(b)) {
        PyErr_SetString(PyExc_TypeError, "expected two types");
        return nullptr;
    }
    Py_INCREF(a);
    Py_INCREF(b);
    t_tensor = reinterpret_cast<PyTypeObject*>(a);
    t_parameter = reinterpret_cast<PyTypeObject*>(b);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"gather_group", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(gather_group)), METH_FASTCALL,
     "rt_tensor_desc rows of the plain tensors of one param group"},
    {"place_row_means", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(place_row_means)), METH_FASTCALL,
     "addresses of the row means of gathered rows"},
    {"same_objects", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(same_objects)), METH_FASTCALL,
     "whether some lists hold the very objects of another"},
    {"verify_layout", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(verify_layout)), METH_FASTCALL,
     "whether every parameter and gradient of a recorded layout is still where it was"},
    {"dict_versions", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(dict_versions)), METH_FASTCALL,
     "modification stamps of a list of dicts"},
    {"verify_versions", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(verify_versions)), METH_FASTCALL,
     "whether none of the dicts has been modified since dict_versions"},
    {"set_types", set_types, METH_VARARGS, "register torch.Tensor and torch.nn.Parameter"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef moddef = {PyModuleDef_HEAD_INIT, "_rt_gather", "descriptor gathering for ramtorch_amd.AdamW", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__rt_gather(void) {
    k_ema = PyUnicode_InternFromString("ema");
    k_ema_squared = PyUnicode_InternFromString("ema_squared");
    k_step = PyUnicode_InternFromString("step");
    if (!k_ema || !k_ema_squared || !k_step) return nullptr;
    h_ema = PyObject_Hash(k_ema);
    h_ema_squared = PyObject_Hash(k_ema_squared);
    h_step = PyObject_Hash(k_step);
    PyObject* m = PyModule_Create(&moddef);
    if (!m) return nullptr;
    PyModule_AddIntConstant(m, "DESC_SIZE", (long)sizeof(rt_tensor_desc));
    PyModule_AddIntConstant(m, "WRITTEN", kWritten);
    PyModule_AddIntConstant(m, "NO_GRAD", kNoGrad);
    PyModule_AddIntConstant(m, "PYTHON", kPython);
    return m;
}
