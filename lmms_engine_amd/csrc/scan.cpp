// What the optimizer step and gradient clipping read off every tensor of a list - device, dtype, shape, whether its rows are contiguous,
// its address - in native code: in Python that is 0.9 us for a gradient and 1.3 us for a parameter with its momentum, 860 us for the
// 392 matrices of a low-rank set whose kernels take 310.
//
// Each function takes lists in which nothing needs a decision: plain parameters on one kind of device with plain contiguous
// gradients and state.  Anything else (a missing gradient or state, a CPU tensor, other strides, a subclass such as DTensor, an
// empty tensor) makes it return None before it has changed anything, and the caller goes through the list itself.
//
// What a function returns are addresses.  Given a list as `held`, it appends an object to it that keeps the memory behind them alive: the
// caller's launches give up the interpreter lock, and another thread may drop a gradient there.  The caller lets go after the last
// launch that uses the addresses (9 ns a tensor; memory that a kernel on the stream still reads is the allocator's affair, as ever).
#define PY_SSIZE_T_CLEAN
#include <torch/csrc/autograd/python_variable.h>

#include <memory>
#include <string>
#include <unordered_set>
#include <vector>

namespace {

// A dtype code of the C ABI for a tensor that the kernels read as it lies; -1 for any other.
int plain(const at::Tensor& t) {
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.is_neg() || t.unsafeGetTensorImpl()->is_python_dispatch()) return -1;
    const int code = t.scalar_type() == at::kFloat ? 0 : t.scalar_type() == at::kBFloat16 ? 1 : -1;
    return code >= 0 && t.numel() > 0 && t.is_contiguous() ? code : -1;
}
int plain_object(PyObject* o) { return o && THPVariable_CheckExact(o) ? plain(THPVariable_Unpack(o)) : -1; }

PyObject* none() {
    if (PyErr_Occurred()) PyErr_Clear();  // a look-up that raised: the caller's own loop raises it again
    Py_RETURN_NONE;
}

// The storages of tensors whose addresses a function hands out.
using Held = std::vector<c10::Storage>;
void let_go(PyObject* capsule) { delete (Held*)PyCapsule_GetPointer(capsule, nullptr); }
// Appends them to the caller's list (null: the caller holds the tensors himself); false with an exception set.
bool hand_over(PyObject* list, std::unique_ptr<Held> held) {
    if (!list) return true;
    PyObject* capsule = PyCapsule_New(held.get(), nullptr, let_go);
    if (!capsule) return false;
    (void)held.release();
    const bool ok = PyList_Append(list, capsule) == 0;
    Py_DECREF(capsule);
    return ok;
}
bool is_holder(PyObject* list) { return !list || PyList_CheckExact(list); }

// state[p][key], borrowed; null if there is no such thing in plain dictionaries
PyObject* state_of(PyObject* state, PyObject* p) {
    PyObject* s = PyDict_GetItemWithError(state, p);
    return s && PyDict_CheckExact(s) ? s : nullptr;
}
PyObject* key_momentum;
PyObject* key_exp_avg;
PyObject* key_exp_avg_sq;
PyObject* key_step;

void put(std::string& s, long long v) { s.append((const char*)&v, sizeof v); }
// The rows of a tensor list's table behind the pointers: element counts, and the first chunk of every tensor with the total behind
// them (include/muon_hip.h, multi-tensor kernels).  Returns the chunks.
long long put_sizes(std::string& words, const std::vector<long long>& numel, long long chunk) {
    for (long long n : numel) put(words, n);
    long long at = 0;
    for (long long n : numel) {
        put(words, at);
        at += (n + chunk - 1) / chunk;
    }
    put(words, at);
    return at;
}

// grads(params, chunk, held = nothing): (device index, [(dtype code, tensors, chunks, table words)]) of the gradients that there are, by dtype in the
// order of their first gradient.
PyObject* grads(PyObject*, PyObject* args) {
    PyObject *params, *held_list = nullptr;
    long long chunk;
    if (!PyArg_ParseTuple(args, "OL|O", &params, &chunk, &held_list)) return nullptr;
    auto held = std::make_unique<Held>();
    if (!PyList_CheckExact(params) || !is_holder(held_list) || chunk < 1) return none();
    struct Group {
        int code;
        std::string ptrs;
        std::vector<long long> numel;
    };
    std::vector<Group> groups;
    int device = -1;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(params); ++i) {
        PyObject* o = PyList_GET_ITEM(params, i);
        if (!THPVariable_CheckExact(o)) return none();
        const at::Tensor& p = THPVariable_Unpack(o);
        if (!p.is_leaf()) return none();
        const at::Tensor& g = p.grad();
        if (!g.defined()) continue;
        const int code = plain(g);
        if (code < 0 || (device >= 0 && g.get_device() != device)) return none();
        device = (int)g.get_device();
        size_t k = 0;
        while (k < groups.size() && groups[k].code != code) ++k;
        if (k == groups.size()) groups.push_back(Group{code, {}, {}});
        put(groups[k].ptrs, (long long)g.data_ptr());
        groups[k].numel.push_back(g.numel());
        if (held_list) held->push_back(g.storage());
    }
    if (groups.empty()) return none();
    if (!hand_over(held_list, std::move(held))) return nullptr;
    PyObject* list = PyList_New(0);
    if (!list) return nullptr;
    for (Group& g : groups) {
        const long long chunks = put_sizes(g.ptrs, g.numel, chunk);
        PyObject* item = Py_BuildValue("(inLN)", g.code, (Py_ssize_t)g.numel.size(), chunks, PyByteArray_FromStringAndSize(g.ptrs.data(), (Py_ssize_t)g.ptrs.size()));
        if (!item || PyList_Append(list, item) < 0) {
            Py_XDECREF(item);
            Py_DECREF(list);
            return nullptr;
        }
        Py_DECREF(item);
    }
    return Py_BuildValue("(iN)", device, list);
}

// muon(params, state, held = nothing): [(device index, rows, cols, parameter, gradient and momentum dtype codes, matrices, their addresses)] by shape and
// dtypes, in the order of their first parameter; the addresses as three strings of 64-bit words.
PyObject* muon(PyObject*, PyObject* args) {
    PyObject *params, *state, *held_list = nullptr;
    if (!PyArg_ParseTuple(args, "OO|O", &params, &state, &held_list)) return nullptr;
    auto held = std::make_unique<Held>();
    if (!PyList_CheckExact(params) || !PyDict_Check(state) || !is_holder(held_list)) return none();
    struct Bucket {
        int device, codes[3];
        long long rows, cols, n;
        std::string ptrs[3];
    };
    std::vector<Bucket> buckets;
    size_t last = 0;
    for (Py_ssize_t i = 0; i < PyList_GET_SIZE(params); ++i) {
        PyObject* o = PyList_GET_ITEM(params, i);
        const int pc = plain_object(o);
        if (pc < 0) return none();
        const at::Tensor& p = THPVariable_Unpack(o);
        if (p.dim() != 2 || !p.is_leaf()) return none();
        const at::Tensor& g = p.grad();
        const int gc = plain(g);
        if (gc < 0) return none();
        PyObject* s = state_of(state, o);
        PyObject* mo = s ? PyDict_GetItemWithError(s, key_momentum) : nullptr;
        const int mc = plain_object(mo);
        if (mc < 0) return none();
        const at::Tensor& m = THPVariable_Unpack(mo);
        const int device = (int)p.get_device();
        if (g.get_device() != device || m.get_device() != device || g.sizes() != p.sizes() || m.sizes() != p.sizes()) return none();
        const long long rows = p.size(0), cols = p.size(1);
        auto same = [&](const Bucket& b) {
            return b.rows == rows && b.cols == cols && b.device == device && b.codes[0] == pc && b.codes[1] == gc && b.codes[2] == mc;
        };
        size_t k = last;
        if (k >= buckets.size() || !same(buckets[k]))
            for (k = 0; k < buckets.size() && !same(buckets[k]);) ++k;
        if (k == buckets.size()) buckets.push_back(Bucket{device, {pc, gc, mc}, rows, cols, 0, {}});
        last = k;
        Bucket& b = buckets[k];
        ++b.n;
        put(b.ptrs[0], (long long)p.data_ptr());
        put(b.ptrs[1], (long long)g.data_ptr());
        put(b.ptrs[2], (long long)m.data_ptr());
        if (held_list)
            for (const at::Tensor* t : {&p, &g, &m}) held->push_back(t->storage());
    }
    if (!hand_over(held_list, std::move(held))) return nullptr;
    PyObject* list = PyList_New((Py_ssize_t)buckets.size());
    if (!list) return nullptr;
    for (size_t k = 0; k < buckets.size(); ++k) {
        const Bucket& b = buckets[k];
        PyObject* item = Py_BuildValue("(iLLiiiLy#y#y#)", b.device, b.rows, b.cols, b.codes[0], b.codes[1], b.codes[2], b.n, b.ptrs[0].data(),
                                       (Py_ssize_t)b.ptrs[0].size(), b.ptrs[1].data(), (Py_ssize_t)b.ptrs[1].size(), b.ptrs[2].data(),
                                       (Py_ssize_t)b.ptrs[2].size());
        if (!item) {
            Py_DECREF(list);
            return nullptr;
        }
        PyList_SET_ITEM(list, (Py_ssize_t)k, item);
    }
    return list;
}

// adam(params, state, chunk, held = nothing): (device index, dtype code, steps, chunks, table words) of parameters of one device and dtype; every step count
// is one higher afterwards.
PyObject* adam(PyObject*, PyObject* args) {
    PyObject *params, *state, *held_list = nullptr;
    long long chunk;
    if (!PyArg_ParseTuple(args, "OOL|O", &params, &state, &chunk, &held_list)) return nullptr;
    auto held = std::make_unique<Held>();
    if (!PyList_CheckExact(params) || !PyDict_Check(state) || !is_holder(held_list) || chunk < 1) return none();
    const Py_ssize_t n = PyList_GET_SIZE(params);
    if (n == 0) return none();
    int device = -1, code = -1;
    std::string ptrs[4];
    std::vector<long long> numel, steps;
    std::vector<PyObject*> states;
    std::unordered_set<PyObject*> seen;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* o = PyList_GET_ITEM(params, i);
        const int pc = plain_object(o);
        if (pc < 0) return none();
        const at::Tensor& p = THPVariable_Unpack(o);
        if (!p.is_leaf()) return none();
        if (i == 0) device = (int)p.get_device(), code = pc;
        PyObject* s = state_of(state, o);
        if (!s) return none();
        PyObject* moments[2] = {PyDict_GetItemWithError(s, key_exp_avg), PyDict_GetItemWithError(s, key_exp_avg_sq)};
        PyObject* step = PyDict_GetItemWithError(s, key_step);
        if (!step || !PyLong_CheckExact(step)) return none();
        const long long count = PyLong_AsLongLong(step);
        if (count < 0 || count > (1LL << 52)) return none();
        const at::Tensor* t[4] = {&p, &p.grad(), nullptr, nullptr};
        for (int k : {0, 1}) {
            if (plain_object(moments[k]) < 0) return none();
            t[2 + k] = &THPVariable_Unpack(moments[k]);
        }
        for (int k = 0; k < 4; ++k) {
            if (plain(*t[k]) != code || t[k]->get_device() != device || t[k]->numel() != p.numel()) return none();
            put(ptrs[k], (long long)t[k]->data_ptr());
            if (held_list) held->push_back(t[k]->storage());
        }
        if (!seen.insert(s).second) return none();  // a parameter that is listed twice steps twice
        numel.push_back(p.numel());
        steps.push_back(count + 1);
        states.push_back(s);
    }
    std::string words = ptrs[0] + ptrs[1] + ptrs[2] + ptrs[3];
    const long long chunks = put_sizes(words, numel, chunk);
    if (!hand_over(held_list, std::move(held))) return nullptr;
    PyObject* list = PyList_New(n);
    if (!list) return nullptr;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* v = PyLong_FromLongLong(steps[i]);
        if (!v || PyDict_SetItem(states[i], key_step, v) < 0) {
            Py_XDECREF(v);
            Py_DECREF(list);
            return nullptr;
        }
        PyList_SET_ITEM(list, i, v);
    }
    return Py_BuildValue("(iiNLN)", device, code, list, chunks, PyByteArray_FromStringAndSize(words.data(), (Py_ssize_t)words.size()));
}

// A tensor that raises when it is asked is one that the caller's loop has to deal with (nothing has been changed by then: `adam` asks
// no tensor after its first change).
template <PyObject* (*F)(PyObject*, PyObject*)>
PyObject* guarded(PyObject* self, PyObject* args) {
    try {
        return F(self, args);
    } catch (...) {
        return none();
    }
}

PyMethodDef methods[] = {{"grads", guarded<grads>, METH_VARARGS, nullptr},
                         {"muon", guarded<muon>, METH_VARARGS, nullptr},
                         {"adam", guarded<adam>, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_scan", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__scan() {
    key_momentum = PyUnicode_InternFromString("momentum_buffer");
    key_exp_avg = PyUnicode_InternFromString("exp_avg");
    key_exp_avg_sq = PyUnicode_InternFromString("exp_avg_sq");
    key_step = PyUnicode_InternFromString("step");
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", SCAN_TORCH_VERSION) < 0) Py_CLEAR(m);
    return m;
}
