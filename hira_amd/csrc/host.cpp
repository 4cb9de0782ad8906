// The host side of the calls that a decode step makes of this package, in one step each: what their Python bodies ask of
// the tensors (types, shapes, device, contiguity, alignment), the C structs, the library call.  A call takes 20 to 60
// such questions, 50 to 100 ns each from Python and a few from here, and its launches are no longer than that.
//
// Every function here takes exactly the form that a running program's calls have (plain tensors of the storage type, on the
// index's device, contiguous) and answers None to any other, before it has changed anything: the Python body, which
// converts or refuses, then has its turn.  Nothing is kept between calls; the addresses that come in are those of
// structs and tensors that the caller holds.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/Generator.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/core/Tensor.h>
#include <ATen/CPUGeneratorImpl.h>
#include <ATen/core/DistributionsHelper.h>
#include <ATen/ops/empty.h>

#include <mutex>
#include <unordered_map>
#include <utility>
#include <vector>

#include "../../include/hira_hip.h"

namespace {

// the library that hira_amd/_lib.py has loaded
struct Library {
    decltype(&hira_enqueue) enqueue;
    decltype(&hira_search) search;
    decltype(&hira_search_sampled) search_sampled;
    decltype(&hira_update_sample) update_sample;
    decltype(&hira_read_state) read_state;
} lib;

// A tensor with memory of its own on device `dev` and nothing that would have a say in how it is read; NULL otherwise.
const at::Tensor* plain(PyObject* o, int64_t dev) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.get_device() != dev || t.layout() != c10::kStrided || at::isTensorSubclassLike(t) ||
        t.is_conj() || t.is_neg() || !t.is_contiguous())
        return nullptr;
    return &t;
}

int type_of(const at::Tensor& t) {
    return t.scalar_type() == at::kFloat ? (int)HIRA_F32 : t.scalar_type() == at::kBFloat16 ? (int)HIRA_BF16 : -1;
}

// One whose rows the kernels read in 16-byte chunks: a contiguous view may start between two of them.
const at::Tensor* in_chunks(PyObject* o, int64_t dev) {
    const at::Tensor* t = plain(o, dev);
    return t != nullptr && reinterpret_cast<uintptr_t>(t->data_ptr()) % 16 == 0 ? t : nullptr;
}

int64_t number(PyObject* o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
}
void* address(PyObject* o) {
    if (o == Py_None) return nullptr;
    void* p = PyLong_AsVoidPtr(o);
    if (p == nullptr && PyErr_Occurred()) throw python_error();
    return p;
}

bool arguments(const char* name, Py_ssize_t have, Py_ssize_t want) {
    if (have == want) return true;
    PyErr_Format(PyExc_TypeError, "%s: %zd arguments, expected %zd", name, have, want);
    return false;
}

// (the library waits for nothing here, but a full queue of launches may make it)
template <typename F>
int without_gil(F f) {
    PyThreadState* state = PyEval_SaveThread();
    const int rc = f();
    PyEval_RestoreThread(state);
    return rc;
}

// bind({name: address})
PyObject* bind(PyObject*, PyObject* functions) {
    HANDLE_TH_ERRORS
    auto get = [&](const char* name) {
        PyObject* o = PyDict_GetItemString(functions, name);
        if (o == nullptr) throw c10::TypeError({__func__, __FILE__, (uint32_t)__LINE__}, std::string("no address of ") + name);
        return address(o);
    };
    lib.enqueue = reinterpret_cast<decltype(lib.enqueue)>(get("hira_enqueue"));
    lib.search = reinterpret_cast<decltype(lib.search)>(get("hira_search"));
    lib.search_sampled = reinterpret_cast<decltype(lib.search_sampled)>(get("hira_search_sampled"));
    lib.update_sample = reinterpret_cast<decltype(lib.update_sample)>(get("hira_update_sample"));
    lib.read_state = reinterpret_cast<decltype(lib.read_state)>(get("hira_read_state"));
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// enqueue(queue_keys (B, H, cap, D), queue_values (B, H, cap, Dv), keys (B, H, 1, D), values (B, H, 1, Dv), at, dev, stream):
// a token's rows into place `at` of every head's queue.  The library's return code.
PyObject* enqueue(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!arguments("enqueue", n, 7)) return nullptr;
    const int64_t at = number(a[4]), dev = number(a[5]);
    const at::Tensor *qk = in_chunks(a[0], dev), *qv = in_chunks(a[1], dev), *k = in_chunks(a[2], dev), *v = in_chunks(a[3], dev);
    if (!qk || !qv || !k || !v || qk->dim() != 4 || qv->dim() != 4 || k->dim() != 4 || v->dim() != 4) Py_RETURN_NONE;
    const int type = type_of(*qk);
    if (type < 0 || type_of(*qv) != type || type_of(*k) != type || type_of(*v) != type) Py_RETURN_NONE;
    const int64_t b = qk->size(0), h = qk->size(1), cap = qk->size(2), d = qk->size(3), dv = qv->size(3);
    if (at < 0 || at >= cap || qv->size(0) != b || qv->size(1) != h || qv->size(2) != cap || k->size(0) != b || k->size(1) != h ||
        k->size(2) != 1 || k->size(3) != d || v->size(0) != b || v->size(1) != h || v->size(2) != 1 || v->size(3) != dv)
        Py_RETURN_NONE;
    const int64_t e = type == HIRA_F32 ? 4 : 2;
    void *qkp = qk->data_ptr(), *qvp = qv->data_ptr(), *kp = k->data_ptr(), *vp = v->data_ptr();
    if (d * e % 16 || dv * e % 16 || b * h > INT32_MAX) Py_RETURN_NONE;
    void* stream = address(a[6]);
    return PyLong_FromLong(without_gil([&] {
        return lib.enqueue(qkp, qvp, type, (int32_t)(b * h), (int32_t)cap, (int32_t)at, 1, (int32_t)d, (int32_t)dv, kp, vp, stream);
    }));
    END_HANDLE_TH_ERRORS
}

// attend((tree, query, sample, queue, out, launch, dev, workspace, bytes of it, queue rows it is for), thresholds (H_q), query
// (B, H_q, 1, D), samples (T, S, D), queue_keys, queue_values (..., cap, D / Dv), rows in use, rule, k, stream): a decode step whose
// thresholds come from a key sample (DecodePlan.run_sampled).  The output (B, 1, H_q, Dv) in the query's type, or the
// library's return code where that is an error.
PyObject* attend(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!arguments("attend", n, 10)) return nullptr;
    if (!PyTuple_CheckExact(a[0]) || PyTuple_GET_SIZE(a[0]) != 10 || !PyLong_CheckExact(a[6]) || !PyLong_CheckExact(a[8])) Py_RETURN_NONE;
    auto part = [&](int i) { return PyTuple_GET_ITEM(a[0], i); };
    const HiraTree* tree = static_cast<const HiraTree*>(address(part(0)));
    HiraQuery* query = static_cast<HiraQuery*>(address(part(1)));
    HiraSample* sample = static_cast<HiraSample*>(address(part(2)));
    HiraQueue* queue = static_cast<HiraQueue*>(address(part(3)));
    HiraSearchOut* out = static_cast<HiraSearchOut*>(address(part(4)));
    const HiraLaunch* launch = static_cast<const HiraLaunch*>(address(part(5)));
    const int64_t dev = number(part(6)), bytes = number(part(8)), rows = number(a[6]), rule = number(a[7]), k = number(a[8]);
    const at::Tensor *ws = plain(part(7), dev), *tau = plain(a[1], dev), *q = in_chunks(a[2], dev), *s = in_chunks(a[3], dev);
    if (!ws || !tau || !q || !s || q->dim() != 4 || s->dim() != 3 || type_of(*q) != tree->dtype || type_of(*s) != tree->dtype ||
        ws->scalar_type() != at::kByte || ws->numel() < bytes || tau->scalar_type() != at::kFloat)
        Py_RETURN_NONE;
    const int64_t b = q->size(0), h = q->size(1);
    if (b * h != query->num_q_heads || tau->numel() < b * h || q->size(2) != 1 || q->size(3) != tree->dim || s->size(0) != tree->num_trees ||
        s->size(2) != tree->dim || s->size(1) > INT32_MAX || k < INT32_MIN || k > INT32_MAX)
        Py_RETURN_NONE;
    const at::Tensor *qk = nullptr, *qv = nullptr;
    int64_t cap = 0;
    if (rows != 0) {
        qk = in_chunks(a[4], dev), qv = in_chunks(a[5], dev);
        if (!qk || !qv || qk->dim() < 2 || qv->dim() < 2 || type_of(*qk) != tree->dtype || type_of(*qv) != tree->dtype) Py_RETURN_NONE;
        cap = qk->size(-2);
        if (rows < 0 || rows > cap || rows > number(part(9)) || cap > INT32_MAX || qv->size(-2) != cap || qk->size(-1) != tree->dim ||
            qv->size(-1) != tree->vdim || qk->numel() != tree->num_trees * cap * tree->dim || qv->numel() != tree->num_trees * cap * tree->vdim)
            Py_RETURN_NONE;
    }
    at::Tensor result = at::empty({b, 1, h, tree->vdim}, q->options());
    query->q = q->data_ptr();
    query->out_dtype = tree->dtype;
    out->attn_out = static_cast<float*>(result.data_ptr());
    if (rows != 0) *queue = HiraQueue{qk->data_ptr(), qv->data_ptr(), (int32_t)rows, (int32_t)cap};
    sample->rows = s->data_ptr();
    sample->num_rows = (int32_t)s->size(1);
    sample->method = (int32_t)rule;
    sample->k = (int32_t)k;
    sample->tau = tau->mutable_data_ptr<float>();
    void *workspace = ws->data_ptr(), *stream = address(a[9]);
    const int rc = without_gil([&] {
        return lib.search_sampled(tree, query, sample, rows != 0 ? queue : nullptr, out, launch, workspace, (size_t)bytes, stream);
    });
    if (rc != HIRA_OK) return PyLong_FromLong(rc);
    return THPVariable_Wrap(std::move(result));
    END_HANDLE_TH_ERRORS
}

// search((tree, query, out, heads, dev, ones), launch, query (H_q, D) or (B, H_q, 1, D), thresholds (H_q), scaling (H_q) or None,
// dense (H_q, n), fill value, stream): HIPSearcher.search in the slots' index space.  The library's return code.
PyObject* search(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!arguments("search", n, 8)) return nullptr;
    if (!PyTuple_CheckExact(a[0]) || PyTuple_GET_SIZE(a[0]) != 6) Py_RETURN_NONE;
    auto part = [&](int i) { return PyTuple_GET_ITEM(a[0], i); };
    const HiraTree* tree = static_cast<const HiraTree*>(address(part(0)));
    HiraQuery* query = static_cast<HiraQuery*>(address(part(1)));
    HiraSearchOut* out = static_cast<HiraSearchOut*>(address(part(2)));
    const int64_t heads = number(part(3)), dev = number(part(4));
    const float* scale = static_cast<const float*>(address(part(5)));
    const at::Tensor *q = in_chunks(a[2], dev), *tau = plain(a[3], dev), *dense = plain(a[5], dev);
    if (!q || !tau || !dense || type_of(*q) != tree->dtype || !(q->dim() == 2 || (q->dim() == 4 && q->size(2) == 1)) ||
        q->size(-1) != tree->dim || q->numel() != heads * tree->dim || tau->scalar_type() != at::kFloat || tau->numel() != heads ||
        dense->scalar_type() != at::kFloat || dense->dim() != 2 || dense->size(0) != heads || dense->size(1) != tree->size[0])
        Py_RETURN_NONE;
    if (a[4] != Py_None) {
        const at::Tensor* s = plain(a[4], dev);
        if (!s || s->scalar_type() != at::kFloat || s->numel() != heads) Py_RETURN_NONE;
        scale = s->const_data_ptr<float>();
    }
    if (scale == nullptr) Py_RETURN_NONE;
    const double fill = PyFloat_AsDouble(a[6]);
    if (fill == -1.0 && PyErr_Occurred()) throw python_error();
    query->q = q->data_ptr();
    query->tau = tau->const_data_ptr<float>();
    query->scaling = scale;
    *out = HiraSearchOut{};
    out->dense = dense->mutable_data_ptr<float>();
    out->dense_stride = tree->size[0];
    out->dense_fill = 1;
    out->dense_fill_value = (float)fill;
    const HiraLaunch* launch = static_cast<const HiraLaunch*>(address(a[1]));
    void* stream = address(a[7]);
    return PyLong_FromLong(without_gil([&] { return lib.search(tree, query, nullptr, out, launch, nullptr, 0, stream); }));
    END_HANDLE_TH_ERRORS
}

// append(tree, keys (..., m, D) of its trees, values (..., m, Dv) or None, m, state, sample rows (T, S, D) or None, slots, which, dev,
// stream, pinned rows or None, ticket): HIPIndexer.update's launch and, into the rows, its read-back of the level sizes.  A list of their largest
// entries over the trees where it read them back, else the library's return code (less kAppended: that of the read-back, behind an
// append that was launched).
constexpr int kAppended = 100;
PyObject* append(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!arguments("append", n, 12)) return nullptr;
    const HiraTree* tree = static_cast<const HiraTree*>(address(a[0]));
    const int64_t m = number(a[3]), dev = number(a[8]);
    const at::Tensor *k = in_chunks(a[1], dev), *v = nullptr, *s = nullptr;
    if (!k || type_of(*k) != tree->dtype || m < 0 || m > INT32_MAX || k->numel() != tree->num_trees * m * tree->dim) Py_RETURN_NONE;
    if (a[2] != Py_None) {
        v = in_chunks(a[2], dev);
        if (!v || type_of(*v) != tree->dtype || v->numel() != tree->num_trees * m * tree->vdim) Py_RETURN_NONE;
    }
    std::vector<int32_t> pairs;
    int64_t count = 0;
    if (a[5] != Py_None) {
        s = in_chunks(a[5], dev);
        if (!s || s->dim() != 3 || type_of(*s) != tree->dtype || s->size(0) != tree->num_trees || s->size(2) != tree->dim ||
            s->size(1) > INT32_MAX || !PyTuple_CheckExact(a[6]) || !PyTuple_CheckExact(a[7]) ||
            PyTuple_GET_SIZE(a[6]) != PyTuple_GET_SIZE(a[7]))
            Py_RETURN_NONE;
        count = PyTuple_GET_SIZE(a[6]);
        pairs.reserve(2 * count);
        for (int half = 6; half <= 7; ++half)
            for (int64_t i = 0; i < count; ++i) {
                PyObject* o = PyTuple_GET_ITEM(a[half], i);
                int overflow = 0;
                const long long x = PyLong_CheckExact(o) ? PyLong_AsLongLongAndOverflow(o, &overflow) : -1;
                if (!PyLong_CheckExact(o) || overflow || x < INT32_MIN || x > INT32_MAX) Py_RETURN_NONE;
                pairs.push_back((int32_t)x);
            }
    }
    int32_t* state = static_cast<int32_t*>(address(a[4]));
    void* stream = address(a[9]);
    constexpr int kColumns = HIRA_MAX_LEVELS + 2;
    uint64_t* rows = nullptr;
    if (a[10] != Py_None) {
        if (!THPVariable_CheckExact(a[10])) Py_RETURN_NONE;
        const at::Tensor& r = THPVariable_Unpack(a[10]);
        if (!r.is_cpu() || at::isTensorSubclassLike(r) || r.scalar_type() != at::kLong || !r.is_contiguous() ||
            r.numel() != (int64_t)tree->num_trees * kColumns)
            Py_RETURN_NONE;
        rows = static_cast<uint64_t*>(r.data_ptr());
    }
    const uint32_t ticket = (uint32_t)number(a[11]);
    int32_t most[kColumns];
    const void *kp = k->data_ptr(), *vp = v ? v->data_ptr() : nullptr;
    void* sp = count ? s->data_ptr() : nullptr;
    const int32_t per_tree = count ? (int32_t)s->size(1) : 0, *slots = count ? pairs.data() : nullptr;
    const int rc = without_gil([&] {
        const int rc = lib.update_sample(tree, kp, vp, (int32_t)m, state, sp, per_tree, slots, slots ? slots + count : nullptr, (int32_t)count, stream);
        if (rc != HIRA_OK || rows == nullptr) return rc;
        const int back = lib.read_state(tree, state, rows, ticket, most, stream);
        return back != HIRA_OK ? back - kAppended : HIRA_OK;
    });
    if (rc != HIRA_OK || rows == nullptr) return PyLong_FromLong(rc);
    THPObjectPtr list(PyList_New(kColumns));
    if (!list) throw python_error();
    for (int i = 0; i < kColumns; ++i) PyList_SET_ITEM(list.get(), i, PyLong_FromLong(most[i]));
    return list.release();
    END_HANDLE_TH_ERRORS
}

// draw(generator, m, first, members, seen): reservoir sampling (HiraCacheLayer._sample_pairs): of m new keys, the first of them number
// `first` of its call and number `seen` of the sequence, key i joins a sample of `members` with probability members / (seen + i + 1) in place of
// a random member.  (members replaced, by which keys): a member drawn twice keeps its last arrival.
PyObject* draw(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (!arguments("draw", n, 5)) return nullptr;
    if (!THPGenerator_Check(a[0])) {
        PyErr_SetString(PyExc_TypeError, "draw: not a generator");
        return nullptr;
    }
    // (the numbers of torch.rand(m) and torch.randint(members, (k,)) on this generator)
    at::CPUGeneratorImpl* g = at::check_generator<at::CPUGeneratorImpl>(THPGenerator_Unwrap(a[0]));
    const int64_t m = number(a[1]), first = number(a[2]), members = number(a[3]), seen = number(a[4]);
    if (members <= 0 || members > INT32_MAX / 16) {
        PyErr_Format(PyExc_ValueError, "draw: a sample of %lld members", (long long)members);
        return nullptr;
    }
    const at::ScalarType type = c10::get_default_dtype_as_scalartype();
    std::vector<int64_t> who;
    std::vector<std::pair<int64_t, int64_t>> pairs;
    {
        std::lock_guard<std::mutex> lock(g->mutex_);
        auto shares = [&](auto zero) {
            using Share = decltype(zero);
            at::uniform_real_distribution<Share> share(0, 1);
            for (int64_t i = 0; i < m; ++i)
                if ((double)static_cast<Share>(share(g)) < (double)members / (double)(seen + i + 1)) who.push_back(first + i);
        };
        // (torch.rand's type is the default type, which a program that loads a model in 16 bits may have set to that)
        if (type == at::kDouble) shares(double());
        else if (type == at::kBFloat16) shares(at::BFloat16());
        else if (type == at::kHalf) shares(at::Half());
        else shares(float());
        at::uniform_int_from_to_distribution<int64_t> member(members, 0);
        std::unordered_map<int64_t, size_t> place;
        for (const int64_t key : who) {
            const int64_t slot = member(g);
            const auto [it, fresh] = place.try_emplace(slot, pairs.size());
            if (fresh) pairs.emplace_back(slot, key);
            else pairs[it->second].second = key;
        }
    }
    THPObjectPtr slot(PyTuple_New(pairs.size())), which(PyTuple_New(pairs.size()));
    if (!slot || !which) throw python_error();
    for (size_t i = 0; i < pairs.size(); ++i) {
        PyTuple_SET_ITEM(slot.get(), i, PyLong_FromLongLong(pairs[i].first));
        PyTuple_SET_ITEM(which.get(), i, PyLong_FromLongLong(pairs[i].second));
    }
    return PyTuple_Pack(2, slot.get(), which.get());
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, "addresses of the library's functions"},
    {"enqueue", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(enqueue)), METH_FASTCALL, "a token's rows into the decode queue"},
    {"attend", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(attend)), METH_FASTCALL, "a decode step with sampled thresholds"},
    {"search", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(search)), METH_FASTCALL, "a dense search"},
    {"append", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(append)), METH_FASTCALL, "new rows into an index"},
    {"draw", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(draw)), METH_FASTCALL, "reservoir sampling"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// BUILT_FOR: torch's version and commit, the interpreter's version (major and minor, a byte each), the library's ABI.  The layouts of
// all three are compiled in, and nothing else would notice that they are others now.
extern "C" __attribute__((visibility("default"))) PyObject* PyInit__host() {
    PyObject* m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddIntConstant(m, "APPENDED", kAppended) < 0) Py_CLEAR(m);
    PyObject* built = m ? Py_BuildValue("(sii)", HIRA_HOST_TORCH, PY_VERSION_HEX >> 16, HIRA_ABI_VERSION) : nullptr;
    if (built == nullptr || PyModule_AddObject(m, "BUILT_FOR", built) < 0) {
        Py_XDECREF(built);
        Py_XDECREF(m);
        return nullptr;
    }
    return m;
}
