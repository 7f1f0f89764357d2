// The launches that a step with a prompt is made of, as functions of a Python module: they check their tensors, allocate what they return and call the kernel
// library's entry points. A step runs some hundred of them one by one, and a short prompt's step is bound by that: written in Python (checks, allocations, an
// address per argument, ctypes) a product took 11 us of the host's time, of which the launch itself is 3; see ops.py for what each function computes.
//
// As with ctypes, other Python threads run while memory is found and the kernel library called: either may wait (for the driver, for room in a queue).
//
// A function returns NotImplemented wherever something about its arguments is not as the plain case has it; its caller then takes the general path, which
// also knows what to refuse and how to say so.
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ops/empty.h>

#include <utility>

#include "../fw_kernels.h"

namespace {

enum { F32 = 0, BF16 = 1 };
enum { STORE = 0, ADD = 1, GATED = 2 };

struct Entries {
    decltype(&fw_gemm_rows) gemm_rows;
    decltype(&fw_gemm_medium) gemm_medium;
    decltype(&fw_gemm_mfma_big_tile) big_tile;
    decltype(&fw_rmsnorm_rows) rmsnorm_rows;
    decltype(&fw_shortconv) shortconv;
    decltype(&fw_qk_norm_rope_kv_write) qk_norm;
    decltype(&fw_attention_prefill) prefill;
    const char* (*last_error)();
} entry;
PyObject *kernel_error = nullptr, *out_of_memory = nullptr;

// A tensor argument; null for None. `plain` turns false where it is neither.
const at::Tensor* tensor(PyObject* o, bool& plain) {
    if (o == Py_None) return nullptr;
    if (!THPVariable_Check(o)) {
        plain = false;
        return nullptr;
    }
    return &THPVariable_Unpack(o);
}
// ... on the GPU, contiguous, of this type and number of dimensions (0: any)
bool is(const at::Tensor* t, at::ScalarType type, int dims = 0) {
    return t && t->is_cuda() && t->scalar_type() == type && (dims == 0 || t->dim() == dims) && t->is_contiguous();
}
bool none_or(const at::Tensor* t, at::ScalarType type, int dims = 0) { return !t || is(t, type, dims); }
bool size_is(const at::Tensor* t, int64_t n) { return !t || (t->dim() == 1 && t->size(0) == n); }
template <typename T>
T* at_of(const at::Tensor* t) { return t ? static_cast<T*>(t->data_ptr()) : nullptr; }
bool same_device(const at::Tensor& a, std::initializer_list<const at::Tensor*> others) {
    for (const at::Tensor* t : others)
        if (t && t->get_device() != a.get_device()) return false;
    return true;
}
at::Tensor make(const at::Tensor& like, int64_t rows, int64_t columns, at::ScalarType type) { return at::empty({rows, columns}, like.options().dtype(type)); }
bool fits(int64_t v) { return v >= 0 && v < (1ll << 31); }

// The interpreter's lock is let go while this lives: nothing of Python's is touched meanwhile.
struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename Call>
int unlocked(Call call) {
    const Unlocked others;
    return call();
}

int whole(PyObject* o) { return (int)PyLong_AsLong(o); }
float number(PyObject* o) { return (float)PyFloat_AsDouble(o); }
void* stream_of(PyObject* o) { return PyLong_AsVoidPtr(o); }

PyObject* other_path() { Py_RETURN_NOTIMPLEMENTED; }
PyObject* answer(int status, PyObject* result) {
    if (status == 0) return result;
    Py_XDECREF(result);
    PyErr_SetString(kernel_error, entry.last_error());
    return nullptr;
}
bool wrong(Py_ssize_t given, Py_ssize_t wanted) {
    if (given == wanted) return false;
    PyErr_Format(PyExc_TypeError, "%zd arguments, wanted %zd", given, wanted);
    return true;
}

// product(a, w, tiled, bias, target, mode, out_code, stored as bfloat16, next norm's weight, one-centred, squares, eps, limit, alpha, shift, plan, counters, stream):
// plan (0, K split, bytes, counters, rows of squares so, rows of squares) for up to 64 rows, or (1, rows, columns, each, slices, bytes, counters).
PyObject* product(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (wrong(n, 18)) return nullptr;
    bool plain = true;
    const at::Tensor *a = tensor(args[0], plain), *w = tensor(args[1], plain), *tiled = tensor(args[2], plain), *bias = tensor(args[3], plain),
                     *target = tensor(args[4], plain), *next_weight = tensor(args[8], plain), *squares = tensor(args[10], plain), *counters = tensor(args[16], plain);
    if (!plain || !is(a, at::kBFloat16, 2) || !is(w, at::kBFloat16, 2) || !none_or(tiled, at::kBFloat16, 5) || !none_or(bias, at::kFloat, 1) ||
        !none_or(next_weight, at::kFloat, 1) || !none_or(squares, at::kFloat, 2) || !same_device(*a, {w, tiled, bias, target, next_weight, squares, counters}))
        return other_path();
    const int mode = whole(args[5]), out_code = whole(args[6]), one_centered = PyObject_IsTrue(args[9]);
    const bool rounded = PyObject_IsTrue(args[7]);
    const int64_t M = a->size(0), K = a->size(1), w_rows = w->size(0), N = mode == GATED ? w_rows / 2 : w_rows;
    if ((uintptr_t)a->data_ptr() % 16 || (uintptr_t)w->data_ptr() % 16) return other_path();
    if (M < 1 || w->size(1) != K || (mode == GATED && w_rows % 2) || !size_is(bias, w_rows) || !fits(M) || !fits(K) || !fits(w_rows)) return other_path();
    if (tiled && (K % 32 || tiled->size(0) != (w_rows + 15) / 16 || tiled->size(1) != K / 32 || tiled->size(2) != 4 || tiled->size(3) != 16 || tiled->size(4) != 8))
        return other_path();
    if ((mode == ADD) != (target != nullptr) || (target && (!is(target, at::kFloat, 2) || target->size(0) != M || target->size(1) != N))) return other_path();
    if (next_weight && (mode != ADD || next_weight->size(0) != N)) return other_path();
    const int64_t stride = M <= 16 ? 16 : 64;
    if (squares && squares->size(1) != stride) return other_path();
    PyObject* plan = args[15];
    if (!PyTuple_Check(plan) || PyTuple_GET_SIZE(plan) < 6) return other_path();
    const bool large = PyLong_AsSsize_t(PyTuple_GET_ITEM(plan, 0)) == 1;
    Py_ssize_t planned[7] = {};
    if (large && (PyTuple_GET_SIZE(plan) != 7 || next_weight || squares)) return other_path();
    for (int i = 1; i < (large ? 7 : 6); ++i) planned[i] = PyLong_AsSsize_t(PyTuple_GET_ITEM(plan, i));
    const float eps = number(args[11]), limit = number(args[12]), alpha = number(args[13]), shift = number(args[14]);
    void* stream = stream_of(args[17]);
    if (PyErr_Occurred()) return nullptr;
    // the large tile that is named, K split over workgroups or the product whose waves split K
    const bool split = !large && planned[1] && (!target || (uintptr_t)target->data_ptr() % 16 == 0);
    const size_t bytes = large ? (size_t)planned[5] : split ? (size_t)planned[2] : 0;
    const int tickets = large ? (int)planned[6] : (int)planned[3];
    if (bytes && (!is(counters, at::kInt, 1) || counters->size(0) < tickets)) return other_path();

    at::Tensor out, workspace, activations, next_squares;
    const int status = unlocked([&] {
        out = target ? *target : make(*a, M, N, rounded ? at::kBFloat16 : at::kFloat);
        if (bytes) workspace = at::empty({(int64_t)(bytes / 4)}, a->options().dtype(at::kFloat));
        if (next_weight) {
            activations = make(*a, M, N, at::kBFloat16);
            next_squares = make(*a, split ? planned[4] : planned[5], stride, at::kFloat);
        }
        void *to = out.data_ptr(), *room = bytes ? workspace.data_ptr() : nullptr, *next = next_weight ? activations.data_ptr() : nullptr;
        const void* operand = (tiled ? tiled : w)->data_ptr();
        int* ticket = bytes ? at_of<int>(counters) : nullptr;
        float* next_sums = next_weight ? static_cast<float*>(next_squares.data_ptr()) : nullptr;
        const int squares_rows = squares ? (int)squares->size(0) : 0;
        if (large)
            return entry.big_tile(a->data_ptr(), w->data_ptr(), at_of<const float>(bias), to, out_code, mode, (int)M, (int)N, (int)K, (int)planned[1], (int)planned[2],
                                  (int)planned[3], (int)planned[4], room, bytes, ticket, tickets, stream);
        if (split)
            return entry.gemm_medium(a->data_ptr(), operand, tiled != nullptr, at_of<const float>(bias), to, out_code, mode, (int)M, (int)N, (int)K, room, bytes, ticket,
                                     bytes ? (int)counters->size(0) : 0, at_of<const float>(next_weight), one_centered, next, next_sums, at_of<const float>(squares),
                                     squares_rows, eps, limit, alpha, shift, stream);
        return entry.gemm_rows(a->data_ptr(), operand, tiled != nullptr, at_of<const float>(bias), to, out_code, mode, (int)M, (int)N, (int)K,
                               at_of<const float>(next_weight), one_centered, next, next_sums, at_of<const float>(squares), squares_rows, eps, limit, alpha, shift, stream);
    });
    if (status) return answer(status, nullptr);
    if (next_weight) {
        PyObject* pair = PyTuple_New(2);
        if (!pair) return nullptr;
        PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(activations)));
        PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(next_squares)));
        return pair;
    }
    if (target) {
        Py_INCREF(args[4]);
        return args[4];
    }
    return THPVariable_Wrap(std::move(out));
}

// rmsnorm(x, weight, row_index, bfloat16 out, eps, one-centred, stream)
PyObject* rmsnorm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (wrong(n, 7)) return nullptr;
    bool plain = true;
    const at::Tensor *x = tensor(args[0], plain), *weight = tensor(args[1], plain), *index = tensor(args[2], plain);
    if (!plain || !is(x, at::kFloat) || x->dim() < 1 || !is(weight, at::kFloat, 1) || !none_or(index, at::kInt) || !same_device(*x, {weight, index})) return other_path();
    const int64_t hidden = x->size(-1);
    if (hidden < 1 || weight->size(0) != hidden) return other_path();
    const int64_t rows = index ? index->numel() : x->numel() / hidden;
    if (!fits(rows) || !fits(hidden)) return other_path();
    const int rounded = PyObject_IsTrue(args[3]), one_centered = PyObject_IsTrue(args[5]);
    const float eps = number(args[4]);
    void* stream = stream_of(args[6]);
    if (PyErr_Occurred()) return nullptr;
    at::Tensor out;
    const int status = unlocked([&] {
        out = make(*x, rows, hidden, rounded ? at::kBFloat16 : at::kFloat);
        return entry.rmsnorm_rows(at_of<const float>(x), at_of<const float>(weight), out.data_ptr(), rounded ? BF16 : F32, at_of<const int32_t>(index), (int)rows,
                                  (int)hidden, eps, one_centered, stream);
    });
    return status ? answer(status, nullptr) : THPVariable_Wrap(std::move(out));
}

// shortconv(bcx, taps, bias, state, row_seg, seg_row0, seg_slot, segments, bfloat16 out, stream)
PyObject* shortconv(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (wrong(n, 10)) return nullptr;
    bool plain = true;
    const at::Tensor *bcx = tensor(args[0], plain), *taps = tensor(args[1], plain), *bias = tensor(args[2], plain), *state = tensor(args[3], plain),
                     *row_seg = tensor(args[4], plain), *seg_row0 = tensor(args[5], plain), *seg_slot = tensor(args[6], plain);
    if (!plain || !bcx || (!is(bcx, at::kFloat, 2) && !is(bcx, at::kBFloat16, 2)) || !is(taps, at::kFloat, 2) || !none_or(bias, at::kFloat, 1) || !is(state, at::kFloat, 3) ||
        !is(row_seg, at::kInt) || !is(seg_row0, at::kInt) || !is(seg_slot, at::kInt) || !same_device(*bcx, {taps, bias, state, row_seg, seg_row0, seg_slot}))
        return other_path();
    const int64_t rows = bcx->size(0), hidden = taps->size(0), kernel = taps->size(1), segments = PyLong_AsLong(args[7]);
    const int rounded = PyObject_IsTrue(args[8]);
    void* stream = stream_of(args[9]);
    if (PyErr_Occurred()) return nullptr;
    if (bcx->size(1) != 3 * hidden || state->size(1) != hidden || state->size(2) != kernel - 1 || !size_is(bias, hidden) || row_seg->numel() < rows ||
        seg_row0->numel() < segments + 1 || seg_slot->numel() < segments || !fits(rows) || !fits(state->size(0)))
        return other_path();
    at::Tensor out;
    const int status = unlocked([&] {
        out = make(*bcx, rows, hidden, rounded ? at::kBFloat16 : at::kFloat);
        return entry.shortconv(bcx->data_ptr(), bcx->scalar_type() == at::kFloat ? F32 : BF16, out.data_ptr(), rounded ? BF16 : F32, at_of<const float>(taps),
                               at_of<const float>(bias), at_of<float>(state), at_of<const int32_t>(row_seg), at_of<const int32_t>(seg_row0),
                               at_of<const int32_t>(seg_slot), (int)rows, (int)segments, (int)hidden, (int)kernel, (int)state->size(0), stream);
    });
    return status ? answer(status, nullptr) : THPVariable_Wrap(std::move(out));
}

bool pages_are(const at::Tensor* k, const at::Tensor* v, int64_t kv_heads, int64_t head_dim, int64_t v_dim, int64_t page, at::ScalarType type) {
    return is(k, type, 4) && is(v, type, 4) && k->size(1) == kv_heads && k->size(2) == page && k->size(3) == head_dim && v->size(0) == k->size(0) &&
           v->size(1) == kv_heads && v->size(2) == v_dim && v->size(3) == page && fits(k->size(0));
}

// qk_norm(qkv, heads, kv heads, head size, q weight, k weight, eps, cos, sin, rotary size, k pages, v pages, table, row_seg, row_pos, write, value size, interleaved,
// queries alone, row scale, tokens of a page, stream)
PyObject* qk_norm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (wrong(n, 22)) return nullptr;
    bool plain = true;
    const at::Tensor *qkv = tensor(args[0], plain), *qw = tensor(args[4], plain), *kw = tensor(args[5], plain), *cos = tensor(args[7], plain), *sin = tensor(args[8], plain),
                     *k = tensor(args[10], plain), *v = tensor(args[11], plain), *table = tensor(args[12], plain), *row_seg = tensor(args[13], plain),
                     *row_pos = tensor(args[14], plain), *scale = tensor(args[19], plain);
    const int64_t heads = PyLong_AsLong(args[1]), kv_heads = PyLong_AsLong(args[2]), head_dim = PyLong_AsLong(args[3]), rotary = PyLong_AsLong(args[9]),
                  v_dim = PyLong_AsLong(args[16]), page = PyLong_AsLong(args[20]);
    const float eps = number(args[6]);
    const int write = PyObject_IsTrue(args[15]), interleaved = PyObject_IsTrue(args[17]), q_only = PyObject_IsTrue(args[18]);
    void* stream = stream_of(args[21]);
    if (PyErr_Occurred()) return nullptr;
    // (rows of qkv that lie apart, and a page type of its own, take the general path)
    if (!plain || !qkv || (!is(qkv, at::kFloat, 2) && !is(qkv, at::kBFloat16, 2)) || !k || (k->scalar_type() != at::kBFloat16 && k->scalar_type() != at::kFloat) ||
        !pages_are(k, v, kv_heads, head_dim, v_dim, page, k->scalar_type()) || !none_or(qw, at::kFloat, 1) || !none_or(kw, at::kFloat, 1) || !size_is(qw, head_dim) ||
        !size_is(kw, head_dim) || !is(table, at::kInt, 2) || !is(row_seg, at::kInt) || !is(row_pos, at::kInt) || !none_or(scale, at::kFloat) ||
        !same_device(*qkv, {qw, kw, cos, sin, k, v, table, row_seg, row_pos, scale}))
        return other_path();
    const int64_t rows = qkv->size(0), width = q_only ? heads * head_dim : (heads + kv_heads) * head_dim + kv_heads * v_dim;
    if (qkv->size(1) != width || (q_only && write) || row_seg->numel() < rows || row_pos->numel() < rows || (scale && scale->numel() < rows) || !fits(rows) ||
        !fits(table->size(1)))
        return other_path();
    for (const at::Tensor* t : {cos, sin}) {
        if (rotary && (!is(t, at::kFloat, 2) || t->size(0) != rows || t->size(1) != rotary / 2)) return other_path();
        if (!rotary && t && !t->is_contiguous()) return other_path();
    }
    at::Tensor out;
    const int status = unlocked([&] {
        out = make(*qkv, rows, heads * head_dim, k->scalar_type());
        return entry.qk_norm(qkv->data_ptr(), qkv->scalar_type() == at::kFloat ? F32 : BF16, (int)width, out.data_ptr(), k->scalar_type() == at::kFloat ? F32 : BF16,
                             at_of<const float>(qw), at_of<const float>(kw), eps, at_of<const float>(cos), at_of<const float>(sin), (int)rotary, k->data_ptr(),
                             v->data_ptr(), at_of<const int32_t>(table), (int)table->size(1), at_of<const int32_t>(row_seg), at_of<const int32_t>(row_pos), (int)rows,
                             (int)heads, (int)kv_heads, (int)head_dim, (int)v_dim, (int)page, (int)k->size(0), write, interleaved, q_only, at_of<const float>(scale), stream);
    });
    return status ? answer(status, nullptr) : THPVariable_Wrap(std::move(out));
}

// prefill(q, heads, kv heads, head size, k pages, v pages, table, tile_seg, tile_row0, seg_row0, row_pos, scale, window, heads together, value size, chunk, softcap,
// kept first keys, sinks, slopes, form, tokens of a page, stream)
PyObject* prefill(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (wrong(n, 23)) return nullptr;
    bool plain = true;
    const at::Tensor *q = tensor(args[0], plain), *k = tensor(args[4], plain), *v = tensor(args[5], plain), *table = tensor(args[6], plain), *tile_seg = tensor(args[7], plain),
                     *tile_row0 = tensor(args[8], plain), *seg_row0 = tensor(args[9], plain), *row_pos = tensor(args[10], plain), *sinks = tensor(args[18], plain),
                     *slopes = tensor(args[19], plain);
    const int64_t heads = PyLong_AsLong(args[1]), kv_heads = PyLong_AsLong(args[2]), head_dim = PyLong_AsLong(args[3]), v_dim = PyLong_AsLong(args[14]),
                  page = PyLong_AsLong(args[21]);
    const int window = whole(args[12]), together = whole(args[13]), chunk = whole(args[15]), kept = whole(args[17]), form = whole(args[20]);
    const float scale = number(args[11]), softcap = number(args[16]);
    void* stream = stream_of(args[22]);
    if (PyErr_Occurred()) return nullptr;
    if (!plain || !is(q, at::kBFloat16, 2) || !pages_are(k, v, kv_heads, head_dim, v_dim, page, at::kBFloat16) || !is(table, at::kInt, 2) || !is(tile_seg, at::kInt) ||
        !is(tile_row0, at::kInt) || !is(seg_row0, at::kInt) || !is(row_pos, at::kInt) || !none_or(sinks, at::kFloat, 1) || !none_or(slopes, at::kFloat, 1) ||
        !size_is(sinks, heads) || !size_is(slopes, heads) || !same_device(*q, {k, v, table, tile_seg, tile_row0, seg_row0, row_pos, sinks, slopes}))
        return other_path();
    const int64_t rows = q->size(0);
    if (q->size(1) != heads * head_dim || row_pos->numel() < rows || tile_seg->numel() != tile_row0->numel() || kept < 0 || (kept && chunk) || !fits(rows) ||
        !fits(table->size(1)))
        return other_path();
    at::Tensor out;
    const int status = unlocked([&] {
        out = make(*q, rows, heads * v_dim, at::kBFloat16);
        return entry.prefill(q->data_ptr(), out.data_ptr(), k->data_ptr(), v->data_ptr(), at_of<const int32_t>(table), (int)table->size(1),
                             at_of<const int32_t>(tile_seg), at_of<const int32_t>(tile_row0), (int)tile_seg->numel(), at_of<const int32_t>(seg_row0),
                             at_of<const int32_t>(row_pos), (int)rows, (int)heads, (int)kv_heads, (int)head_dim, (int)v_dim, scale, window, chunk, softcap,
                             window ? kept : 0, at_of<const float>(sinks), at_of<const float>(slopes), (int)page, (int)k->size(0), together, form, stream);
    });
    return status ? answer(status, nullptr) : THPVariable_Wrap(std::move(out));
}

// bind(addresses of the entry points by name, the exceptions of a refused call and of an allocation that fails): called before anything else
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (wrong(n, 3)) return nullptr;
    bool found = PyDict_Check(args[0]);
    auto take = [&](const char* name, auto& to) {
        PyObject* at = found ? PyDict_GetItemString(args[0], name) : nullptr;
        void* address = at ? PyLong_AsVoidPtr(at) : nullptr;
        if (!address) found = false;
        to = reinterpret_cast<std::decay_t<decltype(to)>>(address);
    };
    take("fw_gemm_rows", entry.gemm_rows);
    take("fw_gemm_medium", entry.gemm_medium);
    take("fw_gemm_mfma_big_tile", entry.big_tile);
    take("fw_rmsnorm_rows", entry.rmsnorm_rows);
    take("fw_shortconv", entry.shortconv);
    take("fw_qk_norm_rope_kv_write", entry.qk_norm);
    take("fw_attention_prefill", entry.prefill);
    take("fw_last_error", entry.last_error);
    if (!found) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: an entry point has no address");
        return nullptr;
    }
    for (auto [held, given] : {std::pair{&kernel_error, args[1]}, std::pair{&out_of_memory, args[2]}}) {
        Py_INCREF(given);
        Py_XDECREF(*held);
        *held = given;
    }
    Py_RETURN_NONE;
}

// No C++ exception (an allocation that fails) may pass into the interpreter.
template <PyObject* (*CALL)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    try {
        return CALL(self, args, n);
    } catch (const c10::OutOfMemoryError& error) {
        PyErr_SetString(out_of_memory, error.what_without_backtrace());
    } catch (const std::exception& error) {
        PyErr_SetString(PyExc_RuntimeError, error.what());
    }
    return nullptr;
}
template <PyObject* (*CALL)(PyObject*, PyObject* const*, Py_ssize_t)>
PyCFunction method() {
    return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&guarded<CALL>));
}

PyMethodDef methods[] = {{"bind", method<bind>(), METH_FASTCALL, nullptr},
                         {"product", method<product>(), METH_FASTCALL, nullptr},
                         {"rmsnorm", method<rmsnorm>(), METH_FASTCALL, nullptr},
                         {"shortconv", method<shortconv>(), METH_FASTCALL, nullptr},
                         {"qk_norm", method<qk_norm>(), METH_FASTCALL, nullptr},
                         {"prefill", method<prefill>(), METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "fw_launch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit_fw_launch() { return PyModule_Create(&module); }
