// The C ABI's per-step calls as functions of a Python module: what tinytitan_amd/engine.py goes through for every layer and
// token.  A decode step on a short context is bound by its host's work (four launches of 2.0-2.5 us each at 15 us on the
// device); through ctypes, with the tensors' checks and pointers and the per-call int arrays made in Python, a layer
// cost 19 us of host time (QKV epilogue 6.7, attention 7.8, projection 4.35), of which the library's own calls are 13.
//
// Every function takes positional arguments, releases the interpreter lock around the library call and returns the
// library's status code; the caller turns it into an exception.  The functions' addresses come from the library that
// the package has loaded (bind), so this module is built against the header alone.
#include <torch/csrc/autograd/python_variable.h>

#include <dlfcn.h>

#include <exception>
#include <vector>

#include "../../include/ctinytitan_hip.h"

namespace {

#define TT_FUNCTIONS(F)                                                                                                  \
    F(tt_hip_attn_decode)                                                                                                \
    F(tt_hip_attn_decode_swa)                                                                                            \
    F(tt_hip_attn_decode_keep)                                                                                           \
    F(tt_hip_attn_decode_keep_indices)                                                                                   \
    F(tt_hip_attn_verify_swa)                                                                                            \
    F(tt_hip_attn_prefill)                                                                                               \
    F(tt_hip_attn_prefill_swa)                                                                                           \
    F(tt_hip_attn_prefill_keep)                                                                                          \
    F(tt_hip_attn_prefill_keep_indices)                                                                                  \
    F(tt_hip_kv_append)                                                                                                  \
    F(tt_hip_qkv_epilogue_append)                                                                                        \
    F(tt_hip_affine_projection)                                                                                          \
    F(tt_hip_qsa_pool_blocks)                                                                                            \
    F(tt_hip_qsa_norm_rope_rows)                                                                                         \
    F(tt_hip_qsa_block_scores)                                                                                           \
    F(tt_hip_qsa_decode_scores)                                                                                          \
    F(tt_hip_qsa_select)

struct {
#define TT_MEMBER(NAME) decltype(&::NAME) NAME;
    TT_FUNCTIONS(TT_MEMBER)
#undef TT_MEMBER
} lib;

// Arguments in order; the first one that does not convert leaves a Python exception set and `ok` false.
struct Args {
    PyObject *const *at;
    bool ok = true;

    Args(PyObject *const *args, Py_ssize_t given, Py_ssize_t wanted) : at(args) {
        if (given != wanted || !lib.tt_hip_attn_decode) {
            ok = false;
            if (given != wanted) PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", wanted, given);
            else PyErr_SetString(PyExc_RuntimeError, "the library has not been bound");
        }
    }
    template <typename T>
    T *handle() {
        PyObject *o = next();
        if (!ok || o == Py_None) return nullptr;
        void *p = PyLong_AsVoidPtr(o);
        if (!p && PyErr_Occurred()) ok = false;
        return static_cast<T *>(p);
    }
    // What ctypes takes for a C integer: an int, or what says of itself that it is one (__index__: a numpy integer, an integer
    // tensor of one element).  No float is rounded to a count here, and bits beyond the C type's are dropped.
    unsigned long long integer() {
        PyObject *o = next();
        if (!ok) return 0;
        if (PyLong_Check(o)) return bits_of(o);
        return bits_of_new(PyNumber_Index(o));
    }
    int i() { return (int)integer(); }
    size_t size() { return (size_t)integer(); }
    float real() {
        PyObject *o = next();
        if (!ok) return 0.0f;
        const double v = PyFloat_AsDouble(o);
        if (v == -1.0 && PyErr_Occurred()) ok = false;
        return (float)v;
    }
    // an fp16 device tensor, or None
    tt_half *half() {
        const at::Tensor *t = tensor();
        if (!t) return nullptr;
        if (!t->is_cuda() || t->scalar_type() != at::kHalf) return fail<tt_half>("expected an fp16 device tensor");
        return static_cast<tt_half *>(address_of(*t));
    }
    // a device tensor of 16-bit elements, taken as bit patterns
    uint16_t *bits16() {
        const at::Tensor *t = tensor();
        if (!t) return nullptr;
        if (!t->is_cuda() || t->element_size() != 2) return fail<uint16_t>("expected a device tensor of 16-bit elements");
        return static_cast<uint16_t *>(address_of(*t));
    }
    // a contiguous device tensor of any type, or None
    void *raw() {
        const at::Tensor *t = tensor();
        if (!t) return nullptr;
        return address_of(*t, true);
    }
    // Whole numbers per sequence, each what int() takes.  As a step's own: a list or a tuple of them, or one number.  As a
    // `table`: whatever has a length and can be gone through (an array, a tensor, a view of a dict), but no number.
    template <int N>
    int ints(int (&inline_ints)[N], std::vector<int> &heap, const int **out, bool table) {
        PyObject *o = next();
        *out = inline_ints;
        if (!ok) return 0;
        bool list = PyList_Check(o) || PyTuple_Check(o);
        if (!list && !table) {
            inline_ints[0] = (int)integer_of(o);
            return 1;
        }
        if (!list && PyObject_Size(o) < 0) {
            ok = false;
            return 0;
        }
        // Items that are ints are read where they lie: no Python code runs meanwhile, so the caller's list stays as it is.  Any
        // other item's conversion may run some that shortens the list, or hand the interpreter lock to a thread that
        // does: those are converted from a copy.
        PyObject *copy = nullptr;
        Py_ssize_t n = list ? PySequence_Fast_GET_SIZE(o) : 0;
        for (Py_ssize_t k = 0; k < n && list; ++k) list = PyLong_Check(PySequence_Fast_GET_ITEM(o, k));
        if (!list) {
            copy = PySequence_Tuple(o);
            if (!copy) {
                ok = false;
                return 0;
            }
            n = PyTuple_GET_SIZE(copy);
        }
        int *to = inline_ints;
        if (n > N) {
            heap.resize((size_t)n);
            to = heap.data();
        }
        for (Py_ssize_t k = 0; k < n && ok; ++k) to[k] = (int)integer_of(copy ? PyTuple_GET_ITEM(copy, k) : PySequence_Fast_GET_ITEM(o, k));
        *out = to;
        Py_XDECREF(copy);
        return (int)n;
    }

private:
    PyObject *next() { return *at++; }
    template <typename T>
    T *fail(const char *what) {
        ok = false;
        PyErr_SetString(PyExc_TypeError, what);
        return nullptr;
    }
    unsigned long long bits_of(PyObject *whole) {
        const unsigned long long v = PyLong_AsUnsignedLongLongMask(whole);
        if (v == ~0ull && PyErr_Occurred()) ok = false;
        return v;
    }
    unsigned long long integer_of(PyObject *o) {
        if (PyLong_Check(o)) return bits_of(o);
        return bits_of_new(PyNumber_Long(o));  // (what int() takes)
    }
    unsigned long long bits_of_new(PyObject *whole) {
        if (!whole) {
            ok = false;
            return 0;
        }
        const unsigned long long v = bits_of(whole);
        Py_DECREF(whole);
        return v;
    }
    // Throws nothing: a tensor without memory of its own (a traced or fake one) is a Python exception.
    void *address_of(const at::Tensor &t, bool raw = false) {
        try {
            if (raw && (!t.is_cuda() || !t.is_contiguous())) return fail<void>("expected a contiguous device tensor");
            return t.data_ptr();
        } catch (const std::exception &e) {
            ok = false;
            PyErr_SetString(PyExc_RuntimeError, e.what());
            return nullptr;
        }
    }
    const at::Tensor *tensor() {
        PyObject *o = next();
        if (!ok || o == Py_None) return nullptr;
        if (!THPVariable_Check(o)) {
            fail<void>("expected a tensor");
            return nullptr;
        }
        return &THPVariable_Unpack(o);
    }
};

struct Ints {  // one per-sequence table of a call: on the stack for the batch sizes a step has
    int on_stack[64];
    std::vector<int> heap;
    const int *values = on_stack;
    int count = 0;
    void take(Args &a, bool table = false) { count = a.ints(on_stack, heap, &values, table); }
};

template <typename Call>
PyObject *finish(const Args &a, Call call) {
    if (!a.ok) return nullptr;
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = call();
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
}

#define TT_CALL(NAME) PyObject *NAME(PyObject *, PyObject *const *args, Py_ssize_t n)

// (ctx, kv, layer, slots, lengths, heads, q, gate, scale, out)
TT_CALL(attn_decode) {
    Args a(args, n, 10);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    auto *kv = a.handle<tt_hip_kv>();
    const int layer = a.i();
    Ints slots, lens;
    slots.take(a);
    lens.take(a);
    const int heads = a.i();
    const tt_half *q = a.half(), *gate = a.half();
    const float scale = a.real();
    tt_half *out = a.half();
    return finish(a, [&] {
        if (slots.count != lens.count) return (int)TT_HIP_ERR_INVALID_ARGUMENT;
        return lib.tt_hip_attn_decode(ctx, kv, layer, slots.count, slots.values, lens.values, heads, q, gate, scale, out);
    });
}

// (ctx, kv, layer, slots, lengths, window, heads, q, gate, scale, out)
TT_CALL(attn_decode_swa) {
    Args a(args, n, 11);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    auto *kv = a.handle<tt_hip_kv>();
    const int layer = a.i();
    Ints slots, lens;
    slots.take(a);
    lens.take(a);
    const int window = a.i(), heads = a.i();
    const tt_half *q = a.half(), *gate = a.half();
    const float scale = a.real();
    tt_half *out = a.half();
    return finish(a, [&] {
        if (slots.count != lens.count) return (int)TT_HIP_ERR_INVALID_ARGUMENT;
        return lib.tt_hip_attn_decode_swa(ctx, kv, layer, slots.count, slots.values, lens.values, window, heads, q, gate, scale, out);
    });
}

// (ctx, kv, layer, slots, lengths, keep_mask, keep_stride, heads, q, gate, scale, out)
TT_CALL(attn_decode_keep) {
    Args a(args, n, 12);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    auto *kv = a.handle<tt_hip_kv>();
    const int layer = a.i();
    Ints slots, lens;
    slots.take(a);
    lens.take(a);
    const auto *mask = static_cast<const uint8_t *>(a.raw());
    const size_t stride = a.size();
    const int heads = a.i();
    const tt_half *q = a.half(), *gate = a.half();
    const float scale = a.real();
    tt_half *out = a.half();
    return finish(a, [&] {
        if (slots.count != lens.count) return (int)TT_HIP_ERR_INVALID_ARGUMENT;
        return lib.tt_hip_attn_decode_keep(ctx, kv, layer, slots.count, slots.values, lens.values, mask, stride, heads, q, gate, scale,
                                           out);
    });
}

// (ctx, kv, layer, slots, lengths, keep_indices, keep_index_stride, keep_counts, heads, q, gate, scale, out)
TT_CALL(attn_decode_keep_indices) {
    Args a(args, n, 13);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    auto *kv = a.handle<tt_hip_kv>();
    const int layer = a.i();
    Ints slots, lens;
    slots.take(a);
    lens.take(a);
    const auto *indices = static_cast<const uint32_t *>(a.raw());
    const size_t stride = a.size();
    const auto *counts = static_cast<const uint32_t *>(a.raw());
    const int heads = a.i();
    const tt_half *q = a.half(), *gate = a.half();
    const float scale = a.real();
    tt_half *out = a.half();
    return finish(a, [&] {
        if (slots.count != lens.count) return (int)TT_HIP_ERR_INVALID_ARGUMENT;
        return lib.tt_hip_attn_decode_keep_indices(ctx, kv, layer, slots.count, slots.values, lens.values, indices, stride, counts, heads,
                                                   q, gate, scale, out);
    });
}

// (ctx, kv, layer, slots, start_positions, rows, window, heads, q, gate, scale, out)
TT_CALL(attn_verify_swa) {
    Args a(args, n, 12);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    auto *kv = a.handle<tt_hip_kv>();
    const int layer = a.i();
    Ints slots, starts;
    slots.take(a, true);
    starts.take(a, true);
    const int rows = a.i(), window = a.i(), heads = a.i();
    const tt_half *q = a.half(), *gate = a.half();
    const float scale = a.real();
    tt_half *out = a.half();
    return finish(a, [&] {
        if (slots.count > starts.count) return (int)TT_HIP_ERR_INVALID_ARGUMENT;  // (positions may be a longer table than the step's)
        return lib.tt_hip_attn_verify_swa(ctx, kv, layer, slots.count, slots.values, starts.values, rows, window, heads, q, gate, scale,
                                          out);
    });
}

// What the chunk calls have in common behind their own arguments: (heads, q, q_stride, gate, gate_stride, scale, out, o_stride)
struct Rows {
    int heads;
    const tt_half *q;
    size_t q_stride;
    const tt_half *gate;
    size_t gate_stride;
    float scale;
    tt_half *out;
    size_t o_stride;
    explicit Rows(Args &a) : heads(a.i()), q(a.half()), q_stride(a.size()), gate(a.half()), gate_stride(a.size()), scale(a.real()),
                             out(a.half()), o_stride(a.size()) {}
};

// (ctx, kv, layer, slot, start, query_count, kv_valid, window, <rows>); window 0: every key up to the row's own
TT_CALL(attn_prefill) {
    Args a(args, n, 16);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    auto *kv = a.handle<tt_hip_kv>();
    const int layer = a.i(), slot = a.i(), start = a.i(), count = a.i(), valid = a.i(), window = a.i();
    const Rows r(a);
    return finish(a, [&] {
        if (window != 0)
            return lib.tt_hip_attn_prefill_swa(ctx, kv, layer, slot, start, count, valid, window, r.heads, r.q, r.q_stride, r.gate,
                                               r.gate_stride, r.scale, r.out, r.o_stride);
        return lib.tt_hip_attn_prefill(ctx, kv, layer, slot, start, count, valid, r.heads, r.q, r.q_stride, r.gate, r.gate_stride, r.scale,
                                       r.out, r.o_stride);
    });
}

// (ctx, kv, layer, slot, start, query_count, kv_valid, keep_mask, keep_stride, <rows>)
TT_CALL(attn_prefill_keep) {
    Args a(args, n, 17);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    auto *kv = a.handle<tt_hip_kv>();
    const int layer = a.i(), slot = a.i(), start = a.i(), count = a.i(), valid = a.i();
    const auto *mask = static_cast<const uint8_t *>(a.raw());
    const size_t stride = a.size();
    const Rows r(a);
    return finish(a, [&] {
        return lib.tt_hip_attn_prefill_keep(ctx, kv, layer, slot, start, count, valid, mask, stride, r.heads, r.q, r.q_stride, r.gate,
                                            r.gate_stride, r.scale, r.out, r.o_stride);
    });
}

// (ctx, kv, layer, slot, start, query_count, kv_valid, keep_indices, keep_index_stride, keep_counts, <rows>)
TT_CALL(attn_prefill_keep_indices) {
    Args a(args, n, 18);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    auto *kv = a.handle<tt_hip_kv>();
    const int layer = a.i(), slot = a.i(), start = a.i(), count = a.i(), valid = a.i();
    const auto *indices = static_cast<const uint32_t *>(a.raw());
    const size_t stride = a.size();
    const auto *counts = static_cast<const uint32_t *>(a.raw());
    const Rows r(a);
    return finish(a, [&] {
        return lib.tt_hip_attn_prefill_keep_indices(ctx, kv, layer, slot, start, count, valid, indices, stride, counts, r.heads, r.q,
                                                    r.q_stride, r.gate, r.gate_stride, r.scale, r.out, r.o_stride);
    });
}

// (kv, layer, slot, position, n_tokens, k, v, token_stride)
TT_CALL(kv_append) {
    Args a(args, n, 8);
    if (!a.ok) return nullptr;
    auto *kv = a.handle<tt_hip_kv>();
    const int layer = a.i(), slot = a.i(), position = a.i(), tokens = a.i();
    const tt_half *k = a.half(), *v = a.half();
    const size_t stride = a.size();
    return finish(a, [&] { return lib.tt_hip_kv_append(kv, layer, slot, position, tokens, k, v, stride); });
}

// (ctx, kv, layer, slots, positions, rows, heads, q_packed, q_packed_stride, k, v, kv_stride, q_norm, k_norm, eps, rotary_dim,
//  theta, q_out, q_stride, gate_out, gate_stride)
TT_CALL(qkv_epilogue_append) {
    Args a(args, n, 21);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    auto *kv = a.handle<tt_hip_kv>();
    const int layer = a.i();
    Ints slots, positions;
    slots.take(a);
    positions.take(a);
    const int rows = a.i(), heads = a.i();
    const tt_half *packed = a.half();
    const size_t packed_stride = a.size();
    const tt_half *k = a.half(), *v = a.half();
    const size_t kv_stride = a.size();
    const uint16_t *q_norm = a.bits16(), *k_norm = a.bits16();
    const float eps = a.real();
    const int rotary = a.i();
    const float theta = a.real();
    tt_half *q = a.half();
    const size_t q_stride = a.size();
    tt_half *gate = a.half();
    const size_t gate_stride = a.size();
    return finish(a, [&] {
        if (slots.count != positions.count) return (int)TT_HIP_ERR_INVALID_ARGUMENT;
        return lib.tt_hip_qkv_epilogue_append(ctx, kv, layer, slots.count, slots.values, positions.values, rows, heads, packed,
                                              packed_stride, k, v, kv_stride, q_norm, k_norm, eps, rotary, theta, q, q_stride, gate,
                                              gate_stride);
    });
}

// (ctx, bits, weights, weights_offset, scales, biases, x, y, rows, columns, tokens, x_stride, y_stride)
TT_CALL(affine_projection) {
    Args a(args, n, 13);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    const int bits = a.i();
    const auto *weights = static_cast<const uint8_t *>(a.raw());
    const size_t offset = a.size();
    const uint16_t *scales = a.bits16(), *biases = a.bits16();
    const tt_half *x = a.half();
    tt_half *y = a.half();
    const int rows = a.i(), columns = a.i(), tokens = a.i();
    const size_t x_stride = a.size(), y_stride = a.size();
    return finish(a, [&] {
        return lib.tt_hip_affine_projection(ctx, bits, weights ? weights + offset : nullptr, scales, biases, x, y, rows, columns, tokens,
                                            x_stride, y_stride);
    });
}

// (ctx, raw, pooled, dim, first_block, block_count, ratio, n_keys, key_norm, eps, theta)
TT_CALL(qsa_pool_blocks) {
    Args a(args, n, 11);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    const tt_half *raw = a.half();
    tt_half *pooled = a.half();
    const int dim = a.i(), first = a.i(), count = a.i(), ratio = a.i(), keys = a.i();
    const uint16_t *norm = a.bits16();
    const float eps = a.real(), theta = a.real();
    return finish(a, [&] { return lib.tt_hip_qsa_pool_blocks(ctx, raw, pooled, dim, first, count, ratio, keys, norm, eps, theta); });
}

// (ctx, rows, tokens, heads, dim, norm, eps, theta, position, position_stride)
TT_CALL(qsa_norm_rope_rows) {
    Args a(args, n, 10);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    tt_half *rows = a.half();
    const int tokens = a.i(), heads = a.i(), dim = a.i();
    const uint16_t *norm = a.bits16();
    const float eps = a.real(), theta = a.real();
    const int position = a.i(), step = a.i();
    return finish(a, [&] { return lib.tt_hip_qsa_norm_rope_rows(ctx, rows, tokens, heads, dim, norm, eps, theta, position, step); });
}

// (ctx, query_rows, pooled, scores, score_stride, dim, heads, blocks, tokens)
TT_CALL(qsa_block_scores) {
    Args a(args, n, 9);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    const tt_half *rows = a.half(), *pooled = a.half();
    auto *scores = static_cast<float *>(a.raw());
    const size_t stride = a.size();
    const int dim = a.i(), heads = a.i(), blocks = a.i(), tokens = a.i();
    return finish(a, [&] { return lib.tt_hip_qsa_block_scores(ctx, rows, pooled, scores, stride, dim, heads, blocks, tokens); });
}

// (ctx, raw, pooled, dim, ratio, n_keys, key_norm, query_rows, heads, query_norm, position, eps, theta, scores)
TT_CALL(qsa_decode_scores) {
    Args a(args, n, 14);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    const tt_half *raw = a.half();
    tt_half *pooled = a.half();
    const int dim = a.i(), ratio = a.i(), keys = a.i();
    const uint16_t *key_norm = a.bits16();
    const tt_half *rows = a.half();
    const int heads = a.i();
    const uint16_t *query_norm = a.bits16();
    const int position = a.i();
    const float eps = a.real(), theta = a.real();
    auto *scores = static_cast<float *>(a.raw());
    return finish(a, [&] {
        return lib.tt_hip_qsa_decode_scores(ctx, raw, pooled, dim, ratio, keys, key_norm, rows, heads, query_norm, position, eps, theta,
                                            scores);
    });
}

// (ctx, scores, score_stride, rows, first_visible, ratio, width, mask, mask_stride, indices, index_stride, counts)
TT_CALL(qsa_select) {
    Args a(args, n, 12);
    if (!a.ok) return nullptr;
    auto *ctx = a.handle<tt_hip_ctx>();
    const auto *scores = static_cast<const float *>(a.raw());
    const size_t stride = a.size();
    const int rows = a.i(), visible = a.i(), ratio = a.i(), width = a.i();
    auto *mask = static_cast<uint8_t *>(a.raw());
    const size_t mask_stride = a.size();
    auto *indices = static_cast<uint32_t *>(a.raw());
    const size_t index_stride = a.size();
    auto *counts = static_cast<uint32_t *>(a.raw());
    return finish(a, [&] {
        return lib.tt_hip_qsa_select(ctx, scores, stride, rows, visible, ratio, width, mask, mask_stride, indices, index_stride, counts);
    });
}

// bind(path): takes the functions' addresses from the library at `path`, which the process has loaded already.
PyObject *bind(PyObject *, PyObject *arg) {
    const char *path = PyUnicode_AsUTF8(arg);
    if (!path) return nullptr;
    void *const handle = dlopen(path, RTLD_NOW | RTLD_NOLOAD);
    if (!handle) return PyErr_Format(PyExc_RuntimeError, "%s is not loaded", path);
#define TT_FIND(NAME)                                                                                        \
    lib.NAME = reinterpret_cast<decltype(lib.NAME)>(dlsym(handle, #NAME));                                   \
    if (!lib.NAME) return PyErr_Format(PyExc_RuntimeError, "%s does not export %s", path, #NAME);
    TT_FUNCTIONS(TT_FIND)
#undef TT_FIND
    dlclose(handle);  // (the package's own handle keeps it loaded)
    Py_RETURN_NONE;
}

#define TT_METHOD(NAME) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(NAME)), METH_FASTCALL, nullptr},
PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    TT_METHOD(attn_decode) TT_METHOD(attn_decode_swa) TT_METHOD(attn_decode_keep) TT_METHOD(attn_decode_keep_indices)
    TT_METHOD(attn_verify_swa) TT_METHOD(attn_prefill) TT_METHOD(attn_prefill_keep) TT_METHOD(attn_prefill_keep_indices)
    TT_METHOD(kv_append) TT_METHOD(qkv_epilogue_append) TT_METHOD(affine_projection) TT_METHOD(qsa_pool_blocks)
    TT_METHOD(qsa_norm_rope_rows) TT_METHOD(qsa_block_scores) TT_METHOD(qsa_decode_scores) TT_METHOD(qsa_select)
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_tt_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tt_calls() { return PyModule_Create(&module); }
