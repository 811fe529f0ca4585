// The calls of llminfer_amd.ops, native: tensors and keyword arguments in, one call of the C ABI out.
//
// An eager decode step is one such call per layer and kernel, a few microseconds of GPU work each, so what a call costs on the
// host is what an eager step costs. Filling the argument structs through ctypes and asking torch for its current stream from
// Python came to 5.5 us on top of the 3.9 us the C call takes (launch included); here the tensors are unpacked where they are
// and the struct is filled in place: back to back on a short context, mha_decode 9.5 -> 3.2 us a call (the prepared C call: 3.0),
// gemv 7.5 -> 2.7; the 36 attention blocks of a step at 700 positions, call by call, 1163 -> 656 us, the GPU's own time.
//
// Nothing is kept from one call to the next. The C ABI's functions, torch's two accessors and the Python side's slow paths
// (which word every error) are handed over once by bind(): the library itself is loaded by llminfer_amd._binding, so a
// variant build is picked up here too.
#include <Python.h>

#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <initializer_list>

#include "llmi_hip.h"

namespace {

// ---- keyword arguments ----
#define LLMI_KEYWORDS(X)                                                                                                          \
    X(query) X(query_raw) X(key_cache) X(value_cache) X(output) X(workspace) X(stream) X(layer_id) X(pos) X(kv_dim) X(kv_mul)    \
    X(head_num) X(head_dim) X(max_seq_len) X(kv_layout) X(force_path) X(num_splits) X(waves_per_group) X(output_f32)             \
    X(pos_device) X(workspace_side) X(key_new) X(value_new) X(norm_weight) X(sin_cache) X(cos_cache) X(eps) X(o_weight)          \
    X(residual) X(one_launch) X(layer_count) X(query_stride) X(key_new_stride) X(value_new_stride) X(norm_weight_stride)         \
    X(output_stride) X(query_src) X(input) X(weight) X(mode) X(key) X(value) X(src_pos_major) X(dst_head_major) X(layer_num)     \
    X(num_pos)

enum Key : int {
#define X(name) k_##name,
    LLMI_KEYWORDS(X)
#undef X
    kKeys
};
static_assert(kKeys <= 64, "a mask bit per keyword");
const char* const kKeyText[] = {
#define X(name) #name,
    LLMI_KEYWORDS(X)
#undef X
};
PyObject* g_key[kKeys];  // interned names

// Keyword names reach a call interned: found by address, in a small table; a name that is not is compared letter by letter.
constexpr int kSlots = 256;
int8_t g_slot[kSlots];
inline unsigned slot_of(PyObject* name) { return (unsigned)((reinterpret_cast<uintptr_t>(name) >> 4) * 0x9E3779B1u >> 24) % kSlots; }

int find_key(PyObject* name) {
    for (unsigned s = slot_of(name);; s = (s + 1) % kSlots) {
        const int k = g_slot[s];
        if (k < 0) break;
        if (g_key[k] == name) return k;
    }
    for (int k = 0; k < kKeys; ++k)
        if (PyUnicode_Compare(g_key[k], name) == 0) return k;
    return -1;
}

constexpr uint64_t bits(std::initializer_list<Key> keys) {
    uint64_t m = 0;
    for (Key k : keys) m |= 1ull << k;
    return m;
}

// One entry point's signature: parameters that may be given by position (in order; the first `required_pos` of them without a
// default), further keywords, and which of those have no default.
struct Signature {
    const char* name;
    const Key* positional;
    int n_positional;
    uint64_t keywords, required;
};

bool parse(const Signature& sig, PyObject* const* args, Py_ssize_t n_args, PyObject* names, PyObject** vals) {
    if (n_args > sig.n_positional) {
        PyErr_Format(PyExc_TypeError, "%s() takes %d positional arguments but %zd were given", sig.name, sig.n_positional, n_args);
        return false;
    }
    for (int i = 0; i < kKeys; ++i) vals[i] = nullptr;
    uint64_t positional = 0;
    for (int i = 0; i < sig.n_positional; ++i) {
        positional |= 1ull << sig.positional[i];
        if (i < n_args) vals[sig.positional[i]] = args[i];
    }
    uint64_t missing = sig.required;
    for (int i = 0; i < n_args; ++i) missing &= ~(1ull << sig.positional[i]);
    const Py_ssize_t n_names = names ? PyTuple_GET_SIZE(names) : 0;
    for (Py_ssize_t i = 0; i < n_names; ++i) {
        PyObject* name = PyTuple_GET_ITEM(names, i);
        const int k = find_key(name);
        if (k < 0 || !((sig.keywords | positional) >> k & 1)) {
            PyErr_Format(PyExc_TypeError, "%s() got an unexpected keyword argument '%U'", sig.name, name);
            return false;
        }
        if (vals[k]) {
            PyErr_Format(PyExc_TypeError, "%s() got multiple values for argument '%U'", sig.name, name);
            return false;
        }
        vals[k] = args[n_args + i];
        missing &= ~(1ull << k);
    }
    if (missing) {
        int k = 0;
        while (!(missing >> k & 1)) ++k;
        PyErr_Format(PyExc_TypeError, "%s() missing required argument: '%s'", sig.name, kKeyText[k]);
        return false;
    }
    return true;
}

// ---- what bind() hands over ----
struct Abi {
    int (*mha_decode)(const llmi_mha_args*);
    int (*mha_decode_append)(const llmi_mha_append_args*);
    int (*mha_decode_append_oproj)(const llmi_attn_oproj_args*);
    int (*mha_oproj_launches)(const llmi_attn_oproj_args*);
    int (*mha_decode_append_stack)(const llmi_mha_stack_args*);
    int (*mha_stack_launches)(const llmi_mha_stack_args*);
    int (*qk_norm_rope_append)(const llmi_qk_norm_rope_args*);
    int (*kv_restride)(const void*, void*, int32_t, int32_t, int32_t, int32_t, int32_t, void*);
    int (*gemv)(const llmi_gemv_args*);
    int (*qkv_gemv)(const llmi_qkv_gemv_args*);
} g_abi;
PyObject *g_get_device, *g_get_stream;   // torch's current device, and its current stream as a number
PyObject *g_check_dev, *g_check_status;  // ops._check_dev, _binding.check: they raise
PyObject *g_bf16_types, *g_f32_types;    // what _check_dev is told to expect

// ---- conversions ----
enum class Kind { bf16, f32 };

inline bool type_fits(const at::Tensor& t, Kind kind) {
    const at::ScalarType s = t.scalar_type();
    return kind == Kind::f32 ? s == at::kFloat : s == at::kBFloat16 || s == at::kShort || s == at::ScalarType::UInt16;
}

// The tensor's address, or nullptr for an absent argument or None; *ok is cleared, with the exception ops._check_dev raises, for
// anything that is not a contiguous device tensor of the kind.
void* address(PyObject* const* vals, Key key, Kind kind, bool* ok) {
    PyObject* o = vals[key];
    if (!o || o == Py_None || !*ok) return nullptr;
    if (THPVariable_Check(o)) {
        const at::Tensor& t = THPVariable_Unpack(o);
        if (t.is_cuda() && type_fits(t, kind) && t.is_contiguous()) return t.data_ptr();
    }
    *ok = false;
    PyObject* r = PyObject_CallFunctionObjArgs(g_check_dev, g_key[key], o, kind == Kind::f32 ? g_f32_types : g_bf16_types, nullptr);
    if (r) {
        Py_DECREF(r);
        PyErr_Format(PyExc_ValueError, "%s is not a tensor this call can take", kKeyText[key]);
    }
    return nullptr;
}

int64_t int64(PyObject* const* vals, Key key, int64_t unset, bool* ok) {
    PyObject* o = vals[key];
    if (!o || !*ok) return unset;
    int64_t v;
    if (PyLong_Check(o)) {
        v = (int64_t)PyLong_AsUnsignedLongLongMask(o);  // (out of range wraps, as it does in the ctypes structs)
    } else {
        PyObject* n = PyNumber_Index(o);
        if (!n) {
            *ok = false;
            return unset;
        }
        v = (int64_t)PyLong_AsUnsignedLongLongMask(n);
        Py_DECREF(n);
    }
    if (v == -1 && PyErr_Occurred()) *ok = false;
    return v;
}
int32_t int32(PyObject* const* vals, Key key, int32_t unset, bool* ok) { return (int32_t)int64(vals, key, unset, ok); }

// An argument that is a tensor or a raw address (the position word).
void* tensor_or_address(PyObject* const* vals, Key key, bool* ok) {
    PyObject* o = vals[key];
    if (!o || o == Py_None || !*ok) return nullptr;
    if (THPVariable_Check(o)) return THPVariable_Unpack(o).data_ptr();
    return reinterpret_cast<void*>((uintptr_t)int64(vals, key, 0, ok));
}

// stream = None: torch's current one; an object with a cuda_stream; or a number.
void* stream_of(PyObject* const* vals, bool* ok) {
    if (!*ok) return nullptr;
    PyObject* s = vals[k_stream];
    PyObject* n = nullptr;
    if (!s || s == Py_None) {
        PyObject* dev = PyObject_CallNoArgs(g_get_device);
        if (dev) n = PyObject_CallOneArg(g_get_stream, dev);
        Py_XDECREF(dev);
    } else if (PyLong_Check(s)) {
        n = Py_NewRef(s);
    } else {
        n = PyObject_GetAttrString(s, "cuda_stream");
        if (!n && PyErr_ExceptionMatches(PyExc_AttributeError)) {
            PyErr_Clear();
            n = PyNumber_Long(s);
        }
    }
    const uintptr_t v = n ? (uintptr_t)PyLong_AsUnsignedLongLongMask(n) : 0;
    Py_XDECREF(n);
    if (PyErr_Occurred()) *ok = false;
    return reinterpret_cast<void*>(v);
}

// The C call, without the interpreter lock (a launch waits while the queue is full).
template <typename F>
bool call(const char* where, F&& f) {
    int rc;
    Py_BEGIN_ALLOW_THREADS;
    rc = f();
    Py_END_ALLOW_THREADS;
    if (rc == LLMI_OK) return true;
    PyObject* r = PyObject_CallFunction(g_check_status, "is", rc, where);
    if (r) {
        Py_DECREF(r);
        PyErr_Format(PyExc_RuntimeError, "%s failed with status %d", where, rc);
    }
    return false;
}

// ---- entry points ----
constexpr uint64_t kMhaKeywords =
    bits({k_stream, k_layer_id, k_pos, k_kv_dim, k_kv_mul, k_head_num, k_head_dim, k_max_seq_len, k_kv_layout, k_force_path, k_num_splits,
          k_waves_per_group, k_output_f32, k_pos_device, k_workspace_side});
constexpr uint64_t kMhaRequired = bits({k_layer_id, k_pos, k_kv_dim, k_kv_mul, k_head_num, k_head_dim, k_max_seq_len});

void fill_mha(PyObject* const* vals, Key query, llmi_mha_args* a, bool* ok) {
    a->query = address(vals, query, Kind::bf16, ok);
    a->key_cache = address(vals, k_key_cache, Kind::bf16, ok);
    a->value_cache = address(vals, k_value_cache, Kind::bf16, ok);
    a->output = address(vals, k_output, Kind::bf16, ok);
    a->workspace = address(vals, k_workspace, Kind::f32, ok);
    if (a->workspace) a->workspace_bytes = THPVariable_Unpack(vals[k_workspace]).nbytes();
    a->output_f32 = static_cast<float*>(address(vals, k_output_f32, Kind::f32, ok));
    a->layer_id = int32(vals, k_layer_id, 0, ok);
    a->pos = int32(vals, k_pos, 0, ok);
    a->kv_dim = int32(vals, k_kv_dim, 0, ok);
    a->kv_mul = int32(vals, k_kv_mul, 0, ok);
    a->head_num = int32(vals, k_head_num, 0, ok);
    a->head_dim = int32(vals, k_head_dim, 0, ok);
    a->max_seq_len = int32(vals, k_max_seq_len, 0, ok);
    a->kv_layout = int32(vals, k_kv_layout, LLMI_KV_LAYOUT_POS_MAJOR, ok);
    a->force_path = int32(vals, k_force_path, LLMI_PATH_AUTO, ok);
    a->num_splits = int32(vals, k_num_splits, 0, ok);
    a->waves_per_group = int32(vals, k_waves_per_group, 0, ok);
    a->pos_device = static_cast<const int32_t*>(tensor_or_address(vals, k_pos_device, ok));
    a->workspace_side = int32(vals, k_workspace_side, 0, ok);
    a->stream = stream_of(vals, ok);
}

void fill_append(PyObject* const* vals, llmi_mha_append_args* a, bool* ok) {
    fill_mha(vals, k_query_raw, &a->mha, ok);
    a->key_new = address(vals, k_key_new, Kind::bf16, ok);
    a->value_new = address(vals, k_value_new, Kind::bf16, ok);
    a->norm_weight = address(vals, k_norm_weight, Kind::bf16, ok);
    a->sin_cache = static_cast<const float*>(address(vals, k_sin_cache, Kind::f32, ok));
    a->cos_cache = static_cast<const float*>(address(vals, k_cos_cache, Kind::f32, ok));
    a->eps = 1e-6f;
    if (*ok && vals[k_eps]) {
        a->eps = (float)PyFloat_AsDouble(vals[k_eps]);
        if (PyErr_Occurred()) *ok = false;
    }
}

#define LLMI_ENTRY(name) PyObject* name(PyObject*, PyObject* const* args, Py_ssize_t n_args, PyObject* names)
#define LLMI_PARSE(sig)              \
    PyObject* vals[kKeys];           \
    if (!parse(sig, args, n_args, names, vals)) return nullptr; \
    bool ok = true

constexpr Key kDecodePos[] = {k_query, k_key_cache, k_value_cache, k_output, k_workspace};
const Signature kDecodeSig = {"mha_decode", kDecodePos, 5, kMhaKeywords,
                              kMhaRequired | bits({k_query, k_key_cache, k_value_cache, k_output, k_workspace})};
LLMI_ENTRY(mha_decode) {
    LLMI_PARSE(kDecodeSig);
    llmi_mha_args a{};
    fill_mha(vals, k_query, &a, &ok);
    if (!ok || !call("llmi_hip_mha_decode", [&] { return g_abi.mha_decode(&a); })) return nullptr;
    return Py_NewRef(vals[k_output]);
}

constexpr Key kAppendPos[] = {k_query_raw, k_key_new, k_value_new, k_norm_weight, k_sin_cache, k_cos_cache, k_key_cache, k_value_cache,
                              k_output, k_workspace};
constexpr uint64_t kAppendRequired = kMhaRequired | bits({k_query_raw, k_key_new, k_value_new, k_norm_weight, k_sin_cache, k_cos_cache,
                                                          k_key_cache, k_value_cache, k_output, k_workspace});
const Signature kAppendSig = {"mha_decode_append", kAppendPos, 10, kMhaKeywords | bits({k_eps, k_o_weight, k_residual, k_one_launch}),
                              kAppendRequired};
LLMI_ENTRY(mha_decode_append) {
    LLMI_PARSE(kAppendSig);
    llmi_attn_oproj_args t{};
    fill_append(vals, &t.attn, &ok);
    if (!ok) return nullptr;
    if (!vals[k_o_weight] || vals[k_o_weight] == Py_None) {
        if (!call("llmi_hip_mha_decode_append", [&] { return g_abi.mha_decode_append(&t.attn); })) return nullptr;
        return Py_NewRef(vals[k_output]);
    }
    t.o_weight = address(vals, k_o_weight, Kind::bf16, &ok);
    t.residual = address(vals, k_residual, Kind::bf16, &ok);
    if (!ok) return nullptr;
    if (t.residual) t.hidden = (int32_t)THPVariable_Unpack(vals[k_residual]).numel();
    if (vals[k_one_launch]) {
        const int yes = PyObject_IsTrue(vals[k_one_launch]);
        if (yes < 0) return nullptr;
        t.one_launch = yes;
    }
    const int launches = t.one_launch ? g_abi.mha_oproj_launches(&t) : 2;  // (invalid arguments: the call says so)
    if (!call("llmi_hip_mha_decode_append_oproj", [&] { return g_abi.mha_decode_append_oproj(&t); })) return nullptr;
    return PyLong_FromLong(launches);
}

const Signature kStackSig = {"mha_decode_append_stack", kAppendPos, 10,
                             kMhaKeywords | bits({k_eps, k_layer_count, k_query_stride, k_key_new_stride, k_value_new_stride,
                                                  k_norm_weight_stride, k_output_stride}),
                             kAppendRequired | bits({k_layer_count, k_query_stride, k_key_new_stride, k_value_new_stride,
                                                     k_norm_weight_stride, k_output_stride})};
LLMI_ENTRY(mha_decode_append_stack) {
    LLMI_PARSE(kStackSig);
    llmi_mha_stack_args t{};
    fill_append(vals, &t.first, &ok);
    t.layer_count = int32(vals, k_layer_count, 0, &ok);
    t.query_stride = int64(vals, k_query_stride, 0, &ok);
    t.key_new_stride = int64(vals, k_key_new_stride, 0, &ok);
    t.value_new_stride = int64(vals, k_value_new_stride, 0, &ok);
    t.norm_weight_stride = int64(vals, k_norm_weight_stride, 0, &ok);
    t.output_stride = int64(vals, k_output_stride, 0, &ok);
    if (!ok) return nullptr;
    const int launches = g_abi.mha_stack_launches(&t);
    if (!call("llmi_hip_mha_decode_append_stack", [&] { return g_abi.mha_decode_append_stack(&t); })) return nullptr;
    return PyLong_FromLong(launches);
}

constexpr Key kNormRopePos[] = {k_query, k_key_new, k_value_new, k_key_cache, k_value_cache, k_norm_weight, k_sin_cache, k_cos_cache};
const Signature kNormRopeSig = {
    "qk_norm_rope_append", kNormRopePos, 8,
    bits({k_layer_id, k_pos, k_kv_dim, k_head_num, k_head_dim, k_max_seq_len, k_kv_layout, k_eps, k_query_src, k_stream}),
    bits({k_query, k_key_new, k_value_new, k_key_cache, k_value_cache, k_norm_weight, k_sin_cache, k_cos_cache, k_layer_id, k_pos, k_kv_dim,
          k_head_num, k_head_dim, k_max_seq_len})};
LLMI_ENTRY(qk_norm_rope_append) {
    LLMI_PARSE(kNormRopeSig);
    llmi_qk_norm_rope_args a{};
    a.query = address(vals, k_query, Kind::bf16, &ok);
    a.query_src = address(vals, k_query_src, Kind::bf16, &ok);
    a.key_new = address(vals, k_key_new, Kind::bf16, &ok);
    a.value_new = address(vals, k_value_new, Kind::bf16, &ok);
    a.key_cache = address(vals, k_key_cache, Kind::bf16, &ok);
    a.value_cache = address(vals, k_value_cache, Kind::bf16, &ok);
    a.norm_weight = address(vals, k_norm_weight, Kind::bf16, &ok);
    a.sin_cache = static_cast<const float*>(address(vals, k_sin_cache, Kind::f32, &ok));
    a.cos_cache = static_cast<const float*>(address(vals, k_cos_cache, Kind::f32, &ok));
    a.layer_id = int32(vals, k_layer_id, 0, &ok);
    a.pos = int32(vals, k_pos, 0, &ok);
    a.kv_dim = int32(vals, k_kv_dim, 0, &ok);
    a.head_num = int32(vals, k_head_num, 0, &ok);
    a.head_dim = int32(vals, k_head_dim, 0, &ok);
    a.max_seq_len = int32(vals, k_max_seq_len, 0, &ok);
    a.kv_layout = int32(vals, k_kv_layout, LLMI_KV_LAYOUT_POS_MAJOR, &ok);
    a.eps = 1e-6f;
    if (ok && vals[k_eps]) {
        a.eps = (float)PyFloat_AsDouble(vals[k_eps]);
        if (PyErr_Occurred()) ok = false;
    }
    a.stream = stream_of(vals, &ok);
    if (!ok || !call("llmi_hip_qk_norm_rope_append", [&] { return g_abi.qk_norm_rope_append(&a); })) return nullptr;
    Py_RETURN_NONE;
}

constexpr Key kRestridePos[] = {k_src_pos_major, k_dst_head_major};
const Signature kRestrideSig = {
    "kv_restride", kRestridePos, 2, bits({k_layer_num, k_max_seq_len, k_kv_dim, k_head_dim, k_num_pos, k_stream}),
    bits({k_src_pos_major, k_dst_head_major, k_layer_num, k_max_seq_len, k_kv_dim, k_head_dim, k_num_pos})};
LLMI_ENTRY(kv_restride) {
    LLMI_PARSE(kRestrideSig);
    const void* src = address(vals, k_src_pos_major, Kind::bf16, &ok);
    void* dst = address(vals, k_dst_head_major, Kind::bf16, &ok);
    if (ok && src && dst &&
        THPVariable_Unpack(vals[k_dst_head_major]).numel() < THPVariable_Unpack(vals[k_src_pos_major]).numel()) {
        PyErr_SetString(PyExc_ValueError, "destination cache is smaller than the source");
        return nullptr;
    }
    const int32_t layers = int32(vals, k_layer_num, 0, &ok), msl = int32(vals, k_max_seq_len, 0, &ok), kv_dim = int32(vals, k_kv_dim, 0, &ok);
    const int32_t head_dim = int32(vals, k_head_dim, 0, &ok), num_pos = int32(vals, k_num_pos, 0, &ok);
    void* stream = stream_of(vals, &ok);
    if (!ok || !call("llmi_hip_kv_restride", [&] { return g_abi.kv_restride(src, dst, layers, msl, kv_dim, head_dim, num_pos, stream); }))
        return nullptr;
    return Py_NewRef(vals[k_dst_head_major]);
}

constexpr Key kGemvPos[] = {k_input, k_weight, k_output};
const Signature kGemvSig = {"gemv", kGemvPos, 3, bits({k_mode, k_stream}), bits({k_input, k_weight, k_output})};
LLMI_ENTRY(gemv) {
    LLMI_PARSE(kGemvSig);
    llmi_gemv_args a{};
    a.mode = int32(vals, k_mode, LLMI_GEMV_OUT_BF16, &ok);
    a.input = address(vals, k_input, Kind::bf16, &ok);
    a.weight = address(vals, k_weight, Kind::bf16, &ok);
    a.output = address(vals, k_output, a.mode == LLMI_GEMV_OUT_F32 ? Kind::f32 : Kind::bf16, &ok);
    if (!ok) return nullptr;
    if (!a.weight || THPVariable_Unpack(vals[k_weight]).dim() < 2) {
        PyErr_SetString(PyExc_ValueError, "weight must be a [n][k] tensor");
        return nullptr;
    }
    const at::Tensor& w = THPVariable_Unpack(vals[k_weight]);
    a.n = (int32_t)w.sizes()[0];
    a.k = (int32_t)w.sizes()[1];
    a.stream = stream_of(vals, &ok);
    if (!ok || !call("llmi_hip_gemv", [&] { return g_abi.gemv(&a); })) return nullptr;
    return Py_NewRef(vals[k_output]);
}

constexpr Key kQkvPos[] = {k_input, k_weight, k_query, k_key, k_value};
const Signature kQkvSig = {"qkv_gemv", kQkvPos, 5, bits({k_stream}), bits({k_input, k_weight, k_query, k_key, k_value})};
LLMI_ENTRY(qkv_gemv) {
    LLMI_PARSE(kQkvSig);
    llmi_qkv_gemv_args a{};
    a.input = address(vals, k_input, Kind::bf16, &ok);
    a.weight = address(vals, k_weight, Kind::bf16, &ok);
    a.query = address(vals, k_query, Kind::bf16, &ok);
    a.key = address(vals, k_key, Kind::bf16, &ok);
    a.value = address(vals, k_value, Kind::bf16, &ok);
    if (!ok) return nullptr;
    if (!a.weight || !a.query || !a.key || !a.value || THPVariable_Unpack(vals[k_weight]).dim() < 2) {
        PyErr_SetString(PyExc_ValueError, "weight must be a [dim + 2*kv_dim][k] tensor and query, key, value tensors");
        return nullptr;
    }
    const at::Tensor& w = THPVariable_Unpack(vals[k_weight]);
    const int64_t dim = THPVariable_Unpack(vals[k_query]).numel(), kv_dim = THPVariable_Unpack(vals[k_key]).numel();
    if (THPVariable_Unpack(vals[k_value]).numel() != kv_dim || w.sizes()[0] != dim + 2 * kv_dim) {
        PyErr_SetString(PyExc_AssertionError, "weight rows do not add up to query + key + value");
        return nullptr;
    }
    a.dim = (int32_t)dim;
    a.kv_dim = (int32_t)kv_dim;
    a.k = (int32_t)w.sizes()[1];
    a.stream = stream_of(vals, &ok);
    if (!ok || !call("llmi_hip_qkv_gemv", [&] { return g_abi.qkv_gemv(&a); })) return nullptr;
    Py_RETURN_NONE;
}

// bind(functions, get_device, get_stream, check_dev, check_status, bf16_types, f32_types); functions: C ABI name -> address
PyObject* bind(PyObject*, PyObject* args) {
    PyObject *functions, *objs[6];
    if (!PyArg_ParseTuple(args, "O!OOOOOO", &PyDict_Type, &functions, &objs[0], &objs[1], &objs[2], &objs[3], &objs[4], &objs[5])) return nullptr;
    struct {
        const char* name;
        void* slot;
    } wanted[] = {{"llmi_hip_mha_decode", &g_abi.mha_decode},
                  {"llmi_hip_mha_decode_append", &g_abi.mha_decode_append},
                  {"llmi_hip_mha_decode_append_oproj", &g_abi.mha_decode_append_oproj},
                  {"llmi_hip_mha_oproj_launches", &g_abi.mha_oproj_launches},
                  {"llmi_hip_mha_decode_append_stack", &g_abi.mha_decode_append_stack},
                  {"llmi_hip_mha_stack_launches", &g_abi.mha_stack_launches},
                  {"llmi_hip_qk_norm_rope_append", &g_abi.qk_norm_rope_append},
                  {"llmi_hip_kv_restride", &g_abi.kv_restride},
                  {"llmi_hip_gemv", &g_abi.gemv},
                  {"llmi_hip_qkv_gemv", &g_abi.qkv_gemv}};
    for (const auto& w : wanted) {
        PyObject* n = PyDict_GetItemString(functions, w.name);  // borrowed
        void* p = n ? PyLong_AsVoidPtr(n) : nullptr;
        if (PyErr_Occurred()) return nullptr;
        if (!p) {
            PyErr_Format(PyExc_ValueError, "bind: no address for %s", w.name);
            return nullptr;
        }
        *static_cast<void**>(w.slot) = p;
    }
    PyObject** const keep[] = {&g_get_device, &g_get_stream, &g_check_dev, &g_check_status, &g_bf16_types, &g_f32_types};
    for (int i = 0; i < 6; ++i) {
        Py_INCREF(objs[i]);
        Py_XSETREF(*keep[i], objs[i]);
    }
    return PyLong_FromLong(LLMI_HIP_ABI_VERSION);
}

// What torch throws at a tensor without storage of its own (one under vmap, say) is a Python error, not the process's end.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t, PyObject*)>
PyObject* entry(PyObject* self, PyObject* const* args, Py_ssize_t n_args, PyObject* names) {
    HANDLE_TH_ERRORS
    return F(self, args, n_args, names);
    END_HANDLE_TH_ERRORS
}

#define LLMI_METHOD(name, signature, doc) \
    {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(entry<name>)), METH_FASTCALL | METH_KEYWORDS, #name signature "\n--\n\n" doc}

PyMethodDef g_methods[] = {
    {"bind", bind, METH_VARARGS, "Hands over the C ABI's addresses and the Python side's helpers; returns the ABI version compiled in."},
    LLMI_METHOD(mha_decode, "($module, query, key_cache, value_cache, output, workspace, *, stream=None, layer_id, pos, kv_dim, kv_mul, "
                            "head_num, head_dim, max_seq_len, kv_layout=0, force_path=0, num_splits=0, waves_per_group=0, output_f32=None, "
                            "pos_device=None, workspace_side=0)",
                "Decode attention for one layer / one token on the current (or given) stream."),
    LLMI_METHOD(mha_decode_append,
                "($module, query_raw, key_new, value_new, norm_weight, sin_cache, cos_cache, key_cache, value_cache, output, workspace, *, "
                "eps=1e-06, stream=None, o_weight=None, residual=None, one_launch=False, layer_id, pos, kv_dim, kv_mul, head_num, head_dim, "
                "max_seq_len, kv_layout=0, force_path=0, num_splits=0, waves_per_group=0, output_f32=None, pos_device=None, workspace_side=0)",
                "QK-Norm + RoPE + K/V append + decode attention as one kernel (llmi_hip_mha_decode_append). With `o_weight`\n"
                "[hidden][head_num*128] and `residual` [hidden]: llmi_hip_mha_decode_append_oproj (`one_launch`: ask for its\n"
                "one-launch form); returns the launch count."),
    LLMI_METHOD(mha_decode_append_stack,
                "($module, query_raw, key_new, value_new, norm_weight, sin_cache, cos_cache, key_cache, value_cache, output, workspace, *, "
                "layer_count, query_stride, key_new_stride, value_new_stride, norm_weight_stride, output_stride, eps=1e-06, stream=None, "
                "layer_id, pos, kv_dim, kv_mul, head_num, head_dim, max_seq_len, kv_layout=0, force_path=0, num_splits=0, waves_per_group=0, "
                "output_f32=None, pos_device=None, workspace_side=0)",
                "llmi_hip_mha_decode_append for `layer_count` consecutive layers (llmi_hip_mha_decode_append_stack): the tensors\n"
                "are the first layer's, layer l uses them moved on by l strides (elements). Returns the launch count."),
    LLMI_METHOD(qk_norm_rope_append,
                "($module, query, key_new, value_new, key_cache, value_cache, norm_weight, sin_cache, cos_cache, *, layer_id, pos, kv_dim, "
                "head_num, head_dim, max_seq_len, kv_layout=0, eps=1e-06, query_src=None, stream=None)",
                "QK-Norm + RoPE of the query and the new K row, K and V rows to the cache (llmi_hip_qk_norm_rope_append)."),
    LLMI_METHOD(kv_restride, "($module, src_pos_major, dst_head_major, *, layer_num, max_seq_len, kv_dim, head_dim, num_pos, stream=None)",
                "Position-major cache rows into a head-major cache (llmi_hip_kv_restride); returns the destination."),
    LLMI_METHOD(gemv, "($module, input, weight, output, *, mode=0, stream=None)",
                "output = weight @ input (bf16 [n][k] x bf16 [k], fp32 accumulate): bf16 or fp32 output, or the\n"
                "bf16 residual in `output` updated in place (llmi_hip_gemv)."),
    LLMI_METHOD(qkv_gemv, "($module, input, weight, query, key, value, *, stream=None)",
                "The packed QKV projection: rows [0, dim) of weight @ input go to query, the next kv_dim to key,\n"
                "the last kv_dim to value (llmi_hip_qkv_gemv)."),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_torch_ops", "Native calls of llminfer_amd.ops.", -1, g_methods};

}  // namespace

PyMODINIT_FUNC PyInit__torch_ops() {
    for (int s = 0; s < kSlots; ++s) g_slot[s] = -1;
    for (int k = 0; k < kKeys; ++k) {
        g_key[k] = PyUnicode_InternFromString(kKeyText[k]);
        if (!g_key[k]) return nullptr;
        unsigned s = slot_of(g_key[k]);
        while (g_slot[s] >= 0) s = (s + 1) % kSlots;
        g_slot[s] = (int8_t)k;
    }
    return PyModule_Create(&g_module);
}
