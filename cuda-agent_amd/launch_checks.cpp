// The per-launch host work of capi.py in native code: checks of the tensors, their pointers and sizes, the current stream
// and the call of the launcher. A decode step of a small layer is bound by this (one GDN step of 7 tensors took 6.0 us of
// host time through Python and ctypes, for a kernel of 3.0 us; 3.5 here, most of it the launch itself).
//
// Every function takes the arguments of the helper of the same name in capi.py and returns 0 (launched), the launcher's
// status (rejected, nothing launched) or -1: not for this path, nothing launched. The helper then goes its own way, which
// handles or refuses whatever is not an ordinary call: tensor subclasses, a stream of the caller's, tensors of other
// types, shapes or devices, sizes beyond int.
#include <Python.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <climits>

#include "../include/cuda_agent_amd.h"

namespace {

constexpr int DECLINED = -1;
struct Decline {};

inline void need(bool condition) {
    if (!condition) throw Decline{};
}

constexpr auto BF16 = at::kBFloat16;
constexpr auto F32 = at::kFloat;
constexpr auto I32 = at::kInt;
constexpr auto U8 = at::kByte;

// A contiguous tensor on a GPU, or none where the argument may be None
class Arg {
 public:
    explicit Arg(PyObject* object, bool optional = false) {
        if (optional && object == Py_None) return;
        need(THPVariable_CheckExact(object));
        t_ = &THPVariable_Unpack(object);
        need(t_->is_cuda() && t_->is_contiguous());
        for (const int64_t size : t_->sizes()) need(size <= INT_MAX);
    }
    explicit operator bool() const { return t_ != nullptr; }
    void* ptr() const { return t_ ? t_->data_ptr() : nullptr; }
    template <typename T>
    T* as() const { return static_cast<T*>(ptr()); }
    int size(int i) const {
        need(i < t_->dim());
        return (int)t_->size(i);
    }
    at::ScalarType type() const { return t_->scalar_type(); }
    size_t bytes() const { return (size_t)t_->numel() * t_->element_size(); }
    // type and shape
    const Arg& is(at::ScalarType type, at::IntArrayRef shape) const {
        need(t_->scalar_type() == type && t_->sizes() == shape);
        return *this;
    }
    const Arg& is_byte(at::IntArrayRef shape) const {
        need(t_->element_size() == 1 && t_->sizes() == shape);
        return *this;
    }
    const Arg& is_e4m3(at::IntArrayRef shape) const {
        need((type() == U8 || type() == at::kFloat8_e4m3fn) && t_->sizes() == shape);
        return *this;
    }
    const Arg& dims(int n) const {
        need(t_->dim() == n);
        return *this;
    }

 private:
    const at::Tensor* t_ = nullptr;
};

int integer(PyObject* object) {
    need(PyLong_CheckExact(object));
    int overflow;
    const long v = PyLong_AsLongAndOverflow(object, &overflow);
    need(overflow == 0 && v >= INT_MIN && v <= INT_MAX);
    return (int)v;
}

float real(PyObject* object) {
    need(PyFloat_CheckExact(object));
    return (float)PyFloat_AS_DOUBLE(object);
}

hipStream_t stream(PyObject* object) {
    need(object == Py_None);
    return c10::hip::getCurrentHIPStream().stream();
}

// The call itself, without the interpreter's lock: it waits when the stream's queue is full.
template <typename... P, typename... A>
void launch(void (*launcher)(P...), A... args) {
    PyThreadState* const thread = PyEval_SaveThread();
    launcher(args...);
    PyEval_RestoreThread(thread);
}

int qkv_type(const Arg& a) {
    need(a.type() == F32 || a.type() == BF16);
    return a.type() == F32 ? 0 : 1;
}

int out_type(const Arg& a) {
    need(a.type() == F32 || a.type() == BF16);
    return a.type() == BF16 ? 0 : 1;
}

struct GdnSizes {
    int B, Hv, Hqk, dk, dv;
};

// state, q, k, v of the three GDN entry points
GdnSizes gdn_sizes(const Arg& state, const Arg& q, const Arg& k, const Arg& v) {
    const GdnSizes s{state.dims(4).size(0), state.size(1), q.size(1), state.size(2), state.size(3)};
    state.is(F32, {s.B, s.Hv, s.dk, s.dv});
    q.is(q.type(), {s.B, s.Hqk, s.dk});
    k.is(q.type(), {s.B, s.Hqk, s.dk});
    v.is(q.type(), {s.B, s.Hv, s.dv});
    return s;
}

void gdn_decode(PyObject* const* a) {
    const Arg o(a[0]), state(a[1]), q(a[2]), k(a[3]), v(a[4]), g(a[5]), beta(a[6]);
    const GdnSizes s = gdn_sizes(state, q, k, v);
    o.is(F32, {s.B, s.Hv, s.dv}), g.is(F32, {s.B, s.Hv}), beta.is(F32, {s.B, s.Hv});
    launch(gdn_decode_launcher, o.as<float>(), state.as<float>(), q.ptr(), k.ptr(), v.ptr(), g.as<float>(), beta.as<float>(), s.B, s.Hv,
                        s.Hqk, s.dk, s.dv, qkv_type(q), integer(a[7]), stream(a[8]));
}

void gdn_decode_fused(PyObject* const* a) {
    const Arg o(a[0]), state(a[1]), q(a[2]), k(a[3]), v(a[4]), ga(a[5]), gb(a[6]), a_log(a[7]), dt_bias(a[8]);
    const GdnSizes s = gdn_sizes(state, q, k, v);
    o.is(F32, {s.B, s.Hv, s.dv}), ga.is(F32, {s.B, s.Hv}), gb.is(F32, {s.B, s.Hv});
    a_log.is(F32, {s.Hv}), dt_bias.is(F32, {s.Hv});
    launch(gdn_decode_fused_launcher, o.as<float>(), state.as<float>(), q.ptr(), k.ptr(), v.ptr(), ga.as<float>(), gb.as<float>(),
                              a_log.as<float>(), dt_bias.as<float>(), s.B, s.Hv, s.Hqk, s.dk, s.dv, qkv_type(q), integer(a[9]),
                              stream(a[10]));
}

void gdn_decode_fused_norm(PyObject* const* a) {
    const Arg out(a[0]), state(a[1]), q(a[2]), k(a[3]), v(a[4]), ga(a[5]), gb(a[6]), a_log(a[7]), dt_bias(a[8]), z(a[9]),
        norm_w(a[10]);
    const GdnSizes s = gdn_sizes(state, q, k, v);
    ga.is(F32, {s.B, s.Hv}), gb.is(F32, {s.B, s.Hv}), a_log.is(F32, {s.Hv}), dt_bias.is(F32, {s.Hv});
    out.is(q.type(), {s.B, s.Hv, s.dv}), z.is(q.type(), {s.B, s.Hv, s.dv}), norm_w.is(q.type(), {s.dv});
    launch(gdn_decode_fused_norm_launcher, out.ptr(), state.as<float>(), q.ptr(), k.ptr(), v.ptr(), ga.as<float>(), gb.as<float>(),
                                   a_log.as<float>(), dt_bias.as<float>(), z.ptr(), norm_w.ptr(), real(a[11]), s.B, s.Hv, s.Hqk,
                                   s.dk, s.dv, qkv_type(q), integer(a[12]), stream(a[13]));
}

void causal_conv1d_update(PyObject* const* a) {
    const Arg q(a[0], true), k(a[1], true), v(a[2]), state(a[3]), x(a[4]), weight(a[5]), bias(a[6], true);
    const int B = state.dims(3).size(0), C = state.size(1), L = state.size(2), K = weight.dims(2).size(1);
    const int type = qkv_type(state);
    need((bool)q == (bool)k);
    const int key_dim = q ? q.dims(2).size(1) : 0, value_dim = v.dims(2).size(1);
    need(2L * key_dim + value_dim == C);
    if (q) q.is(state.type(), {B, key_dim}), k.is(state.type(), {B, key_dim});
    v.is(state.type(), {B, value_dim}), x.is(state.type(), {B, C}), weight.is(state.type(), {C, K});
    if (bias) bias.is(state.type(), {C});
    need(a[7] == Py_True || a[7] == Py_False);
    launch(causal_conv1d_update_launcher, q.ptr(), k.ptr(), v.ptr(), state.ptr(), x.ptr(), weight.ptr(), bias.ptr(), B, key_dim, value_dim,
                                  L, K, a[7] == Py_True ? 1 : 0, type, integer(a[8]), stream(a[9]));
}

constexpr int LATENT_ROW_BYTES = 656;

// out, q, kv, idx, workspace, scale, config, stream
template <bool FP8>
void sparse_mla_decode(PyObject* const* a) {
    const Arg out(a[0]), q(a[1]), kv(a[2]), idx(a[3]), workspace(a[4]);
    const int B = q.dims(3).size(0), H = q.size(1), d = q.size(2), N = kv.dims(3).size(1), topk = idx.dims(2).size(1);
    const int d_v = out.dims(3).size(2), type = out_type(out);
    q.is(BF16, {B, H, d}), idx.is(I32, {B, topk}), out.is(out.type(), {B, H, d_v});
    kv.is(FP8 ? U8 : BF16, {B, N, FP8 ? LATENT_ROW_BYTES : d});
    if (FP8) need(workspace.type() == U8);
    const auto launcher = FP8 ? sparse_mla_decode_fp8_launcher : sparse_mla_decode_launcher;
    launch(launcher, out.ptr(), q.ptr(), kv.ptr(), idx.as<int>(), workspace.ptr(), workspace.bytes(), B, H, N, topk, d, d_v, real(a[5]),
             type, integer(a[6]), stream(a[7]));
}

// out, q, kv_pool, block_table, idx, workspace, scale, config, stream
template <bool FP8>
void sparse_mla_decode_paged(PyObject* const* a) {
    const Arg out(a[0]), q(a[1]), pool(a[2]), table(a[3], true), idx(a[4]), workspace(a[5]);
    const int B = q.dims(3).size(0), H = q.size(1), d = q.size(2), topk = idx.dims(2).size(1);
    const int n_pages = pool.dims(3).size(0), page = pool.size(1), d_v = out.dims(3).size(2), type = out_type(out);
    q.is(BF16, {B, H, d}), idx.is(I32, {B, topk}), out.is(out.type(), {B, H, d_v});
    pool.is(FP8 ? U8 : BF16, {n_pages, page, FP8 ? LATENT_ROW_BYTES : d});
    const int max_pages = table ? table.dims(2).size(1) : 0;
    if (table) table.is(I32, {B, max_pages});
    const auto launcher = FP8 ? sparse_mla_decode_fp8_paged_launcher : sparse_mla_decode_paged_launcher;
    launch(launcher, out.ptr(), q.ptr(), pool.ptr(), table.as<int>(), idx.as<int>(), workspace.ptr(), workspace.bytes(), B, H, n_pages,
             page, max_pages, topk, d, d_v, real(a[6]), type, integer(a[7]), stream(a[8]));
}

const int* lengths_of(const Arg& lengths, int B) {
    if (lengths) lengths.is(I32, {B});
    return lengths.as<int>();
}

// scores, q, k_cache, w, lengths, scale, stream
void mla_index_scores(PyObject* const* a) {
    const Arg scores(a[0]), q(a[1]), keys(a[2]), w(a[3]), lengths(a[4], true);
    const int B = q.dims(3).size(0), Hi = q.size(1), D = q.size(2), N = keys.dims(3).size(1);
    q.is(BF16, {B, Hi, D}), keys.is(BF16, {B, N, D}), w.is(F32, {B, Hi}), scores.is(F32, {B, N});
    launch(mla_index_scores_launcher, scores.as<float>(), q.ptr(), keys.ptr(), w.as<float>(), lengths_of(lengths, B), B, Hi, N, D,
                              real(a[5]), 0, stream(a[6]));
}

// scores, q, k_pool, block_table, w, lengths, scale, stream
void mla_index_scores_paged(PyObject* const* a) {
    const Arg scores(a[0]), q(a[1]), pool(a[2]), table(a[3]), w(a[4]), lengths(a[5], true);
    const int B = q.dims(3).size(0), Hi = q.size(1), D = q.size(2), n_pages = pool.dims(3).size(0), page = pool.size(1);
    const int max_pages = table.dims(2).size(1);
    q.is(BF16, {B, Hi, D}), pool.is(BF16, {n_pages, page, D}), table.is(I32, {B, max_pages}), w.is(F32, {B, Hi});
    scores.is(F32, {B, (int64_t)max_pages * page});
    launch(mla_index_scores_paged_launcher, scores.as<float>(), q.ptr(), pool.ptr(), table.as<int>(), w.as<float>(),
                                    lengths_of(lengths, B), B, Hi, n_pages, page, max_pages, D, real(a[6]), 0, stream(a[7]));
}

// scores, q, k_cache, k_scale, w, lengths, scale, stream
void mla_index_scores_fp8(PyObject* const* a) {
    const Arg scores(a[0]), q(a[1]), keys(a[2]), k_scale(a[3]), w(a[4]), lengths(a[5], true);
    const int B = q.dims(3).size(0), Hi = q.size(1), D = q.size(2), N = keys.dims(3).size(1);
    q.is_e4m3({B, Hi, D}), keys.is_e4m3({B, N, D}), k_scale.is(F32, {B, N}), w.is(F32, {B, Hi}), scores.is(F32, {B, N});
    launch(mla_index_scores_fp8_launcher, scores.as<float>(), q.ptr(), keys.ptr(), k_scale.as<float>(), w.as<float>(),
                                  lengths_of(lengths, B), B, Hi, N, D, real(a[6]), 0, stream(a[7]));
}

// scores, q, k_pool, k_scale_pool, block_table, w, lengths, scale, stream
void mla_index_scores_fp8_paged(PyObject* const* a) {
    const Arg scores(a[0]), q(a[1]), pool(a[2]), k_scale(a[3]), table(a[4]), w(a[5]), lengths(a[6], true);
    const int B = q.dims(3).size(0), Hi = q.size(1), D = q.size(2), n_pages = pool.dims(3).size(0), page = pool.size(1);
    const int max_pages = table.dims(2).size(1);
    q.is_e4m3({B, Hi, D}), pool.is_e4m3({n_pages, page, D}), k_scale.is(F32, {n_pages, page});
    table.is(I32, {B, max_pages}), w.is(F32, {B, Hi}), scores.is(F32, {B, (int64_t)max_pages * page});
    launch(mla_index_scores_fp8_paged_launcher, scores.as<float>(), q.ptr(), pool.ptr(), k_scale.as<float>(), table.as<int>(),
                                        w.as<float>(), lengths_of(lengths, B), B, Hi, n_pages, page, max_pages, D, real(a[7]), 0,
                                        stream(a[8]));
}

void topk_select(PyObject* const* a) {
    const Arg idx(a[0]), scores(a[1]), lengths(a[2], true);
    const int B = scores.dims(2).size(0), n = scores.size(1), k = idx.dims(2).size(1);
    scores.is(F32, {B, n}), idx.is(I32, {B, k});
    launch(topk_select_launcher, idx.as<int>(), scores.as<float>(), lengths_of(lengths, B), B, n, k, 0, stream(a[3]));
}

// out, x, logits, w13_q, w13_s, w2_q, w2_s, workspace, top_k, config, stream; SHARED: one expert more is stored than routed to
template <bool SHARED>
void moe_fp8(PyObject* const* a) {
    const Arg out(a[0]), x(a[1]), logits(a[2]), w13(a[3]), w13_s(a[4]), w2(a[5]), w2_s(a[6]), workspace(a[7]);
    const int T = x.dims(2).size(0), H = x.size(1), stored = w13.dims(3).size(0), I = w13.size(1) / 2;
    const int E = SHARED ? stored - 1 : stored, type = out_type(out);
    x.is(BF16, {T, H}), logits.is(F32, {T, E}), out.is(out.type(), {T, H});
    w13.is_byte({stored, 2 * (int64_t)I, H}), w2.is_byte({stored, H, I});
    w13_s.is(F32, {stored, 2 * (int64_t)I / 128, H / 128}), w2_s.is(F32, {stored, H / 128, I / 128});
    const auto launcher = SHARED ? moe_fp8_fused_shared_launcher : moe_fp8_launcher;
    launch(launcher, out.ptr(), x.ptr(), logits.as<float>(), w13.ptr(), w13_s.as<float>(), w2.ptr(), w2_s.as<float>(), workspace.ptr(),
             workspace.bytes(), T, H, I, E, integer(a[8]), type, integer(a[9]), stream(a[10]));
}

void moe_rmsnorm_quant(PyObject* const* a) {
    const Arg q(a[0]), scales(a[1]), y(a[2], true), x(a[3]), weight(a[4]);
    const int R = x.dims(2).size(0), C = x.size(1);
    x.is(BF16, {R, C}), weight.is(BF16, {C}), q.is_byte({R, C}), scales.is(F32, {R, C / 128});
    if (y) y.is(BF16, {R, C});
    launch(moe_rmsnorm_quant_launcher, q.ptr(), scales.as<float>(), y.ptr(), x.ptr(), weight.ptr(), real(a[5]), R, C, integer(a[6]),
                               stream(a[7]));
}

// logits, x, w or planes, workspace, stream
template <bool SPLIT>
void moe_router_logits(PyObject* const* a) {
    const Arg logits(a[0]), x(a[1]), w(a[2]), workspace(a[3], true);
    const int T = x.dims(2).size(0), H = x.size(1), E = w.dims(SPLIT ? 3 : 2).size(SPLIT ? 1 : 0);
    logits.is(F32, {T, E});
    const size_t bytes = workspace ? workspace.bytes() : 0;
    if (SPLIT) {
        x.is(BF16, {T, H}), w.is(BF16, {3, E, H});
        launch(moe_router_logits_split_launcher, logits.as<float>(), x.ptr(), w.ptr(), workspace.ptr(), bytes, T, H, E, 0, stream(a[4]));
    } else {
        w.is(F32, {E, H});
        launch(moe_router_logits_launcher, logits.as<float>(), x.ptr(), w.as<float>(), workspace.ptr(), bytes, T, H, E, qkv_type(x), 0,
                                   stream(a[4]));
    }
}

// ids, weights, logits, bias, n_group, topk_group, normalise, routed_scaling_factor, stream
void moe_route_grouped(PyObject* const* a) {
    const Arg ids(a[0]), weights(a[1]), logits(a[2]), bias(a[3], true);
    const int T = logits.dims(2).size(0), E = logits.size(1), top_k = ids.dims(2).size(1);
    logits.is(F32, {T, E}), ids.is(I32, {T, top_k}), weights.is(F32, {T, top_k});
    if (bias) bias.is(F32, {E});
    need(a[6] == Py_True || a[6] == Py_False);
    launch(moe_route_grouped_launcher, ids.as<int>(), weights.as<float>(), logits.as<float>(), bias.as<float>(), T, E, top_k,
                               integer(a[4]), integer(a[5]), a[6] == Py_True ? 1 : 0, real(a[7]), 0, stream(a[8]));
}

template <void (*F)(PyObject* const*), int ARGS>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != ARGS) {
        PyErr_Format(PyExc_TypeError, "%d arguments expected, %zd given", ARGS, n);
        return nullptr;
    }
    int result;
    try {
        F(args);
        result = cuda_agent_amd_last_status();
    } catch (...) {  // declined, or a tensor that has no memory: its own error is raised on the other way
        result = DECLINED;
    }
    return PyLong_FromLong(result);
}

#define ENTRY(name, function, args) {name, (PyCFunction)(void (*)())entry<function, args>, METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    ENTRY("gdn_decode", gdn_decode, 9),
    ENTRY("gdn_decode_fused", gdn_decode_fused, 11),
    ENTRY("gdn_decode_fused_norm", gdn_decode_fused_norm, 14),
    ENTRY("causal_conv1d_update", causal_conv1d_update, 10),
    ENTRY("sparse_mla_decode", sparse_mla_decode<false>, 8),
    ENTRY("sparse_mla_decode_fp8", sparse_mla_decode<true>, 8),
    ENTRY("sparse_mla_decode_paged", sparse_mla_decode_paged<false>, 9),
    ENTRY("sparse_mla_decode_fp8_paged", sparse_mla_decode_paged<true>, 9),
    ENTRY("mla_index_scores", mla_index_scores, 7),
    ENTRY("mla_index_scores_paged", mla_index_scores_paged, 8),
    ENTRY("mla_index_scores_fp8", mla_index_scores_fp8, 8),
    ENTRY("mla_index_scores_fp8_paged", mla_index_scores_fp8_paged, 9),
    ENTRY("topk_select", topk_select, 4),
    ENTRY("moe_fp8", moe_fp8<false>, 11),
    ENTRY("moe_fp8_fused_shared", moe_fp8<true>, 11),
    ENTRY("moe_rmsnorm_quant", moe_rmsnorm_quant, 8),
    ENTRY("moe_router_logits", moe_router_logits<false>, 5),
    ENTRY("moe_router_logits_split", moe_router_logits<true>, 5),
    ENTRY("moe_route_grouped", moe_route_grouped, 9),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "launch_checks", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_launch_checks() { return PyModule_Create(&module); }
