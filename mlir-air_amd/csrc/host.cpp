// The host side of the operators that programs call most and of whole prompt passes, in native code: arguments checked, outputs and scratch allocated
// by torch, the C entry points of the two kernel libraries called.  A launch takes the host 2.5 to 3.5 us; in Python the rest took 4 us for a product
// and 6 us for an operator of a prompt pass, longer than the kernels of small sizes run.  us a call, one after the other, in Python / here: int4 Linear
// of one row of 1024 x 1024 6.6 / 4.5; a prompt of 4 tokens, one layer of latent attention and experts of width 1024 146 / 77; of 68 tokens, four
// layers of windowed attention and recurrences of width 1984 455 / 368 (now the GPU's time).  Nothing is kept between calls but the entry points'
// addresses.
//
// Functions return None, with nothing launched, where tensors are not of the form that they take: the operators in Python (ops.py, dense.py) say
// then what is wrong with them.  (Without the module they run always.)
#include <torch/extension.h>

#include <string>
#include <vector>

#include "../../include/dense_lm.h"
#include "../../include/w4a16.h"

namespace py = pybind11;
using at::Tensor;

namespace {

// ---- entry points of the kernel libraries, by name ----------------------------------------------------------------------------
#define DENSE_ENTRIES(X)                                                                                                                   \
    X(dlm_gemm) X(dlm_gemm_slices) X(dlm_gemm_parts) X(dlm_gemm_sliced) X(dlm_gemm_tile_rows) X(dlm_moe_select_parts) X(dlm_moe_max_tiles) \
    X(dlm_moe_plan) X(dlm_residual_norm_parts) X(dlm_residual_norm_rows) X(dlm_add_norm_parts) X(dlm_add_norm_rows) X(dlm_embed_rows)      \
    X(dlm_gemv) X(dlm_gemv_keys) X(dlm_argmax) X(dlm_latent_decode_supported) X(dlm_latent_prefill_supported) X(dlm_latent_prepare)        \
    X(dlm_latent_prefill) X(dlm_latent_splits) X(dlm_latent_absorb) X(dlm_latent_decode) X(dlm_latent_combine) X(dlm_head_splits)          \
    X(dlm_head_decode_supported) X(dlm_head_prefill_supported) X(dlm_head_prepare) X(dlm_head_prefill) X(dlm_head_decode)                  \
    X(dlm_head_merge) X(dlm_short_conv) X(dlm_recurrence_steps) X(dlm_recurrence_chunk_bytes) X(dlm_recurrence_chunks) X(dlm_gated_norm)
#define W4A16_ENTRIES(X)                                                                                                   \
    X(w4a16_gemv_stream_bf16) X(w4a16_gemm_stream_bf16) X(w4a16_gemm_stream_best_scratch_bytes) X(w4a16_gemm_stream_scratch_bf16) \
    X(w4a16_q4nx_gemv_stream_bf16) X(w4a16_q4nx_gemm_stream_best_scratch_bytes) X(w4a16_q4nx_gemm_stream_scratch_bf16)
#define MEMBER(f) decltype(&::f) f = nullptr;
struct {
    DENSE_ENTRIES(MEMBER)
} dense;
struct {
    W4A16_ENTRIES(MEMBER)
} w4a16;
#undef MEMBER
#define BIND(f) s.f = reinterpret_cast<decltype(s.f)>(entries[#f].template cast<uintptr_t>());
void bind_dense(py::dict entries) {
    auto &s = dense;
    DENSE_ENTRIES(BIND)
}
void bind_w4a16(py::dict entries) {
    auto &s = w4a16;
    W4A16_ENTRIES(BIND)
}
#undef BIND
#define NAME(f) names.append(#f);
py::list dense_entries() {
    py::list names;
    DENSE_ENTRIES(NAME)
    return names;
}
py::list w4a16_entries() {
    py::list names;
    W4A16_ENTRIES(NAME)
    return names;
}
#undef NAME
// What the module was compiled against: the ABI versions and the size of every struct that crosses, as _lib.py has them, which compares.
py::dict compiled_for() {
    py::dict d;
    d["w4a16"] = W4A16_ABI_VERSION, d["dense_lm"] = DLM_ABI_VERSION;
    d["Intake"] = sizeof(dlm_intake), d["Router"] = sizeof(dlm_router), d["GemmArgs"] = sizeof(dlm_gemm_args), d["LatentShape"] = sizeof(dlm_latent_shape);
    d["LatentRows"] = sizeof(dlm_latent_rows), d["HeadShape"] = sizeof(dlm_head_shape), d["HeadRows"] = sizeof(dlm_head_rows);
    d["ShortConvArgs"] = sizeof(dlm_short_conv_args), d["RecurrenceArgs"] = sizeof(dlm_recurrence_args);
    return d;
}

// What an entry point refused, on its way to the errors of _lib.py: `check` raises the code's.
struct Refused {
    const char *check;
    int code;
};
void must(int code, const char *check = "check_dense") {
    if (code) throw Refused{check, code};
}
// f, which allocates and launches, without Python's lock, as ctypes calls the entry points: other threads go on, also where the launch queue is full.
// (It takes and gives back no Python objects.  One row of 1024 x 1024, a call: 3.77 us with the lock held, 3.78 so.)
template <class F>
auto unlocked(F f) {
    try {
        py::gil_scoped_release others;
        return f();
    } catch (const Refused &r) {
        py::module_::import("air_hip._lib").attr(r.check)(r.code);
        throw;
    }
}

bool on_gpu(const Tensor &t) { return t.defined() && t.is_cuda() && t.is_contiguous(); }
bool shaped(const Tensor &t, at::IntArrayRef sizes) { return on_gpu(t) && t.sizes() == sizes; }

// ---- int4 Linear ---------------------------------------------------------------------------------------------------------------
// y = bf16(x . W) of a stream-order matrix; `vector`: the form of one row, whose result is [N]
std::optional<Tensor> linear(const Tensor &x, const Tensor &w, int64_t K, int64_t N, bool q4, bool vector, uintptr_t stream) {
    if (!on_gpu(x) || !on_gpu(w) || x.scalar_type() != at::kBFloat16) return std::nullopt;
    const int64_t dims = x.dim();
    if (vector ? x.numel() != K : (dims != 1 && dims != 2) || x.size(-1) != K) return std::nullopt;
    const int64_t M = vector || dims == 1 ? 1 : x.size(0);
    if (M < 1 || M > INT32_MAX || K > INT32_MAX || N > INT32_MAX) return std::nullopt;
    return unlocked([&]() -> std::optional<Tensor> {
        Tensor y = vector || dims == 1 ? at::empty({N}, x.options()) : at::empty({M, N}, x.options());
        const auto *xp = static_cast<const uint16_t *>(x.data_ptr());
        auto *yp = static_cast<uint16_t *>(y.data_ptr());
        void *st = reinterpret_cast<void *>(stream);
        const int m = (int)M, k = (int)K, n = (int)N;
        int rc;
        if (M == 1) {
            rc = q4 ? w4a16.w4a16_q4nx_gemv_stream_bf16(xp, w.data_ptr(), nullptr, yp, k, n, st) : w4a16.w4a16_gemv_stream_bf16(xp, w.data_ptr(), yp, k, n, 128, st);
        } else {
            // plain scratch of the call: of the caller's stream and, in a capture, of its graph
            const size_t bytes = M <= 16 ? 0 : q4 ? w4a16.w4a16_q4nx_gemm_stream_best_scratch_bytes(m, k, n, 0) : w4a16.w4a16_gemm_stream_best_scratch_bytes(m, k, n);
            Tensor scratch;
            if (bytes) scratch = at::empty({(int64_t)bytes}, x.options().dtype(at::kByte));
            void *sp = bytes ? scratch.data_ptr() : nullptr;
            if (q4) rc = w4a16.w4a16_q4nx_gemm_stream_scratch_bf16(xp, w.data_ptr(), nullptr, yp, m, k, n, sp, bytes, st);
            else if (bytes) rc = w4a16.w4a16_gemm_stream_scratch_bf16(xp, w.data_ptr(), yp, m, k, n, 128, sp, bytes, st);
            else rc = w4a16.w4a16_gemm_stream_bf16(xp, w.data_ptr(), yp, m, k, n, 128, st);
        }
        must(rc, "check");
        return y;
    });
}

// ---- dense-weight models: many tokens through every layer ----------------------------------------------------------------------
template <class T>
T get(const py::handle &o, const char *name) {
    return o.attr(name).cast<T>();
}
Tensor maybe(const py::handle &o, const char *name) {   // undefined for None
    const py::object v = o.attr(name);
    return v.is_none() ? Tensor() : v.cast<Tensor>();
}

// What the operators of one pass share; M rows
struct Pass {
    int64_t M;
    int dt;
    at::TensorOptions elem, f32, i32;
    void *stream;

    Pass(int64_t rows, const Tensor &like, uintptr_t st) : M(rows), dt(like.scalar_type() == at::kFloat), elem(like.options()) {
        f32 = elem.dtype(at::kFloat), i32 = elem.dtype(at::kInt), stream = reinterpret_cast<void *>(st);
    }
    Tensor elems(int64_t a, int64_t b) const { return at::empty({a, b}, elem); }
    Tensor floats(at::IntArrayRef s) const { return at::empty(s, f32); }
    bool matrix(const Tensor &w, int64_t K) const { return on_gpu(w) && w.dim() == 2 && w.size(1) == K && w.scalar_type() == elem.dtype(); }
    bool vec(const Tensor &v, int64_t n) const { return on_gpu(v) && v.numel() == n && v.scalar_type() == at::kFloat; }

    dlm_gemm_args args(const void *a, int64_t lda, int64_t rows, const Tensor &w, int epilogue) const {
        dlm_gemm_args g{};
        g.a = a, g.w = w.data_ptr(), g.lda = lda, g.M = (int)rows, g.N = (int)w.size(0), g.K = (int)w.size(1), g.epilogue = epilogue;
        g.ldo = epilogue >= 2 ? g.N / 2 : g.N;
        return g;
    }
    // rows of `a` (row stride lda) times W^T; epilogue as in dlm_gemm, silu on columns of the first
    Tensor gemm(const void *a, int64_t lda, const Tensor &w, int epilogue, int64_t rows = -1, int silu_begin = 0, int silu_end = 0) const {
        dlm_gemm_args g = args(a, lda, rows < 0 ? M : rows, w, epilogue);
        g.silu_begin = silu_begin, g.silu_end = silu_end;
        const int slices = dense.dlm_gemm_slices(dt, g.M, g.N, g.K, epilogue);
        const Tensor out = epilogue == 1 ? floats({g.M, g.ldo}) : elems(g.M, g.ldo);
        Tensor pieces;
        if (slices > 1) pieces = floats({slices, g.M, g.N});
        g.out = out.data_ptr();
        must(dense.dlm_gemm_sliced(dt, &g, slices, slices > 1 ? pieces.data_ptr<float>() : nullptr, stream));
        return out;
    }
    // the same in fp32, in parts [n, M, N] that whoever reads them adds up
    Tensor parts(const Tensor &a, const Tensor &w) const {
        dlm_gemm_args g = args(a.data_ptr(), a.stride(0), M, w, 1);
        const int n = dense.dlm_gemm_parts(dt, g.M, g.N, g.K);
        const Tensor out = floats({n, g.M, g.N});
        if (n == 1) g.out = out.data_ptr();
        must(dense.dlm_gemm_sliced(dt, &g, n, n > 1 ? out.data_ptr<float>() : nullptr, stream));
        return out;
    }
};

struct Experts {
    Tensor correction, w_router, w_gate_up, w_down;
    int top = 0, groups, keep;
    int64_t experts, ff2, N;

    bool read(const py::handle &l, const Pass &p, int64_t W) {
        const py::object r = l.attr("router");
        if (r.is_none()) return true;
        correction = get<Tensor>(r, "correction"), experts = get<int64_t>(r, "experts"), top = get<int>(r, "top"), groups = get<int>(r, "groups"), keep = get<int>(r, "keep");
        w_router = get<Tensor>(l, "w_router"), w_gate_up = get<Tensor>(l, "w_gate_up"), w_down = get<Tensor>(l, "w_down");
        if (!on_gpu(w_gate_up) || w_gate_up.dim() != 3 || top < 1) return false;
        ff2 = w_gate_up.size(1), N = W;
        return p.vec(correction, experts) && p.matrix(w_router, W) && w_router.size(0) >= experts && w_gate_up.size(0) == experts && w_gate_up.size(2) == W &&
               shaped(w_down, {experts, W, ff2 / 2}) && w_gate_up.scalar_type() == p.elem.dtype() && w_down.scalar_type() == p.elem.dtype();
    }
    // the chosen experts' outputs [M * top, N], row token * top + slot, and their weights [M, top]
    std::pair<Tensor, Tensor> run(const Pass &p, const Tensor &h, const Tensor &logits) const {
        const int64_t M = p.M, entries = M * top, ff = ff2 / 2;
        const Tensor ids = at::empty({M, top}, p.i32), weights = p.floats({M, top});
        dlm_router r{logits.data_ptr<float>(), correction.data_ptr<float>(), (int)w_router.size(0), (int)experts, top, groups, keep};
        must(dense.dlm_moe_select_parts(&r, (int)logits.size(0), (int)M, ids.data_ptr<int>(), weights.data_ptr<float>(), p.stream));
        const int tile_rows = dense.dlm_gemm_tile_rows(p.dt, (int)(entries / experts), (int)std::max(ff2, N), (int)experts);
        const int n_tiles = dense.dlm_moe_max_tiles((int)entries, (int)experts, tile_rows);
        const Tensor order = at::empty({entries}, p.i32), tiles = at::empty({n_tiles + 1, 4}, p.i32);
        must(dense.dlm_moe_plan(ids.data_ptr<int>(), (int)entries, (int)experts, tile_rows, order.data_ptr<int>(), tiles.data_ptr<int>(), p.stream));
        const Tensor act = p.elems(entries, ff), out = p.elems(entries, N);
        dlm_gemm_args g{};
        g.tiles = tiles.data_ptr<int>(), g.order = order.data_ptr<int>(), g.M = (int)entries, g.n_tiles = n_tiles, g.tile_rows = tile_rows;
        g.a = h.data_ptr(), g.w = w_gate_up.data_ptr(), g.out = act.data_ptr(), g.lda = N, g.ldo = ff, g.w_stride = ff2 * N, g.N = (int)ff2, g.K = (int)N;
        g.epilogue = 2, g.gather = top;
        must(dense.dlm_gemm(p.dt, &g, p.stream));
        g.a = act.data_ptr(), g.w = w_down.data_ptr(), g.out = out.data_ptr(), g.lda = ff, g.ldo = N, g.w_stride = N * ff, g.N = (int)N, g.K = (int)ff;
        g.epilogue = 0, g.gather = 0;
        must(dense.dlm_gemm(p.dt, &g, p.stream));
        return {out, weights};
    }
};

// One layer of latent attention and experts (kuvonex.KuvonexLayer)
struct LatentLayer {
    dlm_latent_shape shape{};
    Tensor w_in, kv_norm, w_ukv, sink, w_o, norm1, norm2, cache, table;
    int kv_off, gate_off;
    int64_t out_width;
    bool absorbed;
    Experts experts;

    bool read(const py::handle &l, const Tensor &cache_, const Tensor &table_, const Pass &p, int64_t W, int64_t pos, int64_t absorb_most) {
        const py::object s = l.attr("spec");
        shape.heads = get<int>(s, "heads"), shape.dim = get<int>(s, "dim_p"), shape.rot = get<int>(s, "rot_p"), shape.vdim = get<int>(s, "vdim_p");
        shape.rank = get<int>(s, "rank_p"), shape.rot_pairs = get<int>(s, "rot") / 2, shape.true_rank = get<int>(s, "rank"), shape.scale = get<float>(s, "scale");
        w_in = get<Tensor>(l, "w_in"), kv_norm = maybe(l, "kv_norm"), w_ukv = get<Tensor>(l, "w_ukv"), sink = get<Tensor>(l, "sink"), w_o = get<Tensor>(l, "w_o");
        norm1 = get<Tensor>(l, "norm1"), norm2 = maybe(l, "norm2"), kv_off = get<int>(l, "kv_off"), gate_off = get<int>(l, "gate_off");
        cache = cache_, table = table_;
        const int64_t H = shape.heads, width = H * shape.vdim;
        out_width = (width + 63) / 64 * 64;
        if (!on_gpu(cache) || cache.dim() != 2 || cache.size(1) != shape.rank + shape.rot || cache.scalar_type() != p.elem.dtype() || pos + p.M > cache.size(0)) return false;
        if (!on_gpu(table) || table.dim() != 3 || table.size(0) < pos + p.M || table.size(1) != shape.rot_pairs || table.size(2) != 2 || table.scalar_type() != at::kFloat) return false;
        if (!p.matrix(w_in, W) || !p.matrix(w_o, out_width) || w_o.size(0) != W || !p.matrix(w_ukv, shape.rank) || w_ukv.size(0) != H * (shape.dim + shape.vdim)) return false;
        if (!p.vec(sink, H) || !p.vec(norm1, W) || (kv_norm.defined() && !p.vec(kv_norm, shape.rank)) || (kv_off >= 0 && !kv_norm.defined())) return false;
        // columns of the projections: queries, latent and key part, gate
        const int64_t cols = w_in.size(0);
        if (gate_off < H * (shape.dim + shape.rot) || gate_off + width > cols || (kv_off >= 0 && kv_off + shape.rank + shape.rot > cols)) return false;
        const bool decode = dense.dlm_latent_decode_supported(p.dt, &shape), prefill = dense.dlm_latent_prefill_supported(p.dt, &shape);
        if (!decode && !prefill) return false;
        absorbed = decode && (p.M <= absorb_most || !prefill);
        return experts.read(l, p, W) && (!experts.top || p.vec(norm2, W));
    }
    Tensor attend(const Pass &p, const Tensor &proj, int64_t pos) const {
        const int64_t M = p.M, H = shape.heads;
        dlm_latent_rows r{};
        r.proj = proj.data_ptr(), r.lut = table.data_ptr<float>(), r.kv_norm = kv_norm.defined() ? kv_norm.data_ptr<float>() : nullptr, r.cache = cache.data_ptr();
        r.ld = proj.size(1), r.kv_off = kv_off, r.gate_off = gate_off, r.M = (int)M, r.pos = (int)pos, r.eps = eps;
        const bool exact = out_width == H * shape.vdim;
        auto result = [&]() { return exact ? p.elems(M, out_width) : at::zeros({M, out_width}, p.elem); };
        if (!absorbed) {
            must(dense.dlm_latent_prepare(p.dt, &shape, &r, p.stream));
            const Tensor kv = p.gemm(cache.data_ptr(), cache.size(1), w_ukv, 0, pos + M), out = result();
            must(dense.dlm_latent_prefill(p.dt, &shape, &r, kv.data_ptr(), kv.size(1), sink.data_ptr<float>(), out.data_ptr(), out_width, p.stream));
            return out;
        }
        const int64_t rows = M * H;
        const int nsplit = dense.dlm_latent_splits(shape.heads, (int)M, pos + M);
        const Tensor qa = p.elems(rows, shape.rank + shape.rot), part_o = p.floats({rows, nsplit, shape.rank}), part_ml = p.floats({rows, nsplit, 2}), out = result();
        const char *uk = static_cast<const char *>(w_ukv.data_ptr());
        must(dense.dlm_latent_absorb(p.dt, &shape, &r, uk, qa.data_ptr(), p.stream));
        must(dense.dlm_latent_decode(p.dt, &shape, &r, qa.data_ptr(), nsplit, part_o.data_ptr<float>(), part_ml.data_ptr<float>(), p.stream));
        must(dense.dlm_latent_combine(p.dt, &shape, &r, nsplit, part_o.data_ptr<float>(), part_ml.data_ptr<float>(), sink.data_ptr<float>(),
                                      uk + H * shape.dim * shape.rank * w_ukv.element_size(), out.data_ptr(), out_width, p.stream));
        return out;
    }
    float eps = 0;
};

// KuvonexModel._rows: the residual [M, W] behind the last layer
std::optional<Tensor> latent_rows(py::list layers, std::vector<Tensor> caches, std::vector<Tensor> tables, const Tensor &tokens, const Tensor &embed, float embed_scale,
                                  float eps, int width, int64_t pos, int64_t absorb_most, uintptr_t stream) {
    if (!on_gpu(embed) || embed.dim() != 2 || !on_gpu(tokens) || tokens.scalar_type() != at::kInt || tokens.numel() < 1 || pos < 0) return std::nullopt;
    if (embed.scalar_type() != at::kBFloat16 && embed.scalar_type() != at::kFloat) return std::nullopt;
    const Pass p(tokens.numel(), embed, stream);
    const int64_t M = p.M, W = embed.size(1);
    std::vector<LatentLayer> ls(layers.size());
    for (size_t i = 0; i < ls.size(); ++i) {
        ls[i].eps = eps;
        if (!ls[i].read(layers[i], caches[i], tables[i], p, W, pos, absorb_most)) return std::nullopt;
    }
    return unlocked([&]() -> std::optional<Tensor> {
        const Tensor res = p.floats({M, W});
        float *rp = res.data_ptr<float>();
        Tensor h = p.elems(M, W);
        must(dense.dlm_embed_rows(p.dt, tokens.data_ptr<int>(), embed.data_ptr(), embed_scale, rp, h.data_ptr(), (int)M, (int)W, p.stream));
        for (const LatentLayer &l : ls) {
            const Tensor attn = l.attend(p, p.gemm(h.data_ptr(), W, l.w_in, 0), pos), y = p.parts(attn, l.w_o);
            h = p.elems(M, W);
            must(dense.dlm_residual_norm_parts(p.dt, rp, y.data_ptr<float>(), (int)y.size(0), l.norm1.data_ptr<float>(), eps, width, h.data_ptr(), (int)M, (int)W, p.stream));
            if (!l.experts.top) continue;
            const auto [out, weights] = l.experts.run(p, h, p.parts(h, l.experts.w_router));
            h = p.elems(M, W);
            must(dense.dlm_residual_norm_rows(p.dt, rp, out.data_ptr(), weights.data_ptr<float>(), l.experts.top, l.norm2.data_ptr<float>(), eps, width, h.data_ptr(), (int)M,
                                              (int)W, p.stream));
        }
        return res;
    });
}

// One layer of windowed attention beside a recurrence, or of the delta rule (sitirax.SitiraxLayer)
struct MixedLayer {
    bool parallel, few = false;
    dlm_head_shape heads{};
    int64_t H, KH, dim, vdim;                 // of the state, padded
    Tensor w_in, w_o, norm1, norm2, w_gate_up, w_down, norm, state;
    int64_t out_columns;
    Tensor q_norm, k_norm, log2_decay, rows;  // parallel
    int true_cols = 0, gate_off = 0, silu[2] = {0, 0}, offsets[3] = {0, 0, 0};
    Tensor conv, w_a2, w_g2, a_log, dt_bias, history;   // delta rule
    float q_scale = 0;
    int a_off = 0, g_off = 0, b_off = 0;
    int true_vdim = 0;

    int64_t qk_width() const { return KH * dim; }
    int64_t v_width() const { return H * vdim; }
    int64_t channels() const { return 2 * qk_width() + v_width(); }

    bool read(const py::handle &l, const py::dict &c, const Pass &p, int64_t W, int64_t pos, int64_t split_most) {
        const py::object m = l.attr("mixer"), s = m.attr("state");
        parallel = py::hasattr(m, "attn");
        H = get<int64_t>(s, "heads"), KH = get<int64_t>(s, "k_heads"), dim = get<int64_t>(s, "dim_p"), vdim = get<int64_t>(s, "vdim_p"), true_vdim = get<int>(s, "vdim");
        w_in = get<Tensor>(m, "w_in"), w_o = get<Tensor>(m, "w_o"), norm = get<Tensor>(m, "norm"), out_columns = get<int64_t>(m, "out_columns");
        norm1 = get<Tensor>(l, "norm1"), norm2 = maybe(l, "norm2"), w_gate_up = maybe(l, "w_gate_up"), w_down = maybe(l, "w_down");
        state = c["state"].cast<Tensor>();
        if (!p.matrix(w_in, W) || !on_gpu(w_o) || w_o.dim() != 2 || w_o.size(0) != W || w_o.scalar_type() != p.elem.dtype() || w_o.size(1) < out_columns || !p.vec(norm1, W)) return false;
        if (!shaped(state, {H, vdim, dim}) || state.scalar_type() != at::kFloat) return false;
        if (norm2.defined() && (!p.vec(norm2, W) || !p.matrix(w_gate_up, W) || !p.matrix(w_down, w_gate_up.size(0) / 2) || w_down.size(0) != W)) return false;
        const int64_t cols = w_in.size(0);
        if (parallel) {
            const py::object a = m.attr("attn");
            heads.heads = get<int>(a, "heads"), heads.kv_heads = get<int>(a, "kv_heads"), heads.dim = get<int>(a, "dim_p"), heads.vdim = get<int>(a, "vdim_p");
            heads.true_dim = get<int>(a, "dim"), heads.window = (int)std::min<int64_t>(get<int64_t>(a, "window"), 1 << 30), heads.scale = get<float>(a, "scale");
            heads.out_scale = get<float>(a, "out_scale");
            q_norm = get<Tensor>(m, "q_norm"), k_norm = get<Tensor>(m, "k_norm"), log2_decay = get<Tensor>(m, "log2_decay"), rows = c["rows"].cast<Tensor>();
            true_cols = get<int>(m, "true_cols"), gate_off = get<int>(m, "gate_off");
            const auto sl = get<std::pair<int, int>>(m, "silu");
            const auto of = get<std::tuple<int, int, int>>(m, "offsets");
            silu[0] = sl.first, silu[1] = sl.second, offsets[0] = std::get<0>(of), offsets[1] = std::get<1>(of), offsets[2] = std::get<2>(of);
            if (!on_gpu(rows) || rows.dim() != 3 || rows.size(0) != heads.kv_heads || rows.size(2) != heads.dim + heads.vdim || rows.scalar_type() != p.elem.dtype()) return false;
            heads.ring = (int)rows.size(1);
            const int64_t attn_cols = (int64_t)(heads.heads + heads.kv_heads) * heads.dim + (int64_t)heads.kv_heads * heads.vdim;
            if (!p.vec(q_norm, heads.dim) || !p.vec(k_norm, heads.dim) || !p.vec(log2_decay, H) || !p.vec(norm, v_width()) || KH != H) return false;
            if (offsets[0] < attn_cols || offsets[0] + qk_width() > cols || offsets[1] + qk_width() > cols || offsets[2] + v_width() > cols || gate_off + v_width() > cols) return false;
            if (out_columns != (int64_t)heads.heads * heads.vdim + v_width()) return false;
            const bool decode = dense.dlm_head_decode_supported(p.dt, &heads), prefill = dense.dlm_head_prefill_supported(p.dt, &heads);
            if (!decode && !prefill) return false;
            few = decode && (p.M <= split_most || !prefill);
            return true;
        }
        conv = get<Tensor>(m, "conv"), w_a2 = get<Tensor>(m, "w_a2"), w_g2 = get<Tensor>(m, "w_g2"), a_log = get<Tensor>(m, "a_log"), dt_bias = get<Tensor>(m, "dt_bias");
        q_scale = get<float>(m, "q_scale"), a_off = get<int>(m, "a_off"), g_off = get<int>(m, "g_off"), b_off = get<int>(m, "b_off"), history = c["history"].cast<Tensor>();
        if (!on_gpu(conv) || conv.dim() != 2 || conv.size(1) != channels() || conv.scalar_type() != at::kFloat || !on_gpu(history) || history.sizes() != conv.sizes() ||
            history.scalar_type() != p.elem.dtype())
            return false;
        if (a_off < channels() || g_off < a_off || b_off < g_off || b_off + H > cols || !p.matrix(w_a2, g_off - a_off) || w_a2.size(0) != H * dim ||
            !p.matrix(w_g2, b_off - g_off) || w_g2.size(0) != v_width())
            return false;
        return p.vec(a_log, H) && p.vec(dt_bias, H * dim) && p.vec(norm, vdim) && out_columns == v_width();
    }
    // The read-outs fp32 [M, heads * vdim] of a recurrence
    Tensor recur(const Pass &p, dlm_recurrence_args &a, const Tensor &qkv, const int (&off)[3], int64_t pos, int64_t steps_most) const {
        a.qkv = qkv.data_ptr(), a.state = state.data_ptr<float>(), a.ld = qkv.size(1), a.k_heads = (int)KH, a.heads = (int)H, a.dim = (int)dim, a.vdim = (int)vdim;
        a.q_off = off[0], a.k_off = off[1], a.v_off = off[2], a.M = (int)p.M, a.pos = (int)pos;
        const Tensor o = p.floats({p.M, v_width()});
        const size_t bytes = dense.dlm_recurrence_chunk_bytes(&a);
        if (p.M > steps_most && bytes > 0) {
            const Tensor work = at::empty({(int64_t)bytes}, p.elem.dtype(at::kByte));
            must(dense.dlm_recurrence_chunks(p.dt, &a, work.data_ptr(), o.data_ptr<float>(), p.stream));
        } else {
            must(dense.dlm_recurrence_steps(p.dt, &a, o.data_ptr<float>(), p.stream));
        }
        return o;
    }
    Tensor mix(const Pass &p, const Tensor &proj, int64_t pos, float eps, float unit_eps, int64_t steps_most) const {
        const int64_t M = p.M, ldo = w_o.size(1), size = proj.element_size(), ld = proj.size(1);
        const Tensor out = ldo == out_columns ? p.elems(M, ldo) : at::zeros({M, ldo}, p.elem);
        const char *base = static_cast<const char *>(proj.data_ptr());
        if (parallel) {
            dlm_head_rows r{};
            r.proj = proj.data_ptr(), r.q_norm = q_norm.data_ptr<float>(), r.k_norm = k_norm.data_ptr<float>(), r.cache = rows.data_ptr(), r.ld = ld, r.M = (int)M;
            r.pos = (int)pos, r.eps = eps;
            const Tensor q = p.elems(M * heads.heads, heads.dim);
            must(dense.dlm_head_prepare(p.dt, &heads, &r, q.data_ptr(), p.stream));
            if (!few) {
                must(dense.dlm_head_prefill(p.dt, &heads, &r, q.data_ptr(), out.data_ptr(), ldo, p.stream));
            } else {
                const int n = dense.dlm_head_splits(heads.heads, heads.kv_heads, heads.window, (int)M, pos + M);
                const Tensor part_o = p.floats({M * heads.heads, n, heads.vdim}), part_ml = p.floats({M * heads.heads, n, 2});
                must(dense.dlm_head_decode(p.dt, &heads, &r, q.data_ptr(), n, part_o.data_ptr<float>(), part_ml.data_ptr<float>(), p.stream));
                must(dense.dlm_head_merge(p.dt, &heads, &r, n, part_o.data_ptr<float>(), part_ml.data_ptr<float>(), out.data_ptr(), ldo, p.stream));
            }
            dlm_recurrence_args a{};
            a.log2_decay = log2_decay.data_ptr<float>();
            const Tensor o = recur(p, a, proj, offsets, pos, steps_most);
            must(dense.dlm_gated_norm(p.dt, o.data_ptr<float>(), norm.data_ptr<float>(), base + gate_off * size, ld,
                                      static_cast<char *>(out.data_ptr()) + (int64_t)heads.heads * heads.vdim * size, ldo, (int)M, 1, (int)v_width(), true_cols, eps, p.stream));
            return out;
        }
        const Tensor act = p.elems(M, channels()), factors = p.floats({M, 2 * KH});
        dlm_short_conv_args c{};
        c.proj = base, c.w = conv.data_ptr<float>(), c.history = history.data_ptr(), c.factors = factors.data_ptr<float>(), c.ld = ld, c.k_heads = (int)KH, c.heads = (int)H;
        c.dim = (int)dim, c.vdim = (int)vdim, c.taps = (int)conv.size(0), c.M = (int)M, c.pos = (int)pos, c.q_scale = q_scale, c.unit_eps = unit_eps;
        must(dense.dlm_short_conv(p.dt, &c, act.data_ptr(), p.stream));
        const Tensor z = p.gemm(base + a_off * size, ld, w_a2, 1), gate = p.gemm(base + g_off * size, ld, w_g2, 0);
        dlm_recurrence_args a{};
        a.z = z.data_ptr<float>(), a.a_log = a_log.data_ptr<float>(), a.dt_bias = dt_bias.data_ptr<float>(), a.factors = factors.data_ptr<float>();
        a.beta = base + b_off * size, a.ld_beta = ld;
        const int at[3] = {0, (int)qk_width(), (int)(2 * qk_width())};
        const Tensor o = recur(p, a, act, at, pos, steps_most);
        must(dense.dlm_gated_norm(p.dt, o.data_ptr<float>(), norm.data_ptr<float>(), gate.data_ptr(), gate.size(1), out.data_ptr(), ldo, (int)M, (int)H, (int)vdim, true_vdim, eps,
                                  p.stream));
        return out;
    }
};

// SitiraxModel._rows: the residual [M, W] behind the last layer
std::optional<Tensor> mixed_rows(py::list layers, py::list caches, const Tensor &tokens, const Tensor &embed, float eps, int width, int64_t pos, int64_t split_most,
                                 int64_t steps_most, float unit_eps, uintptr_t stream) {
    if (!on_gpu(embed) || embed.dim() != 2 || !on_gpu(tokens) || tokens.scalar_type() != at::kInt || tokens.numel() < 1 || pos < 0) return std::nullopt;
    if (embed.scalar_type() != at::kBFloat16 && embed.scalar_type() != at::kFloat) return std::nullopt;
    if (tokens.numel() == 1) return std::nullopt;   // (mixers of one token share launches, which are the operators')
    const Pass p(tokens.numel(), embed, stream);
    const int64_t M = p.M, W = embed.size(1);
    std::vector<MixedLayer> ls(layers.size());
    for (size_t i = 0; i < ls.size(); ++i)
        if (!ls[i].read(layers[i], caches[i].cast<py::dict>(), p, W, pos, split_most)) return std::nullopt;
    return unlocked([&]() -> std::optional<Tensor> {
        const Tensor res = p.floats({M, W});
        Tensor y;
        bool first = true;
        // the residual brought up to date (from the embedding first), and its norm
        auto add_norm = [&](const Tensor *norm) {
            Tensor h;
            if (norm) h = p.elems(M, W);
            void *hp = norm ? h.data_ptr() : nullptr;
            const float *np = norm ? norm->data_ptr<float>() : nullptr;
            if (y.defined())
                must(dense.dlm_add_norm_parts(p.dt, res.data_ptr<float>(), y.data_ptr<float>(), (int)y.size(0), np, eps, width, hp, (int)M, (int)W, p.stream));
            else
                must(dense.dlm_add_norm_rows(p.dt, res.data_ptr<float>(), nullptr, first ? tokens.data_ptr<int>() : nullptr, first ? embed.data_ptr() : nullptr, 1.0f, np, eps, width, hp,
                                             (int)M, (int)W, p.stream));
            first = false;
            return h;
        };
        for (const MixedLayer &l : ls) {
            const Tensor h = add_norm(&l.norm1);
            const Tensor out = l.mix(p, p.gemm(h.data_ptr(), W, l.w_in, 0, -1, l.silu[0], l.silu[1]), pos, eps, unit_eps, steps_most);
            y = p.parts(out, l.w_o);
            if (l.norm2.defined()) {
                const Tensor h2 = add_norm(&l.norm2), a = p.gemm(h2.data_ptr(), W, l.w_gate_up, 3);
                y = p.parts(a, l.w_down);
            }
        }
        add_norm(nullptr);
        return res;
    });
}

// Logits fp32 [rows of the head] of one row of a finished residual and its greedy choice [1]; mode: the intake of dlm_gemv, 3 or 4
std::optional<std::pair<Tensor, Tensor>> tail(int mode, const Tensor &res, const Tensor &final_w, const Tensor &head, float eps, int width, int n_valid, uintptr_t stream) {
    if (!on_gpu(res) || !on_gpu(final_w) || !on_gpu(head) || head.dim() != 2 || res.numel() != head.size(1) || final_w.numel() != head.size(1)) return std::nullopt;
    if (res.scalar_type() != at::kFloat || final_w.scalar_type() != at::kFloat || (head.scalar_type() != at::kBFloat16 && head.scalar_type() != at::kFloat)) return std::nullopt;
    return unlocked([&]() -> std::optional<std::pair<Tensor, Tensor>> {
        const Pass p(1, head, stream);
        const int K = (int)head.size(1), N = (int)head.size(0), n_keys = dense.dlm_gemv_keys(K, N);
        const Tensor logits = p.floats({N}), keys = at::empty({n_keys}, p.elem.dtype(at::kLong)), best = at::empty({1}, p.i32);
        dlm_intake in{};
        in.mode = mode, in.width = width, in.eps = eps, in.scale = 1.0f, in.res = res.data_ptr<float>(), in.final_w = final_w.data_ptr<float>();
        auto *kp = reinterpret_cast<uint64_t *>(keys.data_ptr<int64_t>());
        must(dense.dlm_gemv(p.dt, head.data_ptr(), &in, nullptr, logits.data_ptr<float>(), kp, n_valid, K, N, p.stream));
        must(dense.dlm_argmax(kp, n_keys, best.data_ptr<int>(), nullptr, nullptr, p.stream));
        return std::make_pair(logits, best);
    });
}

}  // namespace

PYBIND11_MODULE(air_host, m) {
    m.def("bind_dense", &bind_dense);
    m.def("bind_w4a16", &bind_w4a16);
    m.def("dense_entries", &dense_entries);
    m.def("w4a16_entries", &w4a16_entries);
    m.def("compiled_for", &compiled_for);
    m.def("linear", &linear);
    m.def("latent_rows", &latent_rows);
    m.def("mixed_rows", &mixed_rows);
    m.def("tail", &tail);
}
