// The plain case of the Python wrappers in native.py, in C++: checks, output allocation and the call of the C entry.
//
// Every function takes what its wrapper takes and answers None where the call is not the plain one (a tensor that is not
// dense, aligned or of the expected type, an output of the caller's that does not fit): the wrapper then goes the long way,
// which copies or refuses.  An int is the status of a C entry that refused.  A step of a few hundred tokens waits for
// the host, and of its time a third went into the wrappers: per call 5 to 9 us of Python around 3.7 us of launch, here 1 to 2.
#include <torch/extension.h>
#include <torch/version.h>

#include <cstdint>

#include "../../include/odl_fp8.h"

namespace py = pybind11;
using at::Tensor;
using OptTensor = std::optional<Tensor>;
using i64 = int64_t;

namespace {

constexpr i64 kParts = ODL_FP8_AMAX_PARTS;

// entries of the C library: their types from the header, their addresses from native.py, which has loaded it
decltype(&odl_fp8_amax_parts) amax_parts_c;
decltype(&odl_fp8_cast_dynamic_padded) cast_dynamic_c;
decltype(&odl_fp8_quantise_small) quantise_small_c;
decltype(&odl_fp8_gemm_swiglu) gemm_swiglu_c;
decltype(&odl_fp8_cast_delayed_padded) cast_delayed_c;
decltype(&odl_fp8_cast_delayed_many) cast_delayed_many_c;
decltype(&odl_fp8_amax_parts_colsum) amax_colsum_c;
decltype(&odl_fp8_amax_parts_slabs) amax_slabs_c;
decltype(&odl_fp8_slabs_colsum) slabs_colsum_c;
decltype(&odl_fp8_cast_dynamic_colsum) cast_colsum_c;
decltype(&odl_fp8_swiglu_amax_parts) swiglu_c;
decltype(&odl_fp8_swiglu_bwd_amax_parts) swiglu_bwd_c;
decltype(&odl_fp8_gelu_amax_parts) gelu_c;
decltype(&odl_fp8_gelu_bwd_amax_parts) gelu_bwd_c;
decltype(&odl_fp8_gelu_bwd_slabs) gelu_bwd_slabs_c;
decltype(&odl_fp8_rmsnorm_amax_parts) rmsnorm_c;
decltype(&odl_fp8_rmsnorm_bwd) rmsnorm_bwd_c;
decltype(&odl_fp8_layernorm_amax_parts) layernorm_c;
decltype(&odl_fp8_layernorm_bwd) layernorm_bwd_c;
decltype(&odl_fp8_amax_rowcol) amax_rowcol_c;
decltype(&odl_fp8_cast_rowcol_padded) cast_rowcol_c;
decltype(&odl_fp8_gemm_nt_hinted) gemm_nt_c;
decltype(&odl_fp8_gemm_group_route) group_route_c;
decltype(&odl_fp8_gemm_nt_group) gemm_nt_group_c;
decltype(&odl_fp8_gemm_chain_route) chain_route_c;
decltype(&odl_fp8_gemm_nt_chain) gemm_nt_chain_c;
decltype(&odl_fp8_gemm_layouts) gemm_layouts_c;
decltype(&odl_fp8_gemm_runs) runs_c;
decltype(&odl_fp8_mx_cast_padded) mx_cast_c;
decltype(&odl_fp8_block_cast) block_cast_c;
decltype(&odl_fp8_mx_gemm_nt_hinted) mx_gemm_nt_c;

template <class F>
void take(F &f, const py::dict &d, const char *name) { f = reinterpret_cast<F>(py::cast<uintptr_t>(d[name])); }

void bind(const py::dict &d) {
    take(amax_parts_c, d, "odl_fp8_amax_parts");
    take(cast_dynamic_c, d, "odl_fp8_cast_dynamic_padded");
    take(quantise_small_c, d, "odl_fp8_quantise_small");
    take(gemm_swiglu_c, d, "odl_fp8_gemm_swiglu");
    take(cast_delayed_c, d, "odl_fp8_cast_delayed_padded");
    take(cast_delayed_many_c, d, "odl_fp8_cast_delayed_many");
    take(amax_colsum_c, d, "odl_fp8_amax_parts_colsum");
    take(amax_slabs_c, d, "odl_fp8_amax_parts_slabs");
    take(slabs_colsum_c, d, "odl_fp8_slabs_colsum");
    take(cast_colsum_c, d, "odl_fp8_cast_dynamic_colsum");
    take(swiglu_c, d, "odl_fp8_swiglu_amax_parts");
    take(swiglu_bwd_c, d, "odl_fp8_swiglu_bwd_amax_parts");
    take(gelu_c, d, "odl_fp8_gelu_amax_parts");
    take(gelu_bwd_c, d, "odl_fp8_gelu_bwd_amax_parts");
    take(gelu_bwd_slabs_c, d, "odl_fp8_gelu_bwd_slabs");
    take(rmsnorm_c, d, "odl_fp8_rmsnorm_amax_parts");
    take(rmsnorm_bwd_c, d, "odl_fp8_rmsnorm_bwd");
    take(layernorm_c, d, "odl_fp8_layernorm_amax_parts");
    take(layernorm_bwd_c, d, "odl_fp8_layernorm_bwd");
    take(amax_rowcol_c, d, "odl_fp8_amax_rowcol");
    take(cast_rowcol_c, d, "odl_fp8_cast_rowcol_padded");
    take(gemm_nt_c, d, "odl_fp8_gemm_nt_hinted");
    take(group_route_c, d, "odl_fp8_gemm_group_route");
    take(gemm_nt_group_c, d, "odl_fp8_gemm_nt_group");
    take(chain_route_c, d, "odl_fp8_gemm_chain_route");
    take(gemm_nt_chain_c, d, "odl_fp8_gemm_nt_chain");
    take(gemm_layouts_c, d, "odl_fp8_gemm_layouts");
    take(runs_c, d, "odl_fp8_gemm_runs");
    take(mx_cast_c, d, "odl_fp8_mx_cast_padded");
    take(block_cast_c, d, "odl_fp8_block_cast");
    take(mx_gemm_nt_c, d, "odl_fp8_mx_gemm_nt_hinted");
}

// as ctypes does: other Python threads run while a launch waits for room in its queue
template <class F, class... A>
int call(F entry, A... args) {
    py::gil_scoped_release unlocked;
    return entry(args...);
}

// an address, as whatever pointer the entry takes
struct Address {
    void *p;
    template <class T>
    operator T *() const { return static_cast<T *>(p); }
};
Address ptr(const Tensor &t) { return {t.data_ptr()}; }
Address ptr(const OptTensor &t) { return {t ? t->data_ptr() : nullptr}; }
Address str(i64 stream) { return {reinterpret_cast<void *>(stream)}; }
bool aligned(const Tensor &t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }
int src_of(const Tensor &t) { return t.scalar_type() == at::kBFloat16 ? 0 : t.scalar_type() == at::kFloat ? 1 : -1; }
bool dense(const Tensor &t) { return t.is_cuda() && t.is_contiguous() && t.layout() == at::kStrided; }
bool source2d(const Tensor &t) { return dense(t) && t.dim() == 2 && src_of(t) >= 0; }
bool codes2d(const Tensor &t) { return dense(t) && t.dim() == 2 && t.scalar_type() == at::kByte; }
bool floats(const Tensor &t, i64 n) { return dense(t) && t.scalar_type() == at::kFloat && t.numel() == n; }
bool bf16(const Tensor &t) { return dense(t) && t.scalar_type() == at::kBFloat16 && aligned(t); }
Tensor bytes(const Tensor &like, at::IntArrayRef size) { return at::empty(size, like.options().dtype(at::kByte)); }
Tensor f32(const Tensor &like, at::IntArrayRef size) { return at::empty(size, like.options().dtype(at::kFloat)); }
py::object none() { return py::none(); }
py::object status(int rc) { return py::int_(rc); }
py::object obj(const OptTensor &t) { return t ? py::cast(*t) : py::none(); }

// an output of transposed codes: the caller's, if it fits, or a new one
bool transposed_out(const Tensor &x, const OptTensor &given, bool want, i64 cols, i64 rows, OptTensor &out) {
    if (given) {
        if (!codes2d(*given) || given->size(0) != cols || given->size(1) != rows || given->device() != x.device()) return false;
        out = given;
    } else if (want) out = bytes(x, {cols, rows});
    return true;
}

py::object amax_parts(const Tensor &x, i64 stream) {
    if (!source2d(x)) return none();
    Tensor parts = f32(x, {kParts});
    const int rc = call(amax_parts_c, ptr(x), src_of(x), x.size(0), x.size(1), ptr(parts), str(stream));
    return rc ? status(rc) : py::cast(parts);
}

py::object cast_dynamic(const Tensor &x, const Tensor &parts, int fmt, int margin, bool want_q, bool want_t, const OptTensor &out_t,
                        const std::optional<i64> &rows_out, i64 stream) {
    if (!source2d(x) || !(want_q || want_t || out_t)) return none();
    const i64 rows = x.size(0), cols = x.size(1), n = rows_out.value_or(rows);
    if (!floats(parts, kParts)) return none();
    OptTensor q, q_t;
    if (!transposed_out(x, out_t, want_t, cols, n, q_t)) return none();
    if (want_q) q = bytes(x, {n, cols});
    Tensor dyn = f32(x, {3, 1});
    const int rc = call(cast_dynamic_c, ptr(x), src_of(x), rows, cols, n, ptr(parts), fmt, margin, ptr(q), ptr(q_t), ptr(dyn), str(stream));
    if (rc) return status(rc);
    return py::make_tuple(obj(q), obj(q_t), dyn.select(0, 0), dyn.select(0, 1), dyn.select(0, 2));
}

// a small tensor in one launch, row-major codes only
py::object quantise_small(const Tensor &x, int fmt, int margin, i64 stream) {
    const i64 n = x.numel();
    if (!source2d(x) || n == 0 || n * x.element_size() > ODL_FP8_SMALL_BYTES || n % 16 || !aligned(x)) return none();
    Tensor q = bytes(x, {x.size(0), x.size(1)}), dyn = f32(x, {3, 1});
    const int rc = call(quantise_small_c, ptr(x), src_of(x), n, fmt, margin, ptr(q), ptr(dyn), str(stream));
    return rc ? status(rc) : py::make_tuple(q, py::none(), dyn.select(0, 0), dyn.select(0, 1), dyn.select(0, 2));
}

py::object gemm_swiglu(const Tensor &x, const Tensor &gate, const Tensor &up, int fx, int fw, const Tensor &sx, const Tensor &sg, const Tensor &su,
                       i64 stream) {
    if (!codes2d(x) || !codes2d(gate) || !codes2d(up) || gate.sizes() != up.sizes() || x.size(1) != gate.size(1) || !floats(sx, 1) || !floats(sg, 1) ||
        !floats(su, 1))
        return none();
    Tensor h = at::empty({x.size(0), gate.size(0)}, x.options().dtype(at::kBFloat16)), parts = f32(x, {kParts});
    const int rc = call(gemm_swiglu_c, ptr(x), ptr(gate), ptr(up), x.size(0), gate.size(0), x.size(1), fx, fw, ptr(sx), ptr(sg), ptr(su), ptr(h),
                        ptr(parts), str(stream));
    return rc ? status(rc) : py::make_tuple(h, parts);
}

py::object cast_delayed(const Tensor &x, const Tensor &scale, int fmt, const OptTensor &parts, bool want_q, bool want_t, const OptTensor &out_t,
                        const std::optional<i64> &rows_out, i64 stream) {
    if (!source2d(x) || !floats(scale, 1) || (parts && !floats(*parts, kParts)) || !(want_q || want_t || out_t)) return none();
    const i64 rows = x.size(0), cols = x.size(1), n = rows_out.value_or(rows);
    OptTensor q, q_t;
    if (!transposed_out(x, out_t, want_t, cols, n, q_t)) return none();
    if (want_q) q = bytes(x, {n, cols});
    Tensor inv = f32(x, {1});
    const int rc = call(cast_delayed_c, ptr(x), src_of(x), rows, cols, n, ptr(scale), fmt, ptr(q), ptr(q_t), ptr(parts), ptr(inv), str(stream));
    return rc ? status(rc) : py::make_tuple(obj(q), obj(q_t), inv);
}

py::object cast_delayed_many(const Tensor &x, const std::vector<Tensor> &scales, int fmt, const std::vector<Tensor> &parts, i64 rows_out, i64 stream) {
    const size_t n = scales.size();
    if (n < 1 || n > 4 || parts.size() != n || !source2d(x) || x.numel() == 0 || x.size(1) % 8 || rows_out % 16 || rows_out < x.size(0) || !aligned(x))
        return none();
    const float *s[4];
    float *p[4], *inv[4];
    uint8_t *q[4], *q_t[4];
    py::list made(n);
    Tensor invs = f32(x, {(i64)n});
    for (size_t i = 0; i < n; ++i) {
        if (!floats(scales[i], 1) || !floats(parts[i], kParts)) return none();
        Tensor a = bytes(x, {rows_out, x.size(1)}), b = bytes(x, {x.size(1), rows_out});
        s[i] = ptr(scales[i]), p[i] = ptr(parts[i]), inv[i] = static_cast<float *>(ptr(invs)) + i, q[i] = ptr(a), q_t[i] = ptr(b);
        made[i] = py::make_tuple(a, b, invs.narrow(0, (i64)i, 1));
    }
    const int rc = call(cast_delayed_many_c, ptr(x), src_of(x), x.size(0), x.size(1), rows_out, (int)n, s, fmt, q, q_t, p, inv, str(stream));
    return rc ? status(rc) : py::object(made);
}

py::object amax_colsum(const Tensor &x, bool finish, i64 stream) {
    if (!source2d(x)) return none();
    if (!finish && x.size(1) % 8 == 0 && aligned(x)) {
        Tensor parts = f32(x, {kParts}), ws = f32(x, {kParts, ODL_FP8_COLSUM_WORKSPACE / kParts});
        const int rc = call(amax_slabs_c, ptr(x), src_of(x), x.size(0), x.size(1), ptr(parts), ptr(ws), str(stream));
        return rc ? status(rc) : py::make_tuple(parts, ws);
    }
    Tensor parts = f32(x, {kParts}), sums = f32(x, {x.size(1)}), ws = f32(x, {ODL_FP8_COLSUM_WORKSPACE});
    const int rc = call(amax_colsum_c, ptr(x), src_of(x), x.size(0), x.size(1), ptr(parts), ptr(sums), ptr(ws), str(stream));
    return rc ? status(rc) : py::make_tuple(parts, sums);
}

// the column sums of x from the slabs that amax_colsum(x, false) or the producer of x left
py::object slabs_colsum(const Tensor &x, const Tensor &slabs, i64 stream) {
    if (!source2d(x) || x.numel() == 0 || !floats(slabs, ODL_FP8_COLSUM_WORKSPACE)) return none();
    Tensor sums = f32(x, {x.size(1)});
    const int rc = call(slabs_colsum_c, ptr(slabs), src_of(x), x.size(0), x.size(1), ptr(sums), str(stream));
    return rc ? status(rc) : py::cast(sums);
}

py::object cast_colsum(const Tensor &x, const Tensor &parts, const Tensor &slabs, int fmt, int margin, i64 rows_out, int odt, i64 stream) {
    if (!source2d(x) || !aligned(x) || !floats(parts, kParts) || !floats(slabs, ODL_FP8_COLSUM_WORKSPACE) || x.size(1) % 8) return none();
    const i64 rows = x.size(0), cols = x.size(1);
    Tensor q = bytes(x, {rows_out, cols}), q_t = bytes(x, {cols, rows_out}), dyn = f32(x, {3});
    Tensor sums = at::empty({cols}, x.options().dtype(odt ? at::kFloat : at::kBFloat16));
    const int rc = call(cast_colsum_c, ptr(x), src_of(x), rows, cols, rows_out, ptr(parts), fmt, margin, ptr(q), ptr(q_t), ptr(dyn), ptr(slabs), ptr(sums),
                        odt, str(stream));
    return rc ? status(rc) : py::make_tuple(q, q_t, dyn.narrow(0, 2, 1), sums);
}

i64 last(const Tensor &t) { return t.dim() ? t.size(-1) : 1; }

py::object swiglu(const Tensor &gate, const Tensor &up, i64 stream) {
    if (!bf16(gate) || !bf16(up) || gate.sizes() != up.sizes()) return none();
    const i64 cols = last(gate), rows = gate.numel() / std::max<i64>(cols, 1);
    Tensor h = at::empty_like(gate), parts = f32(gate, {kParts});
    const int rc = call(swiglu_c, ptr(gate), ptr(up), rows, cols, ptr(h), ptr(parts), str(stream));
    return rc ? status(rc) : py::make_tuple(h, parts);
}

py::object swiglu_bwd(const Tensor &dh, const Tensor &gate, const Tensor &up, i64 stream) {
    if (!bf16(dh) || !bf16(gate) || !bf16(up) || gate.sizes() != up.sizes() || gate.sizes() != dh.sizes()) return none();
    const i64 cols = last(gate), rows = gate.numel() / std::max<i64>(cols, 1);
    Tensor dg = at::empty_like(gate), du = at::empty_like(up), parts = f32(gate, {2 * kParts});
    Tensor pg = parts.narrow(0, 0, kParts), pu = parts.narrow(0, kParts, kParts);
    const int rc = call(swiglu_bwd_c, ptr(dh), ptr(gate), ptr(up), rows, cols, ptr(dg), ptr(du), ptr(pg), ptr(pu), str(stream));
    return rc ? status(rc) : py::make_tuple(dg, du, pg, pu);
}

py::object gelu(const Tensor &x, const Tensor &table, i64 stream) {
    if (!bf16(x)) return none();
    const i64 cols = last(x), rows = x.numel() / std::max<i64>(cols, 1);
    Tensor y = at::empty_like(x), parts = f32(x, {kParts});
    const int rc = call(gelu_c, ptr(x), rows, cols, ptr(table), ptr(y), ptr(parts), str(stream));
    return rc ? status(rc) : py::make_tuple(y, parts);
}

py::object gelu_bwd(const Tensor &dy, const Tensor &x, const Tensor &table, i64 stream) {
    if (!bf16(dy) || !bf16(x) || dy.sizes() != x.sizes()) return none();
    const i64 cols = last(x), rows = x.numel() / std::max<i64>(cols, 1);
    Tensor dx = at::empty_like(x), parts = f32(x, {kParts});
    const int rc = call(gelu_bwd_c, ptr(dy), ptr(x), rows, cols, ptr(table), ptr(dx), ptr(parts), str(stream));
    return rc ? status(rc) : py::make_tuple(dx, parts);
}

py::object gelu_bwd_slabs(const Tensor &dy, const Tensor &x, const Tensor &table, i64 stream) {
    if (!bf16(dy) || !bf16(x) || dy.sizes() != x.sizes() || x.numel() == 0) return none();
    const i64 cols = last(x), rows = x.numel() / cols;
    if (cols % 8 || cols > kParts * 256) return none();
    Tensor dx = at::empty_like(x), parts = f32(x, {kParts}), ws = f32(x, {kParts, ODL_FP8_COLSUM_WORKSPACE / kParts});
    const int rc = call(gelu_bwd_slabs_c, ptr(dy), ptr(x), rows, cols, ptr(table), ptr(dx), ptr(parts), ptr(ws), str(stream));
    return rc ? status(rc) : py::make_tuple(dx, parts, ws);
}

// rows of a norm: dense, aligned, with vectors of the row length in fp32 on the same device
bool norm_input(const Tensor &x) { return dense(x) && src_of(x) >= 0 && x.dim() > 0 && aligned(x); }
bool norm_vector(const Tensor &w, const Tensor &x) { return floats(w, x.size(-1)) && aligned(w) && w.device() == x.device(); }

py::object rmsnorm(const Tensor &x, const Tensor &w, double eps, i64 stream) {
    if (!norm_input(x) || !norm_vector(w, x)) return none();
    const i64 cols = x.size(-1), rows = x.numel() / std::max<i64>(cols, 1);
    Tensor y = at::empty(x.sizes(), x.options().dtype(at::kBFloat16)), rstd = f32(x, x.sizes().slice(0, x.dim() - 1)), parts = f32(x, {kParts});
    const int rc = call(rmsnorm_c, ptr(x), src_of(x), ptr(w), rows, cols, (float)eps, ptr(y), ptr(rstd), ptr(parts), str(stream));
    return rc ? status(rc) : py::make_tuple(y, rstd, parts);
}

py::object rmsnorm_bwd(const Tensor &dy, const Tensor &x, const Tensor &w, const Tensor &rstd, i64 stream) {
    if (!bf16(dy) || !norm_input(x) || dy.sizes() != x.sizes() || !norm_vector(w, x)) return none();
    const i64 cols = x.size(-1), rows = x.numel() / std::max<i64>(cols, 1);
    if (!floats(rstd, rows)) return none();
    Tensor dx = at::empty_like(x), dw = f32(x, {cols}), ws = f32(x, {ODL_FP8_RMSNORM_BWD_SLABS * cols});
    const int rc = call(rmsnorm_bwd_c, ptr(dy), ptr(x), src_of(x), ptr(w), ptr(rstd), rows, cols, ptr(dx), ptr(dw), ptr(ws), str(stream));
    return rc ? status(rc) : py::make_tuple(dx, dw);
}

py::object layernorm(const Tensor &x, const Tensor &w, const OptTensor &b, double eps, i64 stream) {
    if (!norm_input(x) || !norm_vector(w, x) || (b && !norm_vector(*b, x))) return none();
    const i64 cols = x.size(-1), rows = x.numel() / std::max<i64>(cols, 1);
    std::vector<i64> lead{2};
    for (int d = 0; d + 1 < x.dim(); ++d) lead.push_back(x.size(d));
    Tensor y = at::empty(x.sizes(), x.options().dtype(at::kBFloat16)), stats = f32(x, lead), parts = f32(x, {kParts});
    Tensor mean = stats.select(0, 0), rstd = stats.select(0, 1);
    const int rc = call(layernorm_c, ptr(x), src_of(x), ptr(w), ptr(b), rows, cols, (float)eps, ptr(y), ptr(mean), ptr(rstd), ptr(parts), str(stream));
    return rc ? status(rc) : py::make_tuple(y, mean, rstd, parts);
}

py::object layernorm_bwd(const Tensor &dy, const Tensor &x, const Tensor &w, const Tensor &mean, const Tensor &rstd, i64 stream) {
    if (!bf16(dy) || !norm_input(x) || dy.sizes() != x.sizes() || !norm_vector(w, x)) return none();
    const i64 cols = x.size(-1), rows = x.numel() / std::max<i64>(cols, 1);
    if (!floats(mean, rows) || !floats(rstd, rows)) return none();
    Tensor dx = at::empty_like(x), dwb = f32(x, {2 * cols}), ws = f32(x, {2 * ODL_FP8_RMSNORM_BWD_SLABS * cols});
    Tensor dw = dwb.narrow(0, 0, cols), db = dwb.narrow(0, cols, cols);
    const int rc = call(layernorm_bwd_c, ptr(dy), ptr(x), src_of(x), ptr(w), ptr(mean), ptr(rstd), rows, cols, ptr(dx), ptr(dw), ptr(db), ptr(ws),
                                   str(stream));
    return rc ? status(rc) : py::make_tuple(dx, dw, db);
}

py::object quantize_rowcol(const Tensor &x, int fmt, int margin, const std::optional<i64> &rows_out, i64 stream) {
    if (!source2d(x)) return none();
    const i64 rows = x.size(0), cols = x.size(1), n = rows_out.value_or(rows);
    const i64 pr = (rows + 3) / 4 * 4, pc = (cols + 3) / 4 * 4, o = pr + pc;      // every vector starts on a 16-byte boundary
    Tensor buf = f32(x, {3 * o});
    Tensor a_row = buf.narrow(0, 0, rows), a_col = buf.narrow(0, pr, cols), i_row = buf.narrow(0, 2 * o, rows), i_col = buf.narrow(0, 2 * o + pr, cols);
    float *base = buf.data_ptr<float>();
    Tensor q = bytes(x, {n, cols}), q_t = bytes(x, {cols, n});
    int rc = call(amax_rowcol_c, ptr(x), src_of(x), rows, cols, base, base + pr, str(stream));
    if (!rc)
        rc = call(cast_rowcol_c, ptr(x), src_of(x), rows, cols, n, base, base + pr, fmt, margin, ptr(q), ptr(q_t), base + o, base + 2 * o, base + o + pr,
                           base + 2 * o + pr, str(stream));
    return rc ? status(rc) : py::make_tuple(q, i_row, q_t, i_col, a_row, a_col);
}

bool out_fits(const OptTensor &out, i64 M, i64 N) { return !out || (dense(*out) && src_of(*out) >= 0 && out->dim() == 2 && out->size(0) == M && out->size(1) == N); }
Tensor result(const OptTensor &out, const Tensor &like, i64 M, i64 N, int odt) {
    return out ? *out : at::empty({M, N}, like.options().dtype(odt ? at::kFloat : at::kBFloat16));
}
bool small(i64 M, i64 N, i64 K) { return (M + 256) * K < (i64)1 << 31 && (N + 256) * K < (i64)1 << 31; }

// odt: 0 = bf16, 1 = fp32 (where no `out` decides).  split: K may be cut into runs, which the long way does.
py::object gemm_nt(const Tensor &a, const Tensor &b, int fa, int fb, const Tensor &sa, const Tensor &sb, const OptTensor &bias, int odt,
                   const OptTensor &out, bool accumulate, bool fresh, bool split, i64 stream) {
    if (!codes2d(a) || !codes2d(b) || a.size(1) != b.size(1)) return none();
    const i64 M = a.size(0), K = a.size(1), N = b.size(0), na = sa.numel(), nb = sb.numel();
    if ((na != 1 && na != M) || (nb != 1 && nb != N) || !floats(sa, na) || !floats(sb, nb) || (bias && !floats(*bias, N)) || !out_fits(out, M, N) ||
        (accumulate && !out) || (na > 1 && !aligned(sa)) || (nb > 1 && !aligned(sb)) || (bias && !aligned(*bias)))
        return none();
    if (split && small(M, N, K) && runs_c(M, N, K, 0) > 1) return none();
    Tensor c = result(out, a, M, N, odt);
    const int rc = call(gemm_nt_c, ptr(a), ptr(b), M, N, K, fa, fb, ptr(sa), na, ptr(sb), nb, ptr(bias), 1, ptr(c), src_of(c), accumulate, fresh, str(stream));
    return rc ? status(rc) : py::cast(c);
}

bool group_in_one_launch(const std::vector<i64> &M, const std::vector<i64> &N, i64 K, int odt) {
    return M.size() == N.size() && M.size() <= 4 && group_route_c((int)M.size(), M.data(), N.data(), K, odt) >= 0;
}

// Several products in one launch; None where they run one by one (each then in the way that is its own)
py::object gemm_nt_group(const std::vector<Tensor> &a, const std::vector<Tensor> &b, int fa, int fb, const std::vector<Tensor> &sa,
                         const std::vector<Tensor> &sb, int odt, bool fresh, i64 stream) {
    const size_t n = a.size();
    if (n < 2 || n > 4 || b.size() != n || sa.size() != n || sb.size() != n) return none();
    const uint8_t *pa[4], *pb[4];
    const float *psa[4], *psb[4];
    void *pc[4];
    i64 M[4], N[4];
    for (size_t s = 0; s < n; ++s) {
        if (!codes2d(a[s]) || !codes2d(b[s]) || a[s].size(1) != a[0].size(1) || b[s].size(1) != a[0].size(1) || !floats(sa[s], 1) || !floats(sb[s], 1) ||
            !aligned(a[s]) || !aligned(b[s]))
            return none();
        M[s] = a[s].size(0); N[s] = b[s].size(0);
        pa[s] = ptr(a[s]); pb[s] = ptr(b[s]); psa[s] = ptr(sa[s]); psb[s] = ptr(sb[s]);
    }
    const i64 K = a[0].size(1);
    if (group_route_c((int)n, M, N, K, odt) < 0) return none();
    py::list out;
    for (size_t s = 0; s < n; ++s) {
        Tensor c = result(OptTensor(), a[s], M[s], N[s], odt);
        pc[s] = ptr(c);
        out.append(c);
    }
    const int rc = call(gemm_nt_group_c, (int)n, pa, pb, M, N, K, fa, fb, psa, psb, pc, odt, fresh, str(stream));
    return rc ? status(rc) : py::object(out);
}

bool chain_in_one_launch(const std::vector<i64> &K, i64 M, i64 N) { return K.size() <= 4 && chain_route_c((int)K.size(), K.data(), M, N) >= 0; }

// The bf16 sum of several products in one launch
py::object gemm_nt_chain(const std::vector<Tensor> &a, const std::vector<Tensor> &b, int fa, int fb, const std::vector<Tensor> &sa,
                         const std::vector<Tensor> &sb, i64 stream) {
    const size_t n = a.size();
    if (n < 2 || n > 4 || b.size() != n || sa.size() != n || sb.size() != n) return none();
    const uint8_t *pa[4], *pb[4];
    const float *psa[4], *psb[4];
    i64 K[4];
    for (size_t s = 0; s < n; ++s) {
        if (!codes2d(a[s]) || !codes2d(b[s]) || a[s].size(0) != a[0].size(0) || b[s].size(0) != b[0].size(0) || a[s].size(1) != b[s].size(1)) return none();
        if (!floats(sa[s], 1) || !floats(sb[s], 1)) return none();
        K[s] = a[s].size(1);
        pa[s] = ptr(a[s]); pb[s] = ptr(b[s]); psa[s] = ptr(sa[s]); psb[s] = ptr(sb[s]);
    }
    Tensor c = result(OptTensor(), a[0], a[0].size(0), b[0].size(0), 0);
    const int rc = call(gemm_nt_chain_c, (int)n, pa, pb, K, a[0].size(0), b[0].size(0), fa, fb, psa, psb, ptr(c), str(stream));
    return rc ? status(rc) : py::cast(c);
}

// Not accumulating; whole tiles of the kernel that reads K-slow operands (the caller has checked: gemm_layouts_supported)
py::object gemm_layouts(const Tensor &a, const Tensor &b, int fa, int fb, bool a_slow, bool b_slow, const Tensor &sa, const Tensor &sb,
                        const OptTensor &out, int odt, bool split, i64 stream) {
    if (!codes2d(a) || !codes2d(b) || !floats(sa, 1) || !floats(sb, 1)) return none();
    const i64 M = a.size(a_slow ? 1 : 0), K = a.size(a_slow ? 0 : 1), N = b.size(b_slow ? 1 : 0);
    if (K != b.size(b_slow ? 0 : 1) || !out_fits(out, M, N) || M <= 0 || N <= 0 || M % 256 || N % 256 || K % 128 || K < 512 || !small(M, N, K)) return none();
    if (N * (i64)4 * 264 >= (i64)1 << 31 || (split && runs_c(M, N, K, a_slow || b_slow) > 1)) return none();
    Tensor c = result(out, a, M, N, odt);
    const int rc = call(gemm_layouts_c, ptr(a), ptr(b), M, N, K, fa, fb, a_slow, b_slow, ptr(sa), ptr(sb), ptr(c), src_of(c), str(stream));
    return rc ? status(rc) : py::cast(c);
}

// scale bytes of `rows` rows blocked along `length` elements, in the layout the streaming GEMM reads where the length allows
Tensor mx_scales(const Tensor &x, i64 rows, i64 length, int &layout) {
    layout = length % 128 == 0 && length > 0;
    return layout ? bytes(x, {length / 128, rows, 4}) : bytes(x, {rows, length / 32});
}

py::object mx_cast(const Tensor &x, int fmt, bool want_q, bool want_t, int rule, const std::optional<i64> &rows_out, i64 stream) {
    if (!source2d(x) || !(want_q || want_t)) return none();
    const i64 rows = x.size(0), cols = x.size(1), n = rows_out.value_or(rows);
    OptTensor q, s, q_t, s_t;
    int lay = 0, lay_t = 0;
    if (want_q) { q = bytes(x, {rows, cols}); s = mx_scales(x, rows, cols, lay); }
    if (want_t) { q_t = bytes(x, {cols, n}); s_t = mx_scales(x, cols, n, lay_t); }
    const int rc = call(mx_cast_c, ptr(x), src_of(x), rows, cols, n, fmt, ptr(q), ptr(s), lay, ptr(q_t), ptr(s_t), lay_t, rule, str(stream));
    return rc ? status(rc) : py::make_tuple(obj(q), obj(s), obj(q_t), obj(s_t));
}

py::object block_cast(const Tensor &x, int fmt, int margin, bool two_d, bool want_q, bool want_t, i64 stream) {
    if (!source2d(x) || !(want_q || want_t) || x.size(0) % 128 || x.size(1) % 128) return none();
    const i64 rows = x.size(0), cols = x.size(1);
    OptTensor q, s, q_t, s_t;
    if (want_q) { q = bytes(x, {rows, cols}); s = bytes(x, {cols / 128, rows, 4}); }
    if (want_t) { q_t = bytes(x, {cols, rows}); s_t = bytes(x, {rows / 128, cols, 4}); }
    const int rc = call(block_cast_c, ptr(x), src_of(x), rows, cols, fmt, margin, two_d, ptr(q), ptr(s), ptr(q_t), ptr(s_t), str(stream));
    return rc ? status(rc) : py::make_tuple(obj(q), obj(s), obj(q_t), obj(s_t));
}

py::object mx_gemm_nt(const Tensor &a, const Tensor &sa, const Tensor &b, const Tensor &sb, int fa, int fb, const OptTensor &bias, int odt,
                      const OptTensor &out, bool accumulate, bool fresh, bool split, i64 stream) {
    if (!codes2d(a) || !codes2d(b) || a.size(1) != b.size(1) || !dense(sa) || !dense(sb) || sa.scalar_type() != at::kByte || sb.scalar_type() != at::kByte)
        return none();
    const i64 M = a.size(0), K = a.size(1), N = b.size(0);
    // K-step-major scales only: what the casts of this package make wherever K has whole steps
    if (K % 128 || sa.dim() != 3 || sb.dim() != 3 || sa.size(0) != K / 128 || sa.size(1) != M || sa.size(2) != 4 || sb.size(0) != K / 128 ||
        sb.size(1) != N || sb.size(2) != 4)
        return none();
    if ((bias && !floats(*bias, N)) || !out_fits(out, M, N) || (accumulate && !out)) return none();
    if (split && small(M, N, K) && runs_c(M, N, K, 0) > 1) return none();
    Tensor c = result(out, a, M, N, odt);
    const int rc = call(mx_gemm_nt_c, ptr(a), ptr(sa), ptr(b), ptr(sb), 1, M, N, K, fa, fb, ptr(bias), ptr(c), src_of(c), accumulate, fresh, str(stream));
    return rc ? status(rc) : py::cast(c);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.attr("abi_version") = ODL_FP8_ABI_VERSION;        // of the header this was compiled with
    m.attr("torch_version") = TORCH_VERSION;
    m.def("bind", &bind);
    m.def("amax_parts", &amax_parts);
    m.def("cast_dynamic", &cast_dynamic);
    m.def("quantise_small", &quantise_small);
    m.def("gemm_swiglu", &gemm_swiglu);
    m.def("cast_delayed", &cast_delayed);
    m.def("cast_delayed_many", &cast_delayed_many);
    m.def("amax_colsum", &amax_colsum);
    m.def("slabs_colsum", &slabs_colsum);
    m.def("cast_colsum", &cast_colsum);
    m.def("swiglu", &swiglu);
    m.def("swiglu_bwd", &swiglu_bwd);
    m.def("gelu", &gelu);
    m.def("gelu_bwd", &gelu_bwd);
    m.def("gelu_bwd_slabs", &gelu_bwd_slabs);
    m.def("rmsnorm", &rmsnorm);
    m.def("rmsnorm_bwd", &rmsnorm_bwd);
    m.def("layernorm", &layernorm);
    m.def("layernorm_bwd", &layernorm_bwd);
    m.def("quantize_rowcol", &quantize_rowcol);
    m.def("gemm_nt", &gemm_nt);
    m.def("group_in_one_launch", &group_in_one_launch);
    m.def("gemm_nt_group", &gemm_nt_group);
    m.def("chain_in_one_launch", &chain_in_one_launch);
    m.def("gemm_nt_chain", &gemm_nt_chain);
    m.def("gemm_layouts", &gemm_layouts);
    m.def("mx_cast", &mx_cast);
    m.def("block_cast", &block_cast);
    m.def("mx_gemm_nt", &mx_gemm_nt);
}
