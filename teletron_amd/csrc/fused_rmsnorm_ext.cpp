// Python module `fused_rmsnorm`: the two functions of the reference's module of
// the same name, with the same argument order
// (teletron_op/fused_rmsnorm/rms_ops.cpp:6-13,25-33,47-55), plus the native
// backward that works from the saved input.  Unlike the reference glue, every
// argument is checked, the launch goes to PyTorch's current stream, and a
// failed launch raises.
#include <algorithm>

#include "torch_glue.h"

using namespace ttn_glue;

// output[rows, cols] = rmsnorm(input) * weight;  inv_variance[rows] = 1/rms  (fp32)
void torch_launch_rms_forward(torch::Tensor &output, const torch::Tensor &input,
                              const torch::Tensor &weight, int64_t rows, int64_t cols, double epsilon,
                              torch::Tensor &inv_variance) {
    const auto dev = input.device();
    check_dense_on(input, dev, "input");
    check_dense_on(output, dev, "output");
    check_dense_on(weight, dev, "weight");
    check_dense_on(inv_variance, dev, "inv_variance");
    const int dt = dtype_code(input, "input");
    TORCH_CHECK(rows >= 0 && cols > 0, "rows must be non-negative and cols positive");
    check_elems(input, rows * cols, input.scalar_type(), "input");
    check_elems(output, rows * cols, input.scalar_type(), "output");
    check_elems(weight, cols, input.scalar_type(), "weight");
    check_elems(inv_variance, rows, at::kFloat, "inv_variance");
    c10::DeviceGuard guard(dev);
    raise_on(tt_rmsnorm_forward(output.data_ptr(), inv_variance.data_ptr<float>(), input.data_ptr(),
                                weight.data_ptr(), rows, cols, epsilon, dt, current_stream(input)),
             "tt_rmsnorm_forward");
}

static void rms_backward_impl(torch::Tensor &dinp, torch::Tensor &dweight, const torch::Tensor &dout,
                              const torch::Tensor &saved, const torch::Tensor &weight,
                              const torch::Tensor &inv_variance, int64_t rows, int64_t cols,
                              bool saved_is_output) {
    const auto dev = dout.device();
    check_dense_on(dout, dev, "dout");
    check_dense_on(dinp, dev, "dinp");
    check_dense_on(dweight, dev, "dweight");
    check_dense_on(saved, dev, saved_is_output ? "x_norm" : "input");
    check_dense_on(weight, dev, "weight");
    check_dense_on(inv_variance, dev, "inv_variance");
    const int dt = dtype_code(dout, "dout");
    TORCH_CHECK(rows >= 0 && cols > 0, "rows must be non-negative and cols positive");
    check_elems(dout, rows * cols, dout.scalar_type(), "dout");
    check_elems(dinp, rows * cols, dout.scalar_type(), "dinp");
    check_elems(saved, rows * cols, dout.scalar_type(), saved_is_output ? "x_norm" : "input");
    check_elems(weight, cols, dout.scalar_type(), "weight");
    check_elems(dweight, cols, dout.scalar_type(), "dweight");
    check_elems(inv_variance, rows, at::kFloat, "inv_variance");
    c10::DeviceGuard guard(dev);
    const size_t need = tt_rmsnorm_backward_workspace_bytes(rows, cols, dt);
    TORCH_CHECK(need > 0 || rows == 0, "unsupported RMSNorm shape: cols=", cols);
    at::Tensor ws = scratch(need, dout);
    auto fn = saved_is_output ? tt_rmsnorm_backward_from_out : tt_rmsnorm_backward;
    raise_on(fn(dinp.data_ptr(), dweight.data_ptr(), dout.data_ptr(), saved.data_ptr(), weight.data_ptr(),
                inv_variance.data_ptr<float>(), rows, cols, dt, ws.data_ptr(), need, current_stream(dout)),
             saved_is_output ? "tt_rmsnorm_backward_from_out" : "tt_rmsnorm_backward");
}

// Reference contract: x_norm is the tensor torch_launch_rms_forward wrote to `output`.
void torch_launch_rms_backward(torch::Tensor &dinp, torch::Tensor &dweight, const torch::Tensor &dout,
                               const torch::Tensor &x_norm, const torch::Tensor &weight,
                               const torch::Tensor &inv_variance, int64_t rows, int64_t cols) {
    rms_backward_impl(dinp, dweight, dout, x_norm, weight, inv_variance, rows, cols, true);
}

// Native contract: `input` is the tensor that was normalised (forward then keeps no copy of its output).
void torch_launch_rms_backward_x(torch::Tensor &dinp, torch::Tensor &dweight, const torch::Tensor &dout,
                                 const torch::Tensor &input, const torch::Tensor &weight,
                                 const torch::Tensor &inv_variance, int64_t rows, int64_t cols) {
    rms_backward_impl(dinp, dweight, dout, input, weight, inv_variance, rows, cols, false);
}

// ---- strided views (no reference counterpart: the reference copies to contiguous first) ----
struct View3 {
    int64_t n[3], s[3];
};

// Leading dimensions of a <= 4-D view with contiguous last dimension, padded to three.
static View3 view3(const torch::Tensor &t, int64_t cols, const char *name) {
    TORCH_CHECK(t.dim() >= 1 && t.dim() <= 4, name, " must have 1 to 4 dimensions, got ", t.dim());
    TORCH_CHECK(t.size(-1) == cols && t.stride(-1) == 1, name, " needs a contiguous last dimension of ", cols);
    View3 v{{1, 1, 1}, {0, 0, 0}};
    const int64_t lead = t.dim() - 1;
    for (int64_t d = 0; d < lead; ++d) {
        v.n[3 - lead + d] = t.size(d);
        v.s[3 - lead + d] = t.stride(d);
    }
    return v;
}

// output (contiguous, input's shape) = rmsnorm(input view) * weight; inv_variance in output row order.
void torch_launch_rms_forward_strided(torch::Tensor &output, const torch::Tensor &input,
                                      const torch::Tensor &weight, double epsilon,
                                      torch::Tensor &inv_variance) {
    const auto dev = input.device();
    TORCH_CHECK(input.is_cuda(), "input must be a GPU tensor");
    check_dense_on(output, dev, "output");
    check_dense_on(weight, dev, "weight");
    check_dense_on(inv_variance, dev, "inv_variance");
    const int dt = dtype_code(input, "input");
    const int64_t cols = weight.numel();
    const View3 v = view3(input, cols, "input");
    const int64_t rows = v.n[0] * v.n[1] * v.n[2];
    check_elems(output, rows * cols, input.scalar_type(), "output");
    check_elems(weight, cols, input.scalar_type(), "weight");
    check_elems(inv_variance, rows, at::kFloat, "inv_variance");
    c10::DeviceGuard guard(dev);
    raise_on(tt_rmsnorm_forward_strided(output.data_ptr(), inv_variance.data_ptr<float>(), input.data_ptr(),
                                        weight.data_ptr(), v.n[0], v.n[1], v.n[2], v.s[0], v.s[1], v.s[2], cols,
                                        epsilon, dt, current_stream(input)),
             "tt_rmsnorm_forward_strided");
}

// dinp: any view of input's shape (its strides choose the layout dx is written in); dout contiguous.
void torch_launch_rms_backward_strided(torch::Tensor &dinp, torch::Tensor &dweight, const torch::Tensor &dout,
                                       const torch::Tensor &input, const torch::Tensor &weight,
                                       const torch::Tensor &inv_variance) {
    const auto dev = dout.device();
    TORCH_CHECK(input.is_cuda() && dinp.is_cuda(), "input and dinp must be GPU tensors");
    TORCH_CHECK(input.device() == dev && dinp.device() == dev, "tensors are on different devices");
    check_dense_on(dout, dev, "dout");
    check_dense_on(dweight, dev, "dweight");
    check_dense_on(weight, dev, "weight");
    check_dense_on(inv_variance, dev, "inv_variance");
    const int dt = dtype_code(dout, "dout");
    const int64_t cols = weight.numel();
    const View3 vx = view3(input, cols, "input");
    const View3 vd = view3(dinp, cols, "dinp");
    TORCH_CHECK(input.sizes() == dinp.sizes(), "dinp must have input's shape");
    const int64_t rows = vx.n[0] * vx.n[1] * vx.n[2];
    TORCH_CHECK(input.scalar_type() == dout.scalar_type() && dinp.scalar_type() == dout.scalar_type(),
                "input, dinp and dout must share a dtype");
    check_elems(dout, rows * cols, dout.scalar_type(), "dout");
    check_elems(weight, cols, dout.scalar_type(), "weight");
    check_elems(dweight, cols, dout.scalar_type(), "dweight");
    check_elems(inv_variance, rows, at::kFloat, "inv_variance");
    c10::DeviceGuard guard(dev);
    const size_t need = tt_rmsnorm_backward_workspace_bytes(rows, cols, dt);
    TORCH_CHECK(need > 0 || rows == 0, "unsupported RMSNorm shape: cols=", cols);
    at::Tensor ws = scratch(need, dout);
    raise_on(tt_rmsnorm_backward_strided(dinp.data_ptr(), dweight.data_ptr(), dout.data_ptr(), input.data_ptr(),
                                         weight.data_ptr(), inv_variance.data_ptr<float>(), vx.n[0], vx.n[1],
                                         vx.n[2], vx.s[0], vx.s[1], vx.s[2], vd.s[0], vd.s[1], vd.s[2], cols, dt,
                                         ws.data_ptr(), need, current_stream(dout)),
             "tt_rmsnorm_backward_strided");
}

// dst: any view (<= 4-D, contiguous last dimension) of src's shape; src contiguous.  The value gradient of the
// QK-norm call site goes into its slice of the fused projection's gradient with this.
void torch_launch_copy_rows_strided(torch::Tensor &dst, const torch::Tensor &src) {
    const auto dev = src.device();
    TORCH_CHECK(dst.is_cuda() && dst.device() == dev, "dst and src must be on the same GPU");
    check_dense_on(src, dev, "src");
    TORCH_CHECK(dst.sizes() == src.sizes() && dst.scalar_type() == src.scalar_type(), "dst must have src's shape and dtype");
    const int dt = dtype_code(src, "src");
    const int64_t cols = src.size(-1);
    const View3 vd = view3(dst, cols, "dst");
    c10::DeviceGuard guard(dev);
    raise_on(tt_norm_copy_rows_strided(dst.data_ptr(), src.data_ptr(), vd.n[0], vd.n[1], vd.n[2], vd.s[0], vd.s[1],
                                       vd.s[2], cols, dt, current_stream(src)),
             "tt_norm_copy_rows_strided");
}

// ---- strided QK-norm with the rotary embedding behind it (no reference counterpart: the reference
// runs apply_rotary_emb as separate PyTorch ops on the norm's output) ----
static int64_t check_rope_tables(const torch::Tensor &cos, const torch::Tensor &sin, const at::Device &dev,
                                 int64_t cols, int64_t seq) {
    check_dense_on(cos, dev, "freqs_cos");
    check_dense_on(sin, dev, "freqs_sin");
    TORCH_CHECK(cos.scalar_type() == at::kFloat && sin.scalar_type() == at::kFloat, "freqs_cos/freqs_sin must be float32");
    TORCH_CHECK(cos.dim() == 2 && cos.size(1) == cols && cos.sizes() == sin.sizes(),
                "freqs_cos/freqs_sin must both be [tokens, ", cols, "]");
    TORCH_CHECK(cos.size(0) <= seq, "rotary tables hold ", cos.size(0), " tokens, the view only ", seq);
    return cos.size(0);
}

// input: a [B, H, S, D] view (or fewer leading dimensions); rows at token index >= freqs_cos.size(0) are
// normalised but not rotated.
void torch_launch_rms_rope_forward_strided(torch::Tensor &output, const torch::Tensor &input,
                                           const torch::Tensor &weight, double epsilon,
                                           torch::Tensor &inv_variance, const torch::Tensor &freqs_cos,
                                           const torch::Tensor &freqs_sin) {
    const auto dev = input.device();
    TORCH_CHECK(input.is_cuda(), "input must be a GPU tensor");
    check_dense_on(output, dev, "output");
    check_dense_on(weight, dev, "weight");
    check_dense_on(inv_variance, dev, "inv_variance");
    const int dt = dtype_code(input, "input");
    const int64_t cols = weight.numel();
    const View3 v = view3(input, cols, "input");
    const int64_t rows = v.n[0] * v.n[1] * v.n[2];
    const int64_t tokens = check_rope_tables(freqs_cos, freqs_sin, dev, cols, v.n[2]);
    check_elems(output, rows * cols, input.scalar_type(), "output");
    check_elems(weight, cols, input.scalar_type(), "weight");
    check_elems(inv_variance, rows, at::kFloat, "inv_variance");
    c10::DeviceGuard guard(dev);
    raise_on(tt_rmsnorm_rope_forward_strided(output.data_ptr(), inv_variance.data_ptr<float>(), input.data_ptr(),
                                             weight.data_ptr(), freqs_cos.data_ptr<float>(),
                                             freqs_sin.data_ptr<float>(), tokens, v.n[0], v.n[1], v.n[2], v.s[0],
                                             v.s[1], v.s[2], cols, epsilon, dt, current_stream(input)),
             "tt_rmsnorm_rope_forward_strided");
}

// dout: gradient of the rotated output (contiguous); dinp as in torch_launch_rms_backward_strided.
void torch_launch_rms_rope_backward_strided(torch::Tensor &dinp, torch::Tensor &dweight, const torch::Tensor &dout,
                                            const torch::Tensor &input, const torch::Tensor &weight,
                                            const torch::Tensor &inv_variance, const torch::Tensor &freqs_cos,
                                            const torch::Tensor &freqs_sin) {
    const auto dev = dout.device();
    TORCH_CHECK(input.is_cuda() && dinp.is_cuda(), "input and dinp must be GPU tensors");
    TORCH_CHECK(input.device() == dev && dinp.device() == dev, "tensors are on different devices");
    check_dense_on(dout, dev, "dout");
    check_dense_on(dweight, dev, "dweight");
    check_dense_on(weight, dev, "weight");
    check_dense_on(inv_variance, dev, "inv_variance");
    const int dt = dtype_code(dout, "dout");
    const int64_t cols = weight.numel();
    const View3 vx = view3(input, cols, "input");
    const View3 vd = view3(dinp, cols, "dinp");
    TORCH_CHECK(input.sizes() == dinp.sizes(), "dinp must have input's shape");
    const int64_t rows = vx.n[0] * vx.n[1] * vx.n[2];
    const int64_t tokens = check_rope_tables(freqs_cos, freqs_sin, dev, cols, vx.n[2]);
    TORCH_CHECK(input.scalar_type() == dout.scalar_type() && dinp.scalar_type() == dout.scalar_type(),
                "input, dinp and dout must share a dtype");
    check_elems(dout, rows * cols, dout.scalar_type(), "dout");
    check_elems(weight, cols, dout.scalar_type(), "weight");
    check_elems(dweight, cols, dout.scalar_type(), "dweight");
    check_elems(inv_variance, rows, at::kFloat, "inv_variance");
    c10::DeviceGuard guard(dev);
    const size_t need = tt_rmsnorm_backward_workspace_bytes(rows, cols, dt);
    TORCH_CHECK(need > 0 || rows == 0, "unsupported RMSNorm shape: cols=", cols);
    at::Tensor ws = scratch(need, dout);
    raise_on(tt_rmsnorm_rope_backward_strided(dinp.data_ptr(), dweight.data_ptr(), dout.data_ptr(), input.data_ptr(),
                                              weight.data_ptr(), inv_variance.data_ptr<float>(),
                                              freqs_cos.data_ptr<float>(), freqs_sin.data_ptr<float>(), tokens,
                                              vx.n[0], vx.n[1], vx.n[2], vx.s[0], vx.s[1], vx.s[2], vd.s[0], vd.s[1],
                                              vd.s[2], cols, dt, ws.data_ptr(), need, current_stream(dout)),
             "tt_rmsnorm_rope_backward_strided");
}

// ---- the whole QK-norm call site in one kernel per direction (no reference counterpart) ----
struct QkvShape {
    int64_t B, S, H, cols, tokens;
    int dt;
};

static QkvShape check_qkv(const torch::Tensor &mixed, const torch::Tensor &weight_q, const torch::Tensor &weight_k,
                          const c10::optional<torch::Tensor> &cos, const c10::optional<torch::Tensor> &sin) {
    const auto dev = mixed.device();
    check_dense_on(mixed, dev, "mixed_qkv");
    TORCH_CHECK(mixed.dim() == 4 && mixed.size(3) % 3 == 0, "mixed_qkv must be [B, S, H, 3*D]");
    const int64_t cols = mixed.size(3) / 3;
    for (auto *w : {&weight_q, &weight_k}) {
        check_dense_on(*w, dev, "weight");
        check_elems(*w, cols, mixed.scalar_type(), "weight");
    }
    TORCH_CHECK(cos.has_value() == sin.has_value(), "pass freqs_cos and freqs_sin together, or neither");
    const int64_t tokens = cos.has_value() ? check_rope_tables(*cos, *sin, dev, cols, mixed.size(1)) : 0;
    return {mixed.size(0), mixed.size(1), mixed.size(2), cols, tokens, dtype_code(mixed, "mixed_qkv")};
}

static const float *table_ptr(const c10::optional<torch::Tensor> &t) {
    return t.has_value() ? t->data_ptr<float>() : nullptr;
}

// query, key [B, H, S, D] contiguous = RMSNorm of their slices of mixed, rotated on the tokens of the tables
void torch_launch_qkv_rms_forward(torch::Tensor &query, torch::Tensor &key, const torch::Tensor &mixed,
                                  const torch::Tensor &weight_q, const torch::Tensor &weight_k, double epsilon,
                                  const c10::optional<torch::Tensor> &freqs_cos,
                                  const c10::optional<torch::Tensor> &freqs_sin) {
    const QkvShape s = check_qkv(mixed, weight_q, weight_k, freqs_cos, freqs_sin);
    for (auto *t : {&query, &key}) {
        check_dense_on(*t, mixed.device(), "query/key");
        check_elems(*t, s.B * s.S * s.H * s.cols, mixed.scalar_type(), "query/key");
    }
    c10::DeviceGuard guard(mixed.device());
    raise_on(tt_qkv_rmsnorm_forward(query.data_ptr(), key.data_ptr(), mixed.data_ptr(), weight_q.data_ptr(),
                                    weight_k.data_ptr(), table_ptr(freqs_cos), table_ptr(freqs_sin), s.tokens, s.B, s.S,
                                    s.H, s.cols, epsilon, s.dt, current_stream(mixed)),
             "tt_qkv_rmsnorm_forward");
}

// dmixed is written whole; dquery / dkey / dvalue contiguous [B, H, S, D], or None for an output that was not used
void torch_launch_qkv_rms_backward(torch::Tensor &dmixed, torch::Tensor &dweight_q, torch::Tensor &dweight_k,
                                   const c10::optional<torch::Tensor> &dquery, const c10::optional<torch::Tensor> &dkey,
                                   const c10::optional<torch::Tensor> &dvalue, const torch::Tensor &mixed,
                                   const torch::Tensor &weight_q, const torch::Tensor &weight_k, double epsilon,
                                   const c10::optional<torch::Tensor> &freqs_cos,
                                   const c10::optional<torch::Tensor> &freqs_sin) {
    const QkvShape s = check_qkv(mixed, weight_q, weight_k, freqs_cos, freqs_sin);
    const auto dev = mixed.device();
    const auto st = mixed.scalar_type();
    const int64_t n = s.B * s.S * s.H * s.cols;
    check_dense_on(dmixed, dev, "dmixed");
    check_elems(dmixed, 3 * n, st, "dmixed");
    for (auto *t : {&dweight_q, &dweight_k}) {
        check_dense_on(*t, dev, "dweight");
        check_elems(*t, s.cols, st, "dweight");
    }
    const void *g[3] = {nullptr, nullptr, nullptr};
    const c10::optional<torch::Tensor> *grads[3] = {&dquery, &dkey, &dvalue};
    for (int i = 0; i < 3; ++i) {
        if (!grads[i]->has_value() || !(*grads[i])->defined()) continue;
        check_dense_on(**grads[i], dev, "dquery/dkey/dvalue");
        check_elems(**grads[i], n, st, "dquery/dkey/dvalue");
        g[i] = (*grads[i])->data_ptr();
    }
    c10::DeviceGuard guard(dev);
    const size_t need = tt_qkv_rmsnorm_backward_workspace_bytes(s.B, s.S, s.H, s.cols, s.dt);
    TORCH_CHECK(need > 0 || n == 0, "unsupported head dimension ", s.cols);
    at::Tensor ws = scratch(need, mixed);
    raise_on(tt_qkv_rmsnorm_backward(dmixed.data_ptr(), dweight_q.data_ptr(), dweight_k.data_ptr(), g[0], g[1], g[2],
                                     mixed.data_ptr(), weight_q.data_ptr(), weight_k.data_ptr(), table_ptr(freqs_cos),
                                     table_ptr(freqs_sin), s.tokens, s.B, s.S, s.H, s.cols, epsilon, s.dt, ws.data_ptr(),
                                     need, current_stream(mixed)),
             "tt_qkv_rmsnorm_backward");
}

// ---- whole calls (see torch_glue.h) ----

using Tensors = std::vector<torch::Tensor>;

// Uninitialised tensor of x's shape laid out in x's dimension order but without its gaps.
static torch::Tensor dense_like_layout(const torch::Tensor &x) {
    std::vector<int64_t> order(x.dim()), sizes(x.dim()), place(x.dim());
    for (int64_t d = 0; d < x.dim(); ++d) order[d] = d;
    std::stable_sort(order.begin(), order.end(), [&](int64_t a, int64_t b) { return x.stride(a) > x.stride(b); });
    for (int64_t i = 0; i < x.dim(); ++i) {
        sizes[i] = x.size(order[i]);
        place[order[i]] = i;
    }
    return at::empty(sizes, x.options()).permute(place);
}

// out, inv_variance
static c10::optional<Tensors> rms_forward(const torch::Tensor &x, const torch::Tensor &weight, int64_t cols, double epsilon) {
    if (!ready_rows(x, cols) || !ready(weight, x) || weight.numel() != cols) return c10::nullopt;
    const int64_t rows = x.numel() / cols;
    torch::Tensor out = at::empty(x.sizes(), x.options()), inv_variance = row_statistics(x, rows);
    torch_launch_rms_forward(out, x, weight, rows, cols, epsilon, inv_variance);
    return Tensors{out, inv_variance};
}

// dinp, dweight
static c10::optional<Tensors> rms_backward(const torch::Tensor &dout, const torch::Tensor &x, const torch::Tensor &weight,
                                           const torch::Tensor &inv_variance, int64_t cols, bool strided) {
    if (!ready(dout, x)) return c10::nullopt;
    torch::Tensor dweight = at::empty_like(weight), dinp = strided ? dense_like_layout(x) : at::empty_like(x);
    if (strided)
        torch_launch_rms_backward_strided(dinp, dweight, dout, x, weight, inv_variance);
    else
        rms_backward_impl(dinp, dweight, dout, x, weight, inv_variance, x.numel() / cols, cols, false);
    return Tensors{dinp, dweight};
}

static bool qkv_ready(const torch::Tensor &mixed, const torch::Tensor &weight_q, const torch::Tensor &weight_k,
                      const c10::optional<torch::Tensor> &cos, const c10::optional<torch::Tensor> &sin) {
    if (mixed.dim() != 4 || mixed.size(3) % 3 != 0) return false;
    const int64_t cols = mixed.size(3) / 3;
    if (!ready_rows(mixed, cols) || !tt_qkv_rmsnorm_supported(cols, dtype_code(mixed, "mixed_qkv"))) return false;
    if (!cos.has_value() && mixed.numel() / mixed.size(3) > INT32_MAX) return false;  // beyond the joint kernels' units
    for (auto *w : {&weight_q, &weight_k})
        if (!ready(*w, mixed) || w->numel() != cols) return false;
    if (cos.has_value() != sin.has_value()) return false;
    if (cos.has_value()) {
        for (auto *t : {&*cos, &*sin})
            if (t->scalar_type() != at::kFloat || !ready(*t, *t) || t->device() != mixed.device() || t->dim() != 2 ||
                t->size(1) != cols || cols != 128 || t->size(0) > mixed.size(1))
                return false;
        if (cos->sizes() != sin->sizes()) return false;
    }
    return true;
}

// query, key, value of ready operands: value is the transposed view of its slice of mixed
static Tensors qkv_run(const torch::Tensor &mixed, const torch::Tensor &weight_q, const torch::Tensor &weight_k, double epsilon,
                       const c10::optional<torch::Tensor> &cos, const c10::optional<torch::Tensor> &sin) {
    const int64_t cols = mixed.size(3) / 3;
    const std::vector<int64_t> shape{mixed.size(0), mixed.size(2), mixed.size(1), cols};
    torch::Tensor query = at::empty(shape, mixed.options()), key = at::empty(shape, mixed.options());
    torch_launch_qkv_rms_forward(query, key, mixed, weight_q, weight_k, epsilon, cos, sin);
    return {query, key, mixed.slice(3, 2 * cols, 3 * cols).transpose(1, 2)};
}

static c10::optional<Tensors> qkv_forward(const torch::Tensor &mixed, const torch::Tensor &weight_q,
                                          const torch::Tensor &weight_k, double epsilon,
                                          const c10::optional<torch::Tensor> &cos, const c10::optional<torch::Tensor> &sin) {
    if (!qkv_ready(mixed, weight_q, weight_k, cos, sin)) return c10::nullopt;
    return qkv_run(mixed, weight_q, weight_k, epsilon, cos, sin);
}

// dmixed, dweight_q, dweight_k; a gradient may be None
static c10::optional<Tensors> qkv_backward(const c10::optional<torch::Tensor> &dquery, const c10::optional<torch::Tensor> &dkey,
                                           const c10::optional<torch::Tensor> &dvalue, const torch::Tensor &mixed,
                                           const torch::Tensor &weight_q, const torch::Tensor &weight_k, double epsilon,
                                           const c10::optional<torch::Tensor> &cos, const c10::optional<torch::Tensor> &sin) {
    for (auto *g : {&dquery, &dkey, &dvalue})
        if (g->has_value() && (*g)->defined() && !ready(**g, mixed)) return c10::nullopt;
    torch::Tensor dmixed = at::empty_like(mixed), dwq = at::empty_like(weight_q), dwk = at::empty_like(weight_k);
    torch_launch_qkv_rms_backward(dmixed, dwq, dwk, dquery, dkey, dvalue, mixed, weight_q, weight_k, epsilon, cos, sin);
    return Tensors{dmixed, dwq, dwk};
}

// ---- call sites (see torch_glue.h): RMSNormModelFunction and QKVSplitNormFunction ----

using torch::autograd::AutogradContext;
using torch::autograd::Function;

// A view whose rows the strided kernels read in place: at most 4-D, last dimension contiguous, every other stride a
// non-negative multiple of 16 bytes.
static bool ready_view(const torch::Tensor &x, int64_t cols) {
    const auto st = x.scalar_type();
    if (!x.is_cuda() || (st != at::kBFloat16 && st != at::kHalf && st != at::kFloat)) return false;
    if (x.dim() < 2 || x.dim() > 4 || x.size(-1) != cols || x.stride(-1) != 1 || x.is_contiguous()) return false;
    const int64_t vec = 16 / x.element_size();
    for (int64_t d = 0; d + 1 < x.dim(); ++d)
        if (x.stride(d) < 0 || x.stride(d) % vec != 0) return false;
    return (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0 && tt_norm_supported(cols, dtype_code(x, "input"));
}

static bool ready_parameter(const torch::Tensor &w, const torch::Tensor &x, int64_t cols) {
    return ready(w, w) && w.numel() == cols && w.scalar_type() == x.scalar_type() && w.device() == x.device();
}

struct RmsSite : Function<RmsSite> {
    static torch::Tensor forward(AutogradContext *ctx, const torch::Tensor &x, const torch::Tensor &weight, int64_t cols,
                                 double epsilon, bool strided) {
        const int64_t rows = x.numel() / cols;
        torch::Tensor out = at::empty(x.sizes(), x.options()), inv_variance = row_statistics(x, rows);
        if (strided)
            torch_launch_rms_forward_strided(out, x, weight, epsilon, inv_variance);
        else
            torch_launch_rms_forward(out, x, weight, rows, cols, epsilon, inv_variance);
        ctx->save_for_backward({x, weight, inv_variance});
        ctx->saved_data["cols"] = cols;
        ctx->saved_data["strided"] = strided;
        return out;
    }
    static Tensors backward(AutogradContext *ctx, Tensors grads) {
        const Tensors kept = ctx->get_saved_variables();
        Tensors d = taken(rms_backward(prepared(grads[0], kept[1]), kept[0], kept[1], kept[2], ctx->saved_data["cols"].toInt(),
                                  ctx->saved_data["strided"].toBool()), "rms_backward");
        return first_order({d[0], d[1], {}, {}, {}}, kept, grads);
    }
};

struct QkvSite : Function<QkvSite> {
    static Tensors forward(AutogradContext *ctx, const torch::Tensor &mixed, const torch::Tensor &weight_q,
                           const torch::Tensor &weight_k, double epsilon, const c10::optional<torch::Tensor> &cos,
                           const c10::optional<torch::Tensor> &sin) {
        Tensors outs = qkv_run(mixed, weight_q, weight_k, epsilon, cos, sin);
        ctx->set_materialize_grads(false);
        Tensors keep{mixed, weight_q, weight_k};
        if (cos.has_value()) keep.insert(keep.end(), {*cos, *sin});
        ctx->save_for_backward(std::move(keep));
        ctx->saved_data["epsilon"] = epsilon;
        return outs;
    }
    static Tensors backward(AutogradContext *ctx, Tensors grads) {
        const Tensors kept = ctx->get_saved_variables();
        for (auto &g : grads) g = prepared(g, kept[0]);
        c10::optional<torch::Tensor> cos, sin;
        if (kept.size() > 3) cos = kept[3], sin = kept[4];
        Tensors d = taken(qkv_backward(grads[0], grads[1], grads[2], kept[0], kept[1], kept[2], ctx->saved_data["epsilon"].toDouble(),
                                  cos, sin), "qkv_backward");
        return first_order({d[0], d[1], d[2], {}, {}, {}}, kept, grads);
    }
};

static c10::optional<torch::Tensor> rms_site(const torch::Tensor &x, const torch::Tensor &weight, int64_t cols, double epsilon) {
    if (!ordinary_call({&x, &weight}) || !ready_parameter(weight, x, cols)) return c10::nullopt;
    const bool strided = ready_view(x, cols);
    if (!strided && !ready_rows(x, cols)) return c10::nullopt;
    return RmsSite::apply(x, weight, cols, epsilon, strided);
}

static c10::optional<std::tuple<torch::Tensor, torch::Tensor, torch::Tensor>> qkv_site(
    const torch::Tensor &mixed, const torch::Tensor &weight_q, const torch::Tensor &weight_k, double epsilon,
    const c10::optional<torch::Tensor> &cos, const c10::optional<torch::Tensor> &sin) {
    if (!ordinary_call({&mixed, &weight_q, &weight_k}) || (cos.has_value() && sin.has_value() && !ordinary_call({&*cos, &*sin})) ||
        !qkv_ready(mixed, weight_q, weight_k, cos, sin))
        return c10::nullopt;
    Tensors outs = QkvSite::apply(mixed, weight_q, weight_k, epsilon, cos, sin);
    return std::make_tuple(outs[0], outs[1], outs[2]);
}

PYBIND11_MODULE(fused_rmsnorm, m) {
    m.def("rms_site", &rms_site, "RMSNormModelFunction as a native autograd node; None unless every operand is ready");
    m.def("qkv_site", &qkv_site, "QKVSplitNormFunction as a native autograd node; None unless every operand is ready");
    m.def("rms_forward", &rms_forward, "RMSNorm forward: out, inv_variance; None unless every operand is ready");
    m.def("rms_backward", &rms_backward, "RMSNorm backward: dinp, dweight; None unless the gradient is ready");
    m.def("qkv_forward", &qkv_forward, "query, key, value of a fused projection; None unless every operand is ready");
    m.def("qkv_backward", &qkv_backward, "its backward: dmixed, dweight_q, dweight_k; None unless the gradients are ready");
    m.def("torch_launch_qkv_rms_forward", &torch_launch_qkv_rms_forward,
          "RMSNorm (and rotary embedding) of the query and key slices of a fused projection");
    m.def("torch_launch_qkv_rms_backward", &torch_launch_qkv_rms_backward,
          "backward of torch_launch_qkv_rms_forward: the projection's whole gradient and both weight gradients");
    m.def("torch_launch_copy_rows_strided", &torch_launch_copy_rows_strided,
          "rows of a contiguous tensor into a strided view of the same shape");
    m.def("torch_launch_rms_rope_forward_strided", &torch_launch_rms_rope_forward_strided,
          "strided RMSNorm forward with the rotary embedding applied to the result");
    m.def("torch_launch_rms_rope_backward_strided", &torch_launch_rms_rope_backward_strided,
          "backward of the strided RMSNorm + rotary embedding");
    m.def("torch_launch_rms_forward", &torch_launch_rms_forward, "RMSNorm forward kernel");
    m.def("torch_launch_rms_backward", &torch_launch_rms_backward,
          "RMSNorm backward kernel (from the saved forward output)");
    m.def("torch_launch_rms_backward_x", &torch_launch_rms_backward_x,
          "RMSNorm backward kernel (from the saved input)");
    m.def("torch_launch_rms_forward_strided", &torch_launch_rms_forward_strided,
          "RMSNorm forward kernel reading a strided view (contiguous last dimension) in place");
    m.def("torch_launch_rms_backward_strided", &torch_launch_rms_backward_strided,
          "RMSNorm backward kernel for a strided input view; dx is written through dinp's strides");
    m.def("supported", [](int64_t cols, const torch::Tensor &like) {
        return tt_norm_supported(cols, like.scalar_type() == at::kBFloat16 ? TT_NORM_BF16
                                       : like.scalar_type() == at::kFloat  ? TT_NORM_F32
                                       : like.scalar_type() == at::kHalf   ? TT_NORM_F16 : -1) != 0;
    }, "whether the kernels are built for this column count and dtype");
}

// Same operator namespace as the reference registers (rms_ops.cpp:58-61).
TORCH_LIBRARY(Fused_RMSNorm, m) {
    m.def("torch_launch_rms_forward(Tensor(a!) output, Tensor input, Tensor weight, int rows, int cols, "
          "float epsilon, Tensor(b!) inv_variance) -> ()",
          &torch_launch_rms_forward);
    m.def("torch_launch_rms_backward(Tensor(a!) dinp, Tensor(b!) dweight, Tensor dout, Tensor x_norm, "
          "Tensor weight, Tensor inv_variance, int rows, int cols) -> ()",
          &torch_launch_rms_backward);
}
