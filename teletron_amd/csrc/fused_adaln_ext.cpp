// Python module `fused_adaln`: the two functions of the reference's module of
// the same name, with the same argument order
// (teletron_op/fused_adaln/adaln_ops.cpp:6-15,29-38,52-60), plus the native
// pair that saves row statistics instead of a second full-size tensor.
// scale/shift may hold one row per sample ([batch, cols]); rows are then
// grouped by sample, rows/batch consecutive rows each.
#include "torch_glue.h"

using namespace ttn_glue;

struct AdalnShape {
    int64_t batch, rows_per_sample;
    int dt;
};

static AdalnShape adaln_shape(const torch::Tensor &x, const torch::Tensor &scale, int64_t rows, int64_t cols) {
    TORCH_CHECK(rows >= 0 && cols > 0, "rows must be non-negative and cols positive");
    TORCH_CHECK(scale.numel() > 0 && scale.numel() % cols == 0, "scale has ", scale.numel(),
                " elements, not a multiple of cols=", cols);
    const int64_t batch = scale.numel() / cols;
    TORCH_CHECK(rows % batch == 0, "rows=", rows, " is not a multiple of the ", batch, " modulation rows");
    return {batch, rows / batch, dtype_code(x, "input")};
}

void torch_launch_adaln_forward(torch::Tensor &output, torch::Tensor &x_norm, const torch::Tensor &input,
                                const torch::Tensor &scale, const torch::Tensor &shift, int64_t rows,
                                int64_t cols, double epsilon, torch::Tensor &inv_variance) {
    const auto dev = input.device();
    for (auto *t : {&output, &x_norm, &inv_variance}) check_dense_on(*t, dev, "output tensor");
    for (auto *t : {&input, &scale, &shift}) check_dense_on(*t, dev, "input tensor");
    const AdalnShape s = adaln_shape(input, scale, rows, cols);
    const auto st = input.scalar_type();
    check_elems(input, rows * cols, st, "input");
    check_elems(output, rows * cols, st, "output");
    check_elems(x_norm, rows * cols, st, "x_norm");
    check_elems(shift, scale.numel(), st, "shift");
    check_elems(scale, scale.numel(), st, "scale");
    check_elems(inv_variance, rows, at::kFloat, "inv_variance");
    c10::DeviceGuard guard(dev);
    raise_on(tt_adaln_forward_xnorm(output.data_ptr(), x_norm.data_ptr(), inv_variance.data_ptr<float>(),
                                    input.data_ptr(), scale.data_ptr(), shift.data_ptr(), s.batch,
                                    s.rows_per_sample, cols, epsilon, s.dt, current_stream(input)),
             "tt_adaln_forward_xnorm");
}

static void adaln_forward_stats_impl(torch::Tensor &output, const torch::Tensor &input,
                                     const torch::Tensor &scale, const torch::Tensor &shift, int64_t rows,
                                     int64_t cols, double epsilon, torch::Tensor &mean,
                                     torch::Tensor &inv_variance, bool seq_first) {
    const auto dev = input.device();
    for (auto *t : {&output, &mean, &inv_variance}) check_dense_on(*t, dev, "output tensor");
    for (auto *t : {&input, &scale, &shift}) check_dense_on(*t, dev, "input tensor");
    const AdalnShape s = adaln_shape(input, scale, rows, cols);
    const auto st = input.scalar_type();
    check_elems(input, rows * cols, st, "input");
    check_elems(output, rows * cols, st, "output");
    check_elems(shift, scale.numel(), st, "shift");
    check_elems(scale, scale.numel(), st, "scale");
    check_elems(mean, rows, at::kFloat, "mean");
    check_elems(inv_variance, rows, at::kFloat, "inv_variance");
    c10::DeviceGuard guard(dev);
    if (seq_first)
        raise_on(tt_adaln_forward_seq_first(output.data_ptr(), mean.data_ptr<float>(), inv_variance.data_ptr<float>(),
                                            input.data_ptr(), scale.data_ptr(), shift.data_ptr(), s.batch,
                                            s.rows_per_sample, cols, epsilon, s.dt, current_stream(input)),
                 "tt_adaln_forward_seq_first");
    else
        raise_on(tt_adaln_forward(output.data_ptr(), mean.data_ptr<float>(), inv_variance.data_ptr<float>(),
                                  input.data_ptr(), scale.data_ptr(), shift.data_ptr(), s.batch, s.rows_per_sample,
                                  cols, epsilon, s.dt, current_stream(input)),
                 "tt_adaln_forward");
}

void torch_launch_adaln_forward_stats(torch::Tensor &output, const torch::Tensor &input,
                                      const torch::Tensor &scale, const torch::Tensor &shift, int64_t rows,
                                      int64_t cols, double epsilon, torch::Tensor &mean,
                                      torch::Tensor &inv_variance) {
    adaln_forward_stats_impl(output, input, scale, shift, rows, cols, epsilon, mean, inv_variance, false);
}

// input is [rows / batch, batch, cols] (sequence first): sample b owns rows b, b + batch, ...
void torch_launch_adaln_forward_stats_seq_first(torch::Tensor &output, const torch::Tensor &input,
                                                const torch::Tensor &scale, const torch::Tensor &shift, int64_t rows,
                                                int64_t cols, double epsilon, torch::Tensor &mean,
                                                torch::Tensor &inv_variance) {
    adaln_forward_stats_impl(output, input, scale, shift, rows, cols, epsilon, mean, inv_variance, true);
}

static void adaln_backward_impl(torch::Tensor &dinp, torch::Tensor &dscale, torch::Tensor &dshift,
                                const torch::Tensor &dout, const torch::Tensor &saved,
                                const torch::Tensor &scale, const torch::Tensor *mean,
                                const torch::Tensor &inv_variance, int64_t rows, int64_t cols,
                                bool seq_first = false) {
    const auto dev = dout.device();
    for (auto *t : {&dinp, &dscale, &dshift}) check_dense_on(*t, dev, "output tensor");
    for (auto *t : {&dout, &saved, &scale, &inv_variance}) check_dense_on(*t, dev, "input tensor");
    const AdalnShape s = adaln_shape(dout, scale, rows, cols);
    const auto st = dout.scalar_type();
    check_elems(dout, rows * cols, st, "dout");
    check_elems(dinp, rows * cols, st, "dinp");
    check_elems(saved, rows * cols, st, mean ? "input" : "x_norm");
    check_elems(scale, scale.numel(), st, "scale");
    check_elems(dscale, scale.numel(), st, "dscale");
    check_elems(dshift, scale.numel(), st, "dshift");
    check_elems(inv_variance, rows, at::kFloat, "inv_variance");
    if (mean) {
        check_dense_on(*mean, dev, "mean");
        check_elems(*mean, rows, at::kFloat, "mean");
    }
    c10::DeviceGuard guard(dev);
    const size_t need = tt_adaln_backward_workspace_bytes(s.batch, s.rows_per_sample, cols, s.dt);
    TORCH_CHECK(need > 0 || rows == 0, "unsupported AdaLN shape: cols=", cols);
    at::Tensor ws = scratch(need, dout);
    if (mean && seq_first)
        raise_on(tt_adaln_backward_seq_first(dinp.data_ptr(), dscale.data_ptr(), dshift.data_ptr(), dout.data_ptr(),
                                             saved.data_ptr(), scale.data_ptr(), mean->data_ptr<float>(),
                                             inv_variance.data_ptr<float>(), s.batch, s.rows_per_sample, cols, s.dt,
                                             ws.data_ptr(), need, current_stream(dout)),
                 "tt_adaln_backward_seq_first");
    else if (mean)
        raise_on(tt_adaln_backward(dinp.data_ptr(), dscale.data_ptr(), dshift.data_ptr(), dout.data_ptr(),
                                   saved.data_ptr(), scale.data_ptr(), mean->data_ptr<float>(),
                                   inv_variance.data_ptr<float>(), s.batch, s.rows_per_sample, cols, s.dt,
                                   ws.data_ptr(), need, current_stream(dout)),
                 "tt_adaln_backward");
    else
        raise_on(tt_adaln_backward_from_xnorm(dinp.data_ptr(), dscale.data_ptr(), dshift.data_ptr(),
                                              dout.data_ptr(), saved.data_ptr(), scale.data_ptr(),
                                              inv_variance.data_ptr<float>(), s.batch, s.rows_per_sample, cols,
                                              s.dt, ws.data_ptr(), need, current_stream(dout)),
                 "tt_adaln_backward_from_xnorm");
}

// Reference contract: x_norm is what torch_launch_adaln_forward wrote to `x_norm`.
void torch_launch_adaln_backward(torch::Tensor &dinp, torch::Tensor &dscale, torch::Tensor &dshift,
                                 const torch::Tensor &dout, const torch::Tensor &x_norm,
                                 const torch::Tensor &scale, const torch::Tensor &inv_variance, int64_t rows,
                                 int64_t cols) {
    adaln_backward_impl(dinp, dscale, dshift, dout, x_norm, scale, nullptr, inv_variance, rows, cols);
}

// Native contract: `input`, `mean`, `inv_variance` as seen / written by torch_launch_adaln_forward_stats.
void torch_launch_adaln_backward_x(torch::Tensor &dinp, torch::Tensor &dscale, torch::Tensor &dshift,
                                   const torch::Tensor &dout, const torch::Tensor &input,
                                   const torch::Tensor &scale, const torch::Tensor &mean,
                                   const torch::Tensor &inv_variance, int64_t rows, int64_t cols) {
    adaln_backward_impl(dinp, dscale, dshift, dout, input, scale, &mean, inv_variance, rows, cols);
}

void torch_launch_adaln_backward_x_seq_first(torch::Tensor &dinp, torch::Tensor &dscale, torch::Tensor &dshift,
                                             const torch::Tensor &dout, const torch::Tensor &input,
                                             const torch::Tensor &scale, const torch::Tensor &mean,
                                             const torch::Tensor &inv_variance, int64_t rows, int64_t cols) {
    adaln_backward_impl(dinp, dscale, dshift, dout, input, scale, &mean, inv_variance, rows, cols, true);
}

// Native backward for an input with another consumer: `dres` is the gradient the input receives from it,
// dinp = dx of the norm + dres.  No counterpart in the reference's module.
void torch_launch_adaln_backward_residual(torch::Tensor &dinp, torch::Tensor &dscale, torch::Tensor &dshift,
                                          const torch::Tensor &dout, const torch::Tensor &dres,
                                          const torch::Tensor &input, const torch::Tensor &scale,
                                          const torch::Tensor &mean, const torch::Tensor &inv_variance,
                                          int64_t rows, int64_t cols) {
    const auto dev = dout.device();
    for (auto *t : {&dinp, &dscale, &dshift}) check_dense_on(*t, dev, "output tensor");
    for (auto *t : {&dout, &dres, &input, &scale, &mean, &inv_variance}) check_dense_on(*t, dev, "input tensor");
    const AdalnShape s = adaln_shape(dout, scale, rows, cols);
    const auto st = dout.scalar_type();
    for (auto *t : {&dout, &dres, &input}) check_elems(*t, rows * cols, st, "dout/dres/input");
    check_elems(dinp, rows * cols, st, "dinp");
    check_elems(scale, scale.numel(), st, "scale");
    for (auto *t : {&dscale, &dshift}) check_elems(*t, scale.numel(), st, "dscale/dshift");
    check_elems(mean, rows, at::kFloat, "mean");
    check_elems(inv_variance, rows, at::kFloat, "inv_variance");
    c10::DeviceGuard guard(dev);
    const size_t need = tt_adaln_backward_workspace_bytes(s.batch, s.rows_per_sample, cols, s.dt);
    TORCH_CHECK(need > 0 || rows == 0, "unsupported AdaLN shape: cols=", cols);
    at::Tensor ws = scratch(need, dout);
    raise_on(tt_adaln_backward_residual(dinp.data_ptr(), dscale.data_ptr(), dshift.data_ptr(), dout.data_ptr(),
                                        dres.data_ptr(), input.data_ptr(), scale.data_ptr(),
                                        mean.data_ptr<float>(), inv_variance.data_ptr<float>(), s.batch,
                                        s.rows_per_sample, cols, s.dt, ws.data_ptr(), need, current_stream(dout)),
             "tt_adaln_backward_residual");
}

// Gated residual update fused with the norm that follows it:
// h2 = input + attn * gate[b];  output = AdaLN(h2).  No counterpart in the reference's module.
void torch_launch_gated_adaln_forward(torch::Tensor &h2, torch::Tensor &output, const torch::Tensor &input,
                                      const torch::Tensor &attn, const torch::Tensor &gate,
                                      const torch::Tensor &scale, const torch::Tensor &shift, int64_t rows,
                                      int64_t cols, double epsilon, torch::Tensor &mean,
                                      torch::Tensor &inv_variance) {
    const auto dev = input.device();
    for (auto *t : {&h2, &output, &mean, &inv_variance}) check_dense_on(*t, dev, "output tensor");
    for (auto *t : {&input, &attn, &gate, &scale, &shift}) check_dense_on(*t, dev, "input tensor");
    const AdalnShape s = adaln_shape(input, scale, rows, cols);
    const auto st = input.scalar_type();
    for (auto *t : {&input, &attn}) check_elems(*t, rows * cols, st, "input/attn");
    check_elems(h2, rows * cols, st, "h2");
    check_elems(output, rows * cols, st, "output");
    for (auto *t : {&gate, &scale, &shift}) check_elems(*t, scale.numel(), st, "gate/scale/shift");
    check_elems(mean, rows, at::kFloat, "mean");
    check_elems(inv_variance, rows, at::kFloat, "inv_variance");
    c10::DeviceGuard guard(dev);
    raise_on(tt_gated_residual_adaln_forward(h2.data_ptr(), output.data_ptr(), mean.data_ptr<float>(),
                                             inv_variance.data_ptr<float>(), input.data_ptr(), attn.data_ptr(),
                                             gate.data_ptr(), scale.data_ptr(), shift.data_ptr(), s.batch,
                                             s.rows_per_sample, cols, epsilon, s.dt, current_stream(input)),
             "tt_gated_residual_adaln_forward");
}

// dh2: gradient reaching h2 from its other uses, or None.
void torch_launch_gated_adaln_backward(torch::Tensor &dinp, torch::Tensor &dattn, torch::Tensor &dgate,
                                       torch::Tensor &dscale, torch::Tensor &dshift, const torch::Tensor &dout,
                                       const c10::optional<torch::Tensor> &dh2, const torch::Tensor &h2,
                                       const torch::Tensor &attn, const torch::Tensor &gate,
                                       const torch::Tensor &scale, const torch::Tensor &mean,
                                       const torch::Tensor &inv_variance, int64_t rows, int64_t cols) {
    const auto dev = dout.device();
    for (auto *t : {&dinp, &dattn, &dgate, &dscale, &dshift}) check_dense_on(*t, dev, "output tensor");
    for (auto *t : {&dout, &h2, &attn, &gate, &scale, &mean, &inv_variance}) check_dense_on(*t, dev, "input tensor");
    const AdalnShape s = adaln_shape(dout, scale, rows, cols);
    const auto st = dout.scalar_type();
    for (auto *t : {&dout, &h2, &attn}) check_elems(*t, rows * cols, st, "dout/h2/attn");
    for (auto *t : {&dinp, &dattn}) check_elems(*t, rows * cols, st, "dinp/dattn");
    for (auto *t : {&gate, &scale}) check_elems(*t, scale.numel(), st, "gate/scale");
    for (auto *t : {&dgate, &dscale, &dshift}) check_elems(*t, scale.numel(), st, "dgate/dscale/dshift");
    check_elems(mean, rows, at::kFloat, "mean");
    check_elems(inv_variance, rows, at::kFloat, "inv_variance");
    const void *dh2_ptr = nullptr;
    if (dh2.has_value() && dh2->defined()) {
        check_dense_on(*dh2, dev, "dh2");
        check_elems(*dh2, rows * cols, st, "dh2");
        dh2_ptr = dh2->data_ptr();
    }
    c10::DeviceGuard guard(dev);
    const size_t need = tt_gated_residual_adaln_backward_workspace_bytes(s.batch, s.rows_per_sample, cols, s.dt);
    TORCH_CHECK(need > 0 || rows == 0, "unsupported gated AdaLN shape: cols=", cols);
    at::Tensor ws = scratch(need, dout);
    raise_on(tt_gated_residual_adaln_backward(dinp.data_ptr(), dattn.data_ptr(), dgate.data_ptr(),
                                              dscale.data_ptr(), dshift.data_ptr(), dout.data_ptr(), dh2_ptr,
                                              h2.data_ptr(), attn.data_ptr(), gate.data_ptr(), scale.data_ptr(),
                                              mean.data_ptr<float>(), inv_variance.data_ptr<float>(), s.batch,
                                              s.rows_per_sample, cols, s.dt, ws.data_ptr(), need,
                                              current_stream(dout)),
             "tt_gated_residual_adaln_backward");
}

// ---- whole calls (see torch_glue.h) ----

using Tensors = std::vector<torch::Tensor>;

// Modulation rows of [B, cols] (or one row) that belong to x as it lies.
static bool ready_modulation(const torch::Tensor &x, const torch::Tensor &scale, int64_t cols, bool seq_first) {
    if (scale.numel() == 0 || scale.numel() % cols != 0) return false;
    const int64_t batch = scale.numel() / cols;
    if (seq_first) return x.dim() == 3 && x.size(1) == batch;
    return batch == 1 || (x.dim() >= 2 && x.size(0) == batch);
}

static bool adaln_ready(const torch::Tensor &x, const torch::Tensor &scale, const torch::Tensor &shift, int64_t cols,
                        bool seq_first) {
    return ready_rows(x, cols) && ready(scale, x) && ready(shift, x) && shift.numel() == scale.numel() &&
           ready_modulation(x, scale, cols, seq_first);
}

// out, mean, inv_variance of ready operands
static Tensors adaln_run(const torch::Tensor &x, const torch::Tensor &scale, const torch::Tensor &shift, int64_t cols,
                         double epsilon, bool seq_first) {
    const int64_t rows = x.numel() / cols;
    torch::Tensor out = at::empty_like(x), mean = row_statistics(x, rows), inv_variance = row_statistics(x, rows);
    adaln_forward_stats_impl(out, x, scale, shift, rows, cols, epsilon, mean, inv_variance, seq_first);
    return {out, mean, inv_variance};
}

static c10::optional<Tensors> adaln_forward(const torch::Tensor &x, const torch::Tensor &scale, const torch::Tensor &shift,
                                            int64_t cols, double epsilon, bool seq_first) {
    if (!adaln_ready(x, scale, shift, cols, seq_first)) return c10::nullopt;
    return adaln_run(x, scale, shift, cols, epsilon, seq_first);
}

// dinp, dscale, dshift; dres is the gradient the input receives from its other consumer, or None
static c10::optional<Tensors> adaln_backward(const torch::Tensor &dout, const c10::optional<torch::Tensor> &dres,
                                             const torch::Tensor &x, const torch::Tensor &scale, const torch::Tensor &mean,
                                             const torch::Tensor &inv_variance, int64_t cols, bool seq_first) {
    const bool residual = dres.has_value() && dres->defined();
    if (!ready(dout, x) || (residual && !ready(*dres, x))) return c10::nullopt;
    const int64_t rows = x.numel() / cols;
    torch::Tensor dinp = at::empty_like(x), dscale = at::empty_like(scale), dshift = at::empty_like(scale);
    if (residual)
        torch_launch_adaln_backward_residual(dinp, dscale, dshift, dout, *dres, x, scale, mean, inv_variance, rows, cols);
    else
        adaln_backward_impl(dinp, dscale, dshift, dout, x, scale, &mean, inv_variance, rows, cols, seq_first);
    return Tensors{dinp, dscale, dshift};
}

static bool gated_ready(const torch::Tensor &h, const torch::Tensor &attn, const torch::Tensor &gate,
                        const torch::Tensor &scale, const torch::Tensor &shift) {
    if (h.dim() < 1 || !ready_rows(h, h.size(-1)) || !ready(attn, h) || attn.sizes() != h.sizes()) return false;
    for (auto *t : {&gate, &scale, &shift})
        if (!ready(*t, h) || t->numel() != scale.numel()) return false;
    // backward shapes the gradients after gate and scale, the rows it keeps: shift's is scale's
    return shift.sizes() == scale.sizes() && ready_modulation(h, scale, h.size(-1), false);
}

// h2, out, mean, inv_variance of ready operands
static Tensors gated_run(const torch::Tensor &h, const torch::Tensor &attn, const torch::Tensor &gate,
                         const torch::Tensor &scale, const torch::Tensor &shift, double epsilon) {
    const int64_t cols = h.size(-1), rows = h.numel() / cols;
    torch::Tensor h2 = at::empty_like(h), out = at::empty_like(h);
    torch::Tensor mean = row_statistics(h, rows), inv_variance = row_statistics(h, rows);
    torch_launch_gated_adaln_forward(h2, out, h, attn, gate, scale, shift, rows, cols, epsilon, mean, inv_variance);
    return {h2, out, mean, inv_variance};
}

static c10::optional<Tensors> gated_forward(const torch::Tensor &h, const torch::Tensor &attn, const torch::Tensor &gate,
                                            const torch::Tensor &scale, const torch::Tensor &shift, double epsilon) {
    if (!gated_ready(h, attn, gate, scale, shift)) return c10::nullopt;
    return gated_run(h, attn, gate, scale, shift, epsilon);
}

// dh, dattn, dgate, dscale, dshift; dh2 may be None
static c10::optional<Tensors> gated_backward(const torch::Tensor &dout, const c10::optional<torch::Tensor> &dh2,
                                             const torch::Tensor &h2, const torch::Tensor &attn, const torch::Tensor &gate,
                                             const torch::Tensor &scale, const torch::Tensor &mean,
                                             const torch::Tensor &inv_variance, int64_t cols) {
    if (!ready(dout, h2) || (dh2.has_value() && dh2->defined() && !ready(*dh2, h2))) return c10::nullopt;
    torch::Tensor dh = at::empty_like(h2), dattn = at::empty_like(h2);
    torch::Tensor dgate = at::empty_like(gate), dscale = at::empty_like(scale), dshift = at::empty_like(scale);
    torch_launch_gated_adaln_backward(dh, dattn, dgate, dscale, dshift, dout, dh2, h2, attn, gate, scale, mean, inv_variance,
                                      h2.numel() / cols, cols);
    return Tensors{dh, dattn, dgate, dscale, dshift};
}

// ---- call sites (see torch_glue.h): AdaLNModelFunction, AdaLNResidualFunction and GatedResidualAdaLNFunction ----

using torch::autograd::AutogradContext;
using torch::autograd::Function;

// adaln_backward returns both modulation gradients in scale's shape; a shift that came in another shape of as many
// elements gets its gradient in its own.
static void keep_shift_shape(AutogradContext *ctx, const torch::Tensor &scale, const torch::Tensor &shift) {
    if (shift.sizes() != scale.sizes()) ctx->saved_data["shift_shape"] = shift.sizes().vec();
}

static torch::Tensor in_shift_shape(AutogradContext *ctx, const torch::Tensor &dshift) {
    const auto kept = ctx->saved_data.find("shift_shape");
    return kept == ctx->saved_data.end() ? dshift : dshift.view(kept->second.toIntVector());
}

struct AdalnSite : Function<AdalnSite> {
    static torch::Tensor forward(AutogradContext *ctx, const torch::Tensor &x, const torch::Tensor &scale,
                                 const torch::Tensor &shift, int64_t cols, double epsilon, bool seq_first) {
        Tensors done = adaln_run(x, scale, shift, cols, epsilon, seq_first);
        ctx->save_for_backward({x, scale, done[1], done[2]});
        ctx->saved_data["cols"] = cols;
        ctx->saved_data["seq_first"] = seq_first;
        keep_shift_shape(ctx, scale, shift);
        return done[0];
    }
    static Tensors backward(AutogradContext *ctx, Tensors grads) {
        const Tensors kept = ctx->get_saved_variables();
        Tensors d = taken(adaln_backward(prepared(grads[0], kept[0]), c10::nullopt, kept[0], kept[1], kept[2], kept[3],
                                    ctx->saved_data["cols"].toInt(), ctx->saved_data["seq_first"].toBool()), "adaln_backward");
        return first_order({d[0], d[1], in_shift_shape(ctx, d[2]), {}, {}, {}}, kept, grads);
    }
};

struct AdalnResidualSite : Function<AdalnResidualSite> {
    static Tensors forward(AutogradContext *ctx, const torch::Tensor &x, const torch::Tensor &scale, const torch::Tensor &shift,
                           double epsilon) {
        Tensors done = adaln_run(x, scale, shift, x.size(-1), epsilon, false);
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({x, scale, done[1], done[2]});
        keep_shift_shape(ctx, scale, shift);
        return {x, done[0]};
    }
    static Tensors backward(AutogradContext *ctx, Tensors grads) {
        const Tensors kept = ctx->get_saved_variables();
        if (!grads[1].defined()) return {grads[0], {}, {}, {}};  // only the stream was used: the function was an identity
        Tensors d = taken(adaln_backward(prepared(grads[1], kept[0]), prepared(grads[0], kept[0]), kept[0], kept[1], kept[2], kept[3],
                                    kept[0].size(-1), false), "adaln_backward");
        return first_order({d[0], d[1], in_shift_shape(ctx, d[2]), {}}, kept, grads);
    }
};

struct GatedResidualSite : Function<GatedResidualSite> {
    static Tensors forward(AutogradContext *ctx, const torch::Tensor &h, const torch::Tensor &attn, const torch::Tensor &gate,
                           const torch::Tensor &scale, const torch::Tensor &shift, double epsilon) {
        Tensors done = gated_run(h, attn, gate, scale, shift, epsilon);
        ctx->set_materialize_grads(false);  // an unused h2 costs no zero tensor and no read
        ctx->save_for_backward({done[0], attn, gate, scale, done[2], done[3]});
        return {done[0], done[1]};
    }
    static Tensors backward(AutogradContext *ctx, Tensors grads) {
        const Tensors kept = ctx->get_saved_variables();
        const torch::Tensor dout = grads[1].defined() ? prepared(grads[1], kept[0]) : at::zeros_like(kept[0]);
        Tensors d = taken(gated_backward(dout, prepared(grads[0], kept[0]), kept[0], kept[1], kept[2], kept[3], kept[4], kept[5],
                                    kept[0].size(-1)), "gated_backward");
        return first_order({d[0], d[1], d[2], d[3], d[4], {}}, kept, grads);
    }
};

static c10::optional<torch::Tensor> adaln_site(const torch::Tensor &x, const torch::Tensor &scale, const torch::Tensor &shift,
                                               int64_t cols, double epsilon, bool seq_first) {
    if (!ordinary_call({&x, &scale, &shift}) || !adaln_ready(x, scale, shift, cols, seq_first)) return c10::nullopt;
    return AdalnSite::apply(x, scale, shift, cols, epsilon, seq_first);
}

using Pair = std::tuple<torch::Tensor, torch::Tensor>;

static c10::optional<Pair> adaln_residual_site(const torch::Tensor &x, const torch::Tensor &scale, const torch::Tensor &shift,
                                               double epsilon) {
    if (!ordinary_call({&x, &scale, &shift}) || x.dim() < 1 || !adaln_ready(x, scale, shift, x.size(-1), false))
        return c10::nullopt;
    Tensors outs = AdalnResidualSite::apply(x, scale, shift, epsilon);
    return Pair{outs[0], outs[1]};
}

static c10::optional<Pair> gated_residual_site(const torch::Tensor &h, const torch::Tensor &attn, const torch::Tensor &gate,
                                               const torch::Tensor &scale, const torch::Tensor &shift, double epsilon) {
    if (!ordinary_call({&h, &attn, &gate, &scale, &shift}) || !gated_ready(h, attn, gate, scale, shift)) return c10::nullopt;
    Tensors outs = GatedResidualSite::apply(h, attn, gate, scale, shift, epsilon);
    return Pair{outs[0], outs[1]};
}

PYBIND11_MODULE(fused_adaln, m) {
    m.def("adaln_site", &adaln_site, "AdaLNModelFunction as a native autograd node; None unless every operand is ready");
    m.def("adaln_residual_site", &adaln_residual_site, "AdaLNResidualFunction as a native autograd node; or None");
    m.def("gated_residual_site", &gated_residual_site, "GatedResidualAdaLNFunction as a native autograd node; or None");
    m.def("adaln_forward", &adaln_forward, "AdaLN forward: out, mean, inv_variance; None unless every operand is ready");
    m.def("adaln_backward", &adaln_backward, "AdaLN backward: dinp, dscale, dshift; None unless every operand is ready");
    m.def("gated_forward", &gated_forward, "gated residual update + AdaLN: h2, out, mean, inv_variance; or None");
    m.def("gated_backward", &gated_backward, "its backward: dh, dattn, dgate, dscale, dshift; or None");
    m.def("torch_launch_adaln_backward_residual", &torch_launch_adaln_backward_residual,
          "AdaLN backward kernel with the input's other gradient added in");
    m.def("torch_launch_gated_adaln_forward", &torch_launch_gated_adaln_forward,
          "gated residual update + AdaLN forward kernel");
    m.def("torch_launch_gated_adaln_backward", &torch_launch_gated_adaln_backward,
          "gated residual update + AdaLN backward kernel");
    m.def("torch_launch_adaln_forward", &torch_launch_adaln_forward, "AdaLN forward kernel");
    m.def("torch_launch_adaln_backward", &torch_launch_adaln_backward,
          "AdaLN backward kernel (from the saved normalised rows)");
    m.def("torch_launch_adaln_forward_stats", &torch_launch_adaln_forward_stats,
          "AdaLN forward kernel that saves mean and inv_variance instead of x_norm");
    m.def("torch_launch_adaln_backward_x", &torch_launch_adaln_backward_x,
          "AdaLN backward kernel (from the saved input and statistics)");
    m.def("torch_launch_adaln_forward_stats_seq_first", &torch_launch_adaln_forward_stats_seq_first,
          "AdaLN forward kernel on sequence-first rows [S, B, C]");
    m.def("torch_launch_adaln_backward_x_seq_first", &torch_launch_adaln_backward_x_seq_first,
          "AdaLN backward kernel on sequence-first rows [S, B, C]");
    m.def("supported", [](int64_t cols, const torch::Tensor &like) {
        return tt_norm_supported(cols, like.scalar_type() == at::kBFloat16 ? TT_NORM_BF16
                                       : like.scalar_type() == at::kFloat  ? TT_NORM_F32
                                       : like.scalar_type() == at::kHalf   ? TT_NORM_F16 : -1) != 0;
    }, "whether the kernels are built for this column count and dtype");
}

// Same operator namespace as the reference registers (adaln_ops.cpp:62-65).
TORCH_LIBRARY(layernorm_block_smem, m) {
    m.def("torch_launch_adaln_forward(Tensor(a!) output, Tensor(b!) x_norm, Tensor input, Tensor scale, "
          "Tensor shift, int rows, int cols, float epsilon, Tensor(c!) inv_variance) -> ()",
          &torch_launch_adaln_forward);
    m.def("torch_launch_adaln_backward(Tensor(a!) dinp, Tensor(b!) dscale, Tensor(c!) dshift, Tensor dout, "
          "Tensor x_norm, Tensor scale, Tensor inv_variance, int rows, int cols) -> ()",
          &torch_launch_adaln_backward);
}
