// The host path of the ops whose kernels take a few microseconds: argument checks, output and scratch allocation, the call
// of the library and the autograd node, in C++.  A small layer's training step spent most of its time in the interpreter
// (linear over 96 tokens, 64 -> 128, forward and gradients: 137 us behind 38 us of kernels; the torch node of the same
// shape 85 us): an op was a Python autograd function, whose backward the engine's thread enters the interpreter for, around
// ctypes calls of 9 us.  What each op computes is unchanged: the formulas of the gradients and the order of the checks
// are those of pam_amd/cuda_bindings.py and of the entry points in include/pam_hip.h.
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <map>
#include <mutex>
#include <sstream>
#include <string>
#include <utility>
#include <vector>

#include "../../include/pam_hip.h"
#include "../../include/pam_hip_extra.h"

// what this module was built on (pam_amd/build.py reads it from the file's bytes)
extern "C" __attribute__((used, visibility("default"))) const char pam_host_build[] = "pam_host_build=" PAM_HOST_BUILD;

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---------------------------------------------------------------- checks, streams, scratch

void check_tensor(const Tensor& t)
{
    TORCH_CHECK(t.is_cuda(), "argument must be a CUDA tensor");                 // CHECK_CUDA, pam/cuda_kernels.cu:8
    TORCH_CHECK_TYPE(t.scalar_type() == at::kFloat, "PAM kernels compute in float32, got torch.", c10::getDtypeNames(t.scalar_type()).first);
}

// a tensor's shape as Python prints it
std::string shape(const Tensor& t)
{
    std::ostringstream text;
    text << '(';
    for (int64_t i = 0; i < t.dim(); ++i) text << (i ? ", " : "") << t.size(i);
    text << (t.dim() == 1 ? ",)" : ")");
    return text.str();
}

void check_call(int rc, const char* name)
{
    if (rc == PAM_HIP_OK) return;
    TORCH_CHECK_VALUE(rc != PAM_HIP_ERR_ARGUMENT, "pam_hip_", name, " failed (", rc, "): ", pam_hip_last_error());
    TORCH_CHECK(false, "pam_hip_", name, " failed (", rc, "): ", pam_hip_last_error());
}

struct OnDevice {                         // the tensor's device made current, and its current stream
    c10::hip::HIPGuardMasqueradingAsCUDA guard;
    void* stream;
    explicit OnDevice(const Tensor& t) : guard(t.device()), stream((void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream()) {}
};

float* data(const Tensor& t) { return t.data_ptr<float>(); }
float* data_or_null(const Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; }

Tensor new_floats(at::IntArrayRef shape, const Tensor& like) { return at::empty(shape, like.options().dtype(at::kFloat).memory_format(c10::nullopt).requires_grad(false)); }

// The matrix products' scratch (pieces of cut tiles, their arrival words): one buffer per device and stream, kept and
// grown as needed.  Products on one stream run one after the other, and each leaves the arrival words ready for the
// next one; products on different streams may overlap in time and must not share a buffer.  The lock covers the table
// only: buffers are allocated and given back outside it, since the allocator may wait for the device or for the
// interpreter (its hooks), which another thread that waits for the lock might hold.  While the stream is captured a buffer
// is the graph's own, given back to the graph's memory at once: graphs recorded on one stream may be replayed side by side.
Tensor gemm_workspace(const Tensor& like, void* stream, size_t bytes)
{
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing((hipStream_t)stream, &capturing) == hipSuccess && capturing != hipStreamCaptureStatusNone)
        return new_floats({(int64_t)(bytes / 4 + 64)}, like);
    static std::mutex lock;
    static auto* kept = new std::map<std::pair<int, void*>, Tensor>;           // (not destroyed after the allocator at exit)
    const std::pair<int, void*> key{like.device().index(), stream};
    const auto fits = [&](const Tensor& t) { return t.defined() && (size_t)t.numel() * 4 >= bytes; };
    {
        std::lock_guard<std::mutex> hold(lock);
        const auto at = kept->find(key);
        if (at != kept->end() && fits(at->second)) return at->second;
    }
    Tensor ws = new_floats({(int64_t)(std::max(bytes, (size_t)1 << 20) / 4 + 64)}, like);
    std::lock_guard<std::mutex> hold(lock);
    Tensor& entry = (*kept)[key];
    if (!fits(entry)) std::swap(entry, ws);          // (ws, the smaller one or a second one, goes after the lock has)
    return entry;
}

// ---------------------------------------------------------------- products

// (the last dim is contiguous, or the one before it, or a contiguous copy: pam/cuda_bindings.py:106-115)
Tensor row_major(const Tensor& t, int64_t dims)
{
    TORCH_CHECK_VALUE(t.dim() == dims, "tensor.dim()=", t.dim(), " is not equal to target_dim=", dims);
    return t.stride(-1) == 1 || t.stride(-2) == 1 ? t : t.contiguous();
}

enum Kind { kPam = 0, kStandard = 1, kSlope = 2 };

// L (x) R: PAM products (bias: one value per column, added to the finished sums), ordinary ones, or the exact gradient's,
// where `other` is the forward operand whose gradient is wanted and delta_left says which operand is the upstream gradient
Tensor product(int kind, const Tensor& L, const Tensor& R, const Tensor& other, bool delta_left, const Tensor& bias, double offset)
{
    check_tensor(L); check_tensor(R);
    if (other.defined()) check_tensor(other);
    if (bias.defined()) check_tensor(bias);
    const bool batched = L.dim() == 3;
    static const char* const names[2][3] = {{"pam_matmul_fwd", "standard_matmul", "pam_matmul_bwd"}, {"pam_bmm_fwd", "standard_bmm", "pam_bmm_bwd"}};
    const char* name = bias.defined() ? "linear_fwd" : names[batched][kind];
    TORCH_CHECK_TYPE(kind != kSlope || other.defined(), name, ": the forward operand is missing");
    const int64_t nd = batched ? 3 : 2;
    TORCH_CHECK_VALUE(L.dim() == nd && R.dim() == nd && (!other.defined() || other.dim() == nd), name, ": expected ", nd, "-D operands");
    const int64_t batch = batched ? L.size(0) : 1, m = L.size(-2), k = L.size(-1), n = R.size(-1);
    TORCH_CHECK_VALUE(k == R.size(-2) && (!batched || batch == R.size(0)), name, ": shapes ", shape(L), " and ", shape(R), " do not multiply");
    TORCH_CHECK_VALUE(!other.defined() || (other.size(-2) == m && other.size(-1) == n), name, ": third operand must have the shape of the result");
    TORCH_CHECK_VALUE(!bias.defined() || (bias.numel() == n && bias.is_contiguous()), "linear_fwd: bias must be contiguous with one value per output column");
    const OnDevice on(L);
    Tensor out = batched ? new_floats({batch, m, n}, L) : new_floats({m, n}, L);
    if (out.numel() == 0) return out;
    const size_t bytes = pam_hip_gemm_workspace_bytes(batch, m, n, k);
    Tensor ws;
    if (bytes) ws = gemm_workspace(L, on.stream, bytes);
    void* scratch = data_or_null(ws);
    const float off = (float)offset;
    int rc;
    if (batched) {
#define PAM_MAT(t) data(t), t.stride(0), t.stride(1), t.stride(2)
        if (kind == kPam) rc = pam_hip_pam_bmm_fwd(PAM_MAT(L), PAM_MAT(R), PAM_MAT(out), batch, m, n, k, off, scratch, bytes, on.stream);
        else if (kind == kStandard) rc = pam_hip_standard_bmm(PAM_MAT(L), PAM_MAT(R), PAM_MAT(out), batch, m, n, k, off, scratch, bytes, on.stream);
        else rc = pam_hip_pam_bmm_bwd(PAM_MAT(L), PAM_MAT(R), PAM_MAT(other), PAM_MAT(out), batch, m, n, k, delta_left, off, scratch, bytes, on.stream);
#undef PAM_MAT
    } else {
#define PAM_MAT(t) data(t), t.stride(0), t.stride(1)
        if (kind == kPam && bias.defined()) rc = pam_hip_pam_linear_fwd(PAM_MAT(L), PAM_MAT(R), data(bias), PAM_MAT(out), m, n, k, off, scratch, bytes, on.stream);
        else if (kind == kPam) rc = pam_hip_pam_matmul_fwd(PAM_MAT(L), PAM_MAT(R), PAM_MAT(out), m, n, k, off, scratch, bytes, on.stream);
        else if (kind == kStandard) rc = pam_hip_standard_matmul(PAM_MAT(L), PAM_MAT(R), PAM_MAT(out), m, n, k, off, scratch, bytes, on.stream);
        else rc = pam_hip_pam_matmul_bwd(PAM_MAT(L), PAM_MAT(R), PAM_MAT(other), PAM_MAT(out), m, n, k, delta_left, off, scratch, bytes, on.stream);
#undef PAM_MAT
    }
    check_call(rc, bias.defined() ? "pam_linear_fwd" : name);
    return out;
}

// ---------------------------------------------------------------- sums over rows

// Whether the sum over the rows of t runs on the kernel: not where autograd is to record it (a gradient's gradient).
bool summable(const Tensor& t)
{
    return t.is_cuda() && t.scalar_type() == at::kFloat && t.dim() == 2 && t.stride(1) == 1 && t.numel() > 0
        && !(t.requires_grad() && at::GradMode::is_enabled());
}

// the sums over the rows of one matrix, or of two of one shape
std::pair<Tensor, Tensor> column_sums(const Tensor& a, const Tensor& b)
{
    check_tensor(a);
    TORCH_CHECK_VALUE(a.dim() == 2 && (a.stride(1) == 1 || a.size(1) <= 1), "column_sums: expected a matrix whose rows are contiguous");
    if (b.defined()) {
        check_tensor(b);
        TORCH_CHECK_VALUE(b.sizes() == a.sizes() && b.device() == a.device() && (b.stride(1) == 1 || b.size(1) <= 1),
                          "column_sums: the second matrix must have the first one's shape and device, and contiguous rows");
    }
    const OnDevice on(a);
    const int64_t rows = a.size(0), n = a.size(1);
    Tensor a_sums = new_floats({n}, a), b_sums, ws;
    if (b.defined()) b_sums = new_floats({n}, a);
    const size_t bytes = pam_hip_column_sums_workspace_bytes(rows, n, b.defined() ? 2 : 1);
    if (bytes) ws = new_floats({(int64_t)(bytes / 4)}, a);
    check_call(pam_hip_column_sums(data(a), a.stride(0), data(a_sums), data_or_null(b), b.defined() ? b.stride(0) : 0, data_or_null(b_sums),
                                   rows, n, data_or_null(ws), bytes, on.stream), "column_sums");
    return {a_sums, b_sums};
}

Tensor sum_rows(const Tensor& t) { return summable(t) ? column_sums(t, Tensor()).first : t.sum(0); }

// What `approx_bwd` asks for, per operand of the products (first, second) and for exp and log: the approximate gradient or
// the exact one.
struct Approx {
    bool a, b, e;
    void save(AutogradContext* ctx) const { ctx->saved_data["a"] = a; ctx->saved_data["b"] = b; ctx->saved_data["e"] = e; }
    static Approx saved(AutogradContext* ctx)
    {
        return Approx{ctx->saved_data["a"].toBool(), ctx->saved_data["b"].toBool(), ctx->saved_data["e"].toBool()};
    }
};

// dA = dY (x) B^T and dB = A^T (x) dY of Y = A (x) B; the exact variant weighs each product by the slope of the forward
// operand's affine piece instead of multiplying (pam/cuda_bindings.py:132-166)
struct ProductGrads { Tensor dA, dB; };
ProductGrads product_grads(const Tensor& A, const Tensor& B, const Tensor& dY, int64_t dims, const Approx& f, double off, bool need_A, bool need_B)
{
    ProductGrads g;
    if (need_A) {
        const Tensor Bt = row_major(B.mT(), dims);
        g.dA = f.a ? product(kPam, dY, Bt, Tensor(), false, Tensor(), off) : product(kSlope, dY, Bt, A, true, Tensor(), off);
    }
    if (need_B) {
        const Tensor At = row_major(A.mT(), dims);
        g.dB = f.b ? product(kPam, At, dY, Tensor(), false, Tensor(), off) : product(kSlope, At, dY, B, false, Tensor(), off);
    }
    return g;
}

struct MatmulNode : torch::autograd::Function<MatmulNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& A_in, const Tensor& B_in, int64_t dims, double offset, bool a, bool b)
    {
        const Tensor A = row_major(A_in, dims), B = row_major(B_in, dims);
        ctx->saved_data["dims"] = dims; ctx->saved_data["offset"] = offset;
        Approx{a, b, false}.save(ctx);
        ctx->save_for_backward({A, B});
        return product(kPam, A, B, Tensor(), false, Tensor(), offset);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const Approx f = Approx::saved(ctx);
        const int64_t dims = ctx->saved_data["dims"].toInt();
        const at::AutoGradMode no_graph(false);
        const ProductGrads g = product_grads(saved[0], saved[1], row_major(grads[0], dims), dims, f, ctx->saved_data["offset"].toDouble(),
                                             ctx->needs_input_grad(0), ctx->needs_input_grad(1));
        return {g.dA, g.dB, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// X W^T + bias in one kernel; the gradient of the bias is the sum of the upstream gradient over the rows
struct LinearNode : torch::autograd::Function<LinearNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& X_in, const Tensor& W, const Tensor& bias, double offset, bool a, bool b)
    {
        const Tensor X = row_major(X_in, 2), Wt = row_major(W.t(), 2);
        ctx->saved_data["offset"] = offset;
        Approx{a, b, false}.save(ctx);
        ctx->save_for_backward({X, Wt});
        return product(kPam, X, Wt, Tensor(), false, bias.contiguous(), offset);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const Approx f = Approx::saved(ctx);
        const Tensor dY = row_major(grads[0], 2);
        ProductGrads g;
        {
            const at::AutoGradMode no_graph(false);
            g = product_grads(saved[0], saved[1], dY, 2, f, ctx->saved_data["offset"].toDouble(), ctx->needs_input_grad(0), ctx->needs_input_grad(1));
            if (g.dB.defined()) g.dB = g.dB.t();
        }
        return {g.dA, g.dB, ctx->needs_input_grad(2) ? sum_rows(dY) : Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// A saved tensor as a backward pass reads it.  It comes back through the program's saved-tensor hooks, which may return any
// tensor for it: another type, device or shape is refused, and other strides are copied.
Tensor whole(const Tensor& saved, const Tensor& grad, at::IntArrayRef sizes, const char* name)
{
    check_tensor(saved);
    TORCH_CHECK_VALUE(saved.sizes() == sizes && saved.device() == grad.device(), name, ": a saved tensor has not the shape or the device that it was saved with");
    return saved.contiguous();
}

// ---------------------------------------------------------------- rows

// softmax over the last dimension of a contiguous tensor; the gradient is the chain of the primitives' gradients
// (pam/cuda_bindings.py:43-57, 78-97, 224-239)
struct SoftmaxNode : torch::autograd::Function<SoftmaxNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, double offset, bool a, bool b, bool e)
    {
        check_tensor(x);
        TORCH_CHECK_VALUE(x.dim() >= 1 && x.is_contiguous(), "softmax: expected a contiguous tensor");
        const OnDevice on(x);
        const int64_t n = x.size(-1), rows = n ? x.numel() / n : 0;
        const Tensor y = new_floats(x.sizes(), x), row_sum = new_floats({rows}, x), shift = new_floats({1}, x);
        if (x.numel()) {
            const size_t bytes = pam_hip_rowop_workspace_bytes();
            const Tensor ws = new_floats({(int64_t)(bytes / 4)}, x);
            check_call(pam_hip_softmax_fwd(data(x), data(y), data(row_sum), data(shift), rows, n, (float)offset, data(ws), bytes, on.stream), "softmax_fwd");
        }
        ctx->saved_data["offset"] = offset;
        Approx{a, b, e}.save(ctx);
        ctx->save_for_backward({x, row_sum, shift});
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const Approx f = Approx::saved(ctx);
        const at::AutoGradMode no_graph(false);
        const Tensor g = grads[0].contiguous();
        check_tensor(g);
        const int64_t n = g.size(-1), rows = n ? g.numel() / n : 0;
        const Tensor x = whole(saved[0], g, g.sizes(), "softmax_bwd"), row_sum = whole(saved[1], g, {rows}, "softmax_bwd"), shift = whole(saved[2], g, {1}, "softmax_bwd");
        const OnDevice on(g);
        const Tensor dx = new_floats(g.sizes(), g);
        if (g.numel())
            check_call(pam_hip_softmax_bwd(data(x), data(g), data(row_sum), data(shift), data(dx), rows, n,
                                           (float)ctx->saved_data["offset"].toDouble(), f.a, f.b, f.e, on.stream), "softmax_bwd");
        return {dx, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// layer_norm over the last n values; weight and bias of n values, or undefined
struct LayerNormNode : torch::autograd::Function<LayerNormNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, int64_t n, const std::optional<Tensor>& weight, const std::optional<Tensor>& bias,
                          double eps, double offset, bool a, bool b, bool e)
    {
        const Tensor w = weight ? weight->contiguous() : Tensor(), c = bias ? bias->contiguous() : Tensor();
        check_tensor(x);
        if (w.defined()) check_tensor(w);
        if (c.defined()) check_tensor(c);
        TORCH_CHECK_VALUE(x.is_contiguous() && n > 0 && x.numel() % n == 0, "layer_norm: expected contiguous rows");
        TORCH_CHECK_VALUE((!w.defined() || w.numel() == n) && (!c.defined() || c.numel() == n),
                          "layer_norm_fwd: weight and bias must have one value per column");
        const OnDevice on(x);
        const Tensor y = new_floats(x.sizes(), x);
        if (x.numel())
            check_call(pam_hip_layer_norm_fwd(data(x), data_or_null(w), data_or_null(c), data(y), x.numel() / n, n, (float)eps, (float)offset, on.stream),
                       "layer_norm_fwd");
        ctx->saved_data["n"] = n; ctx->saved_data["eps"] = eps; ctx->saved_data["offset"] = offset;
        if (w.defined()) ctx->saved_data["weight"] = w.sizes();
        if (c.defined()) ctx->saved_data["bias"] = c.sizes();
        Approx{a, b, e}.save(ctx);
        ctx->save_for_backward({x, w});
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const Approx f = Approx::saved(ctx);
        const Tensor g = grads[0].contiguous();
        check_tensor(g);
        const int64_t n = ctx->saved_data["n"].toInt(), rows = g.numel() / n;
        const Tensor x = whole(saved[0], g, g.sizes(), "layer_norm_bwd");
        const Tensor w = saved[1].defined() ? whole(saved[1], g, ctx->saved_data["weight"].toIntVector(), "layer_norm_bwd") : Tensor();
        const bool has_bias = ctx->saved_data.count("bias") != 0;
        // (edges are counted over the tensors that are there)
        const bool want_w = w.defined() && ctx->needs_input_grad(1), want_b = has_bias && ctx->needs_input_grad(w.defined() ? 2 : 1);
        const OnDevice on(g);
        const Tensor dx = new_floats(g.sizes(), g), terms = want_w ? new_floats({rows, n}, g) : Tensor();
        if (g.numel())
            check_call(pam_hip_layer_norm_bwd(data(x), data_or_null(w), data(g), data(dx), data_or_null(terms), rows, n,
                                              (float)ctx->saved_data["eps"].toDouble(), (float)ctx->saved_data["offset"].toDouble(),
                                              f.a, f.b, f.e, on.stream), "layer_norm_bwd");
        // the broadcast weight and bias collect their gradients by a sum over the rows, as autograd's expand does
        Tensor dw, db;
        const Tensor g_rows = want_b ? g.view({rows, n}) : Tensor();
        if (want_w && want_b && summable(g_rows)) {
            std::tie(dw, db) = column_sums(terms, g_rows);
        } else {
            if (want_w) dw = sum_rows(terms);
            if (want_b) db = sum_rows(g_rows);
        }
        if (want_w) dw = dw.view(w.sizes());
        if (want_b) db = db.view(ctx->saved_data["bias"].toIntVector());
        return {dx, Tensor(), dw, db, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// logsumexp over the last dimension of a contiguous tensor (the result keeps it, with one value), or log_softmax = x less
// that.  nonfinite, checked: as pam_hip_logsumexp_fwd_finite takes them, or null: the caller waits and looks.
struct LogsumexpNode : torch::autograd::Function<LogsumexpNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, bool log_softmax, int64_t nonfinite, int64_t checked, double offset, bool a, bool b, bool e)
    {
        check_tensor(x);
        TORCH_CHECK_VALUE(x.dim() >= 1 && x.is_contiguous() && x.numel() > 0, "logsumexp: expected a contiguous tensor");
        const OnDevice on(x);
        const int64_t n = x.size(-1), rows = x.numel() / n;
        std::vector<int64_t> shape = x.sizes().vec();
        if (!log_softmax) shape.back() = 1;
        const Tensor y = new_floats(shape, x), shift = new_floats({1}, x);
        const size_t bytes = pam_hip_rowop_workspace_bytes();
        const Tensor ws = new_floats({(int64_t)(bytes / 4)}, x);
        float* const lse = log_softmax ? nullptr : data(y);
        float* const out = log_softmax ? data(y) : nullptr;
        if (nonfinite)
            check_call(pam_hip_logsumexp_fwd_finite(data(x), lse, out, data(shift), rows, n, (float)offset, reinterpret_cast<int*>(nonfinite),
                                                    reinterpret_cast<void*>(checked), data(ws), bytes, on.stream), "logsumexp_fwd_finite");
        else
            check_call(pam_hip_logsumexp_fwd(data(x), lse, out, data(shift), rows, n, (float)offset, data(ws), bytes, on.stream), "logsumexp_fwd");
        ctx->saved_data["offset"] = offset; ctx->saved_data["log_softmax"] = log_softmax; ctx->saved_data["n"] = n;
        Approx{a, b, e}.save(ctx);
        ctx->save_for_backward({x, shift});
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const Approx f = Approx::saved(ctx);
        const at::AutoGradMode no_graph(false);
        const Tensor g = grads[0].contiguous();
        check_tensor(g);
        const bool log_softmax = ctx->saved_data["log_softmax"].toBool();
        const int64_t n = ctx->saved_data["n"].toInt(), rows = log_softmax ? g.numel() / n : g.numel();
        std::vector<int64_t> shape = g.sizes().vec();
        shape.back() = n;
        const Tensor x = whole(saved[0], g, shape, "logsumexp_bwd"), shift = whole(saved[1], g, {1}, "logsumexp_bwd");
        const OnDevice on(g);
        const Tensor dx = new_floats(shape, g);
        check_call(pam_hip_logsumexp_bwd(data(x), data(g), data(shift), data(dx), rows, n, log_softmax,
                                         (float)ctx->saved_data["offset"].toDouble(), f.a, f.b, f.e, on.stream), "logsumexp_bwd");
        return {dx, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// ---------------------------------------------------------------- elementwise

// A (*) B or A (/) B of contiguous tensors of one shape that both want a gradient or both do not; both gradients in one pass
template <bool DIVIDE>
struct PairNode : torch::autograd::Function<PairNode<DIVIDE>> {
    static Tensor forward(AutogradContext* ctx, const Tensor& A, const Tensor& B, double offset, bool a, bool b)
    {
        check_tensor(A);
        check_tensor(B);
        TORCH_CHECK_VALUE(A.sizes() == B.sizes() && A.is_contiguous() && B.is_contiguous(), "expected contiguous operands of one shape");
        const OnDevice on(A);
        const Tensor y = new_floats(A.sizes(), A);
        check_call((DIVIDE ? pam_hip_pad_fwd : pam_hip_pam_fwd)(data(A), data(B), data(y), A.numel(), (float)offset, on.stream), DIVIDE ? "pad_fwd" : "pam_fwd");
        ctx->saved_data["offset"] = offset;
        Approx{a, b, false}.save(ctx);
        ctx->save_for_backward({A, B});
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const char* const name = DIVIDE ? "pad_bwd_pair" : "pam_bwd_pair";
        const Approx f = Approx::saved(ctx);
        const at::AutoGradMode no_graph(false);
        const Tensor g = grads[0].contiguous();
        check_tensor(g);
        const Tensor A = whole(saved[0], g, g.sizes(), name), B = whole(saved[1], g, g.sizes(), name);
        const OnDevice on(g);
        const Tensor dA = new_floats(g.sizes(), g), dB = new_floats(g.sizes(), g);
        check_call((DIVIDE ? pam_hip_pad_bwd_pair : pam_hip_pam_bwd_pair)(data(A), data(B), data(g), data(dA), data(dB), g.numel(),
                   (float)ctx->saved_data["offset"].toDouble(), f.a, f.b, on.stream), name);
        return {dA, dB, Tensor(), Tensor(), Tensor()};
    }
};

// base ** x, log_base x, x ** p of a contiguous tensor.  The approximate gradient is that of the base e
// (pam/cuda_bindings.py:224-239, 262-276): exp(x) (*) g, g (/) x.
enum { kExp = 0, kLog = 1, kPow = 2 };
struct UnaryNode : torch::autograd::Function<UnaryNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, int64_t op, double number, double offset, bool a, bool e)
    {
        check_tensor(x);
        TORCH_CHECK_VALUE(x.is_contiguous(), "expected a contiguous tensor");
        const OnDevice on(x);
        const Tensor y = new_floats(x.sizes(), x);
        check_call((op == kExp ? pam_hip_pa_exp_fwd : op == kLog ? pam_hip_pa_log_fwd : pam_hip_pow_fwd)(data(x), data(y), x.numel(), (float)number,
                   (float)offset, on.stream), op == kExp ? "pa_exp_fwd" : op == kLog ? "pa_log_fwd" : "pow_fwd");
        ctx->saved_data["op"] = op; ctx->saved_data["number"] = number; ctx->saved_data["offset"] = offset;
        Approx{a, false, e}.save(ctx);
        ctx->save_for_backward({x});
        return y;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        const variable_list saved = ctx->get_saved_variables();
        const Approx f = Approx::saved(ctx);
        const int64_t op = ctx->saved_data["op"].toInt();
        const float number = (float)ctx->saved_data["number"].toDouble(), offset = (float)ctx->saved_data["offset"].toDouble();
        const at::AutoGradMode no_graph(false);
        const Tensor g = grads[0].contiguous();
        check_tensor(g);
        const Tensor x = whole(saved[0], g, g.sizes(), op == kExp ? "pa_exp_bwd" : op == kLog ? "pa_log_bwd" : "pow_bwd");
        const OnDevice on(g);
        const Tensor dx = new_floats(g.sizes(), g);
        const size_t n = g.numel();
        if (op == kPow) {
            check_call(pam_hip_pow_bwd(data(x), data(g), data(dx), n, number, offset, f.a, f.e, on.stream), "pow_bwd");
        } else if (!f.e) {
            check_call((op == kExp ? pam_hip_pa_exp_bwd : pam_hip_pa_log_bwd)(data(x), data(g), data(dx), n, number, offset, on.stream), op == kExp ? "pa_exp_bwd" : "pa_log_bwd");
        } else if (op == kExp) {
            const Tensor y = new_floats(g.sizes(), g);
            check_call(pam_hip_pa_exp_fwd(data(x), data(y), n, number, offset, on.stream), "pa_exp_fwd");
            check_call(pam_hip_pam_fwd(data(y), data(g), data(dx), n, offset, on.stream), "pam_fwd");
        } else {
            check_call(pam_hip_pad_fwd(data(g), data(x), data(dx), n, offset, on.stream), "pad_fwd");
        }
        return {dx, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// ---------------------------------------------------------------- optimizer

// The parameters from `start` on that one launch can update: those with a gradient and moments that are contiguous fp32
// tensors of one shape on one GPU, up to the first other one or one with another step count or device (parameters without
// a gradient are passed over).  Counts their step and returns (index behind them, step, device index, table as
// pam_hip_adam_tensor entries); an empty table: the parameter at the index is not such a one.
py::tuple adam_collect(py::list params, size_t start, py::dict state)
{
    static PyObject* const key_step = PyUnicode_InternFromString("step");
    static PyObject* const key_m = PyUnicode_InternFromString("exp_avg");
    static PyObject* const key_v = PyUnicode_InternFromString("exp_avg_sq");
    std::vector<pam_hip_adam_tensor> table;
    py::object step = py::none(), next = py::none();
    c10::Device device(c10::kCPU);
    size_t i = start;
    for (; i < params.size(); ++i) {
        const py::handle item = params[i];
        if (!THPVariable_Check(item.ptr())) break;
        const Tensor p = THPVariable_Unpack(item.ptr());
        const Tensor& g = p.grad();
        if (!g.defined()) continue;
        PyObject* entry = PyDict_GetItemWithError(state.ptr(), item.ptr());
        if (!entry && PyErr_Occurred()) throw py::error_already_set();
        if (!entry || !PyDict_Check(entry)) break;
        PyObject* count = PyDict_GetItemWithError(entry, key_step);
        PyObject* m_object = PyDict_GetItemWithError(entry, key_m);
        PyObject* v_object = PyDict_GetItemWithError(entry, key_v);
        if (!count || !PyLong_CheckExact(count) || !m_object || !v_object || !THPVariable_Check(m_object) || !THPVariable_Check(v_object)) break;
        const Tensor m = THPVariable_Unpack(m_object), v = THPVariable_Unpack(v_object);
        bool fits = p.is_cuda();
        for (const Tensor* t : {&p, &g, &m, &v})
            fits = fits && t->layout() == at::kStrided && t->scalar_type() == at::kFloat && t->device() == p.device() && t->sizes() == p.sizes() && t->is_contiguous();
        if (!fits) break;
        if (table.empty()) {
            step = py::reinterpret_borrow<py::object>(count);
            next = step + py::int_(1);
            device = p.device();
        } else if (device != p.device() || !step.equal(py::handle(count))) {
            break;
        }
        if (PyDict_SetItem(entry, key_step, next.ptr()) != 0) throw py::error_already_set();
        if (p.numel()) table.push_back({data(p), data(g), data(m), data(v), (size_t)p.numel()});
        else table.push_back({nullptr, nullptr, nullptr, nullptr, 0});
    }
    return py::make_tuple(i, next, (int)device.index(), py::bytes((const char*)table.data(), table.size() * sizeof(table[0])));
}

}  // namespace

// The interpreter is free for other threads while an op checks, allocates and launches, each of which may wait (a full
// launch queue, device memory, the table of workspaces); only adam_collect reads Python objects.
PYBIND11_MODULE(_pam_host, module)
{
    const py::call_guard<py::gil_scoped_release> unlocked;
    module.def("product", [](int kind, const Tensor& L, const Tensor& R, const std::optional<Tensor>& other, bool delta_left,
                             const std::optional<Tensor>& bias, double offset) {
        return product(kind, L, R, other.value_or(Tensor()), delta_left, bias.value_or(Tensor()), offset);
    }, unlocked);
    module.def("column_sums", [](const Tensor& a, const std::optional<Tensor>& b) {
        std::pair<Tensor, Tensor> sums;
        {
            const py::gil_scoped_release release;
            sums = column_sums(a, b.value_or(Tensor()));
        }
        return b ? py::cast(sums) : py::cast(sums.first);
    });
    module.def("sum_rows", &sum_rows, unlocked);
    module.def("matmul", [](const Tensor& A, const Tensor& B, int64_t dims, double offset, bool a, bool b) {
        return MatmulNode::apply(A, B, dims, offset, a, b);
    }, unlocked);
    module.def("linear", [](const Tensor& X, const Tensor& W, const Tensor& bias, double offset, bool a, bool b) {
        return LinearNode::apply(X, W, bias, offset, a, b);
    }, unlocked);
    module.def("softmax", [](const Tensor& x, double offset, bool a, bool b, bool e) { return SoftmaxNode::apply(x, offset, a, b, e); }, unlocked);
    module.def("layer_norm", [](const Tensor& x, int64_t n, const std::optional<Tensor>& weight, const std::optional<Tensor>& bias, double eps,
                                double offset, bool a, bool b, bool e) {
        return LayerNormNode::apply(x, n, weight, bias, eps, offset, a, b, e);
    }, unlocked);
    module.def("logsumexp", [](const Tensor& x, bool log_softmax, int64_t nonfinite, int64_t checked, double offset, bool a, bool b, bool e) {
        return LogsumexpNode::apply(x, log_softmax, nonfinite, checked, offset, a, b, e);
    }, unlocked);
    module.def("mul", [](const Tensor& A, const Tensor& B, double offset, bool a, bool b) { return PairNode<false>::apply(A, B, offset, a, b); }, unlocked);
    module.def("div", [](const Tensor& A, const Tensor& B, double offset, bool a, bool b) { return PairNode<true>::apply(A, B, offset, a, b); }, unlocked);
    module.def("unary", [](const Tensor& x, int64_t op, double number, double offset, bool a, bool e) { return UnaryNode::apply(x, op, number, offset, a, e); }, unlocked);
    module.def("adam_collect", &adam_collect);
}
