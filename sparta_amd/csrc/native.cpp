// Native host path of the operators: the Python extension module sparta_amd._native.
//
// One operator call is one call into this file: operand checks, the output allocation, the
// autograd node and the launch through the C ABI of libsparta_hip.so.  The same steps in
// Python (an autograd.Function, a ctypes call with 25 arguments, a pointer object per
// tensor) cost 15 - 19 us per forward call and 90 us per training step on kernels of 5 - 60 us.
//
// Errors keep the exception types of the Python layer: AssertionError for operands or
// configurations that do not fit (a failed trial for the tuner), ValueError for unsupported
// types and alignments, RuntimeError for the rest.
#include <torch/extension.h>
#include <ATen/EmptyTensor.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <c10/hip/HIPStream.h>

#include <array>
#include <atomic>
#include <memory>
#include <mutex>
#include <optional>
#include <string>
#include <vector>

#include "../../include/sparta_hip.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// ---- errors --------------------------------------------------------------------------------
struct AssertionFailure : std::runtime_error {
    using std::runtime_error::runtime_error;
};
struct ValueFailure : std::runtime_error {
    using std::runtime_error::runtime_error;
};
struct AttributeFailure : std::runtime_error {
    using std::runtime_error::runtime_error;
};

template <typename... Args>
[[noreturn]] void assertion(const Args&... args) { throw AssertionFailure(c10::str(args...)); }

void check_rc(int rc, const char* what) {
    if (rc == 0) return;
    const std::string msg = c10::str(what, ": ", spx_last_error(), " (code ", rc, ")");
    if (rc == SPX_E_SHAPE || rc == SPX_E_CONFIG) throw AssertionFailure(msg);
    if (rc == SPX_E_NULL || rc == SPX_E_DTYPE || rc == SPX_E_ALIGN || rc == SPX_E_WORKSPACE) throw ValueFailure(msg);
    throw std::runtime_error(msg);
}

// In a backward pass the exception crosses the autograd engine, which carries Python errors
// through unchanged but turns every other type into RuntimeError.
template <typename F>
auto with_python_errors(F&& body) -> decltype(body()) {
    PyObject* type = nullptr;
    std::string msg;
    try {
        return body();
    } catch (const AssertionFailure& e) {
        type = PyExc_AssertionError;
        msg = e.what();
    } catch (const ValueFailure& e) {
        type = PyExc_ValueError;
        msg = e.what();
    } catch (const AttributeFailure& e) {
        type = PyExc_AttributeError;
        msg = e.what();
    }
    py::gil_scoped_acquire gil;
    PyErr_SetString(type, msg.c_str());
    python_error err;
    err.persist();
    throw err;
}

// ---- operands --------------------------------------------------------------------------------
int dtype_code(const Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return SPX_F32;
        case at::kHalf: return SPX_F16;
        case at::kBFloat16: return SPX_BF16;
        default:
            throw ValueFailure(c10::str("unsupported dtype torch.", c10::toString(t.scalar_type()),
                                        ": expected float32, float16 or bfloat16"));
    }
}

void* device_ptr(const Tensor& t) {
    if (!t.is_cuda()) throw std::runtime_error("sparta_amd kernels run on the GPU only: got a CPU tensor");
    return t.data_ptr();
}
void* device_ptr(const std::optional<Tensor>& t) { return t.has_value() && t->defined() ? device_ptr(*t) : nullptr; }

spx_stream_t stream_of(const Tensor& t) { return (spx_stream_t)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void require_numel(const char* what, const char* name, const Tensor& t, int64_t numel) {
    if (t.numel() != numel)
        assertion(what, ": ", name, " has ", t.numel(), " elements (shape ", t.sizes(), "), the kernel is bound to ", numel);
}

// Whether a call may take the native autograd node.  Not while it is traced (the tracer would record the output
// allocation and nothing else), not with a forward-mode tangent on an input (the node has no rule for it and would
// drop it), not under the transforms of torch.func or with their tensors, whose data is not behind data_ptr():
// those calls go through the Python autograd.Function of the operator, which records or refuses them.
bool plain_call(std::initializer_list<const Tensor*> inputs) {
    constexpr c10::DispatchKeySet modes({c10::DispatchKey::Tracer, c10::DispatchKey::FuncTorchDynamicLayerFrontMode});
    constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::Functionalize,
                                           c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::FuncTorchBatched});
    if (c10::impl::tls_local_dispatch_key_set().included_.has_any(modes)) return false;
    for (const Tensor* t : inputs)
        if (t && t->defined() && (t->key_set().has_any(wrapped) || t->_fw_grad(0).defined())) return false;
    return true;
}

bool records(std::initializer_list<const Tensor*> inputs) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor* t : inputs)
        if (t && t->defined() && t->requires_grad()) return true;
    return false;
}

// ---- block-sparse matmul ---------------------------------------------------------------------
// One bound spx_matmul call.  Never changes after it is published (but for the tile hint), so
// a backward pass may keep the plan of its forward pass while the kernel is bound to a new mask.
struct MatmulPlan {
    int mode, trans_a, trans_b, compressed, biased;
    int batch, M, K, N, BM, BK, BN;
    int idx_kind, nnz;
    int64_t sparse_stride;
    int64_t numel_a, numel_b;
    std::optional<Tensor> ptr, idx, sched, nnz_dev;
    mutable std::atomic<int> tile_cfg;
    mutable std::atomic<bool> strict{false};   // a refused tile configuration is an error (tuner trials)

    bool sparse_out() const { return mode == SPX_DDS && compressed; }

    // `out_shape` has the number of elements of the result; it lets the caller have the
    // result (a gradient) in the shape of another tensor.
    Tensor run(const Tensor& a_in, const Tensor& b_in, const Tensor* bias_in, at::IntArrayRef out_shape) const {
        if (a_in.scalar_type() != b_in.scalar_type())
            assertion("operand dtypes differ: ", a_in.dtype(), " vs ", b_in.dtype());
        require_numel("spx_matmul", "A", a_in, numel_a);
        require_numel("spx_matmul", "B", b_in, numel_b);
        if (biased) {
            if (!bias_in || !bias_in->defined()) assertion("spx_matmul: bias is required");
            require_numel("spx_matmul", "bias", *bias_in, (int64_t)batch * N);
        } else if (bias_in && bias_in->defined()) {
            throw py::type_error("spx_matmul: the kernel was built without a bias and takes two operands");
        }
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        const int code = dtype_code(a_in);
        const Tensor a = a_in.contiguous(), b = b_in.contiguous();
        Tensor bias;
        if (biased) bias = bias_in->to(a.scalar_type()).contiguous();
        void *pa = device_ptr(a), *pb = device_ptr(b);
        void* pbias = bias.defined() ? device_ptr(bias) : nullptr;
        if (mode == SPX_DDS) {
            const size_t ws_bytes = split_workspace(code, false);
            if (ws_bytes > 0) return run_split(code, a, b, nullptr, ws_bytes, out_shape);
        }
        // a dense sparse-output result keeps zeros in dead tiles; every other result is fully
        // overwritten by the kernel
        Tensor c = mode == SPX_DDS && !compressed ? at::zeros(out_shape, a.options()) : at::empty(out_shape, a.options());
        int cfg = tile_cfg.load(std::memory_order_relaxed);
        int rc;
        while (true) {
            rc = spx_matmul(mode, code, trans_a, trans_b, compressed, pa, pb, pbias, c.data_ptr(),
                            (const int32_t*)device_ptr(ptr), device_ptr(idx), idx_kind, (const int32_t*)device_ptr(sched), nnz,
                            (const int32_t*)device_ptr(nnz_dev), sparse_stride, batch, M, K, N, BM, BK, BN, cfg, stream_of(a));
            if (rc == SPX_E_CONFIG && (cfg & 0xffff) && !strict) {
                // the configured tile variant does not take these shapes (nothing was launched):
                // the library's own choice from here on
                cfg &= ~0xffff;
                tile_cfg.store(cfg, std::memory_order_relaxed);
                continue;
            }
            break;
        }
        check_rc(rc, "spx_matmul");
        return c;
    }

    // A sparse-output product may be split along k (spx_matmul_split); the bytes that takes, 0: not split.
    size_t split_workspace(int code, bool colsum) const {
        if (nnz_dev.has_value() || biased || has_tile_cfg()) return 0;
        // the whole reduction is one or two stages deep: the block-row kernels of spx_matmul
        if (!trans_a && trans_b && K * (code == SPX_F32 ? 4 : 2) <= 256) return 0;
        return spx_matmul_split_workspace_bytes(code, trans_a, trans_b, nnz, batch, M, K, N, BM, BN, 0, colsum);
    }
    // `colsum` (may be null) receives the sums of op(A) over k.  Contiguous operands.
    Tensor run_split(int code, const Tensor& a, const Tensor& b, Tensor* colsum, size_t ws_bytes, at::IntArrayRef out_shape) const {
        Tensor c = compressed ? at::empty(out_shape, a.options()) : at::zeros(out_shape, a.options());
        Tensor ws;
        if (ws_bytes > 0) ws = at::empty({(int64_t)ws_bytes}, a.options().dtype(at::kByte));
        check_rc(spx_matmul_split(code, trans_a, trans_b, compressed, device_ptr(a), device_ptr(b), c.data_ptr(),
                                  colsum ? device_ptr(*colsum) : nullptr, (const int32_t*)device_ptr(ptr),
                                  (const int32_t*)device_ptr(idx), nnz, sparse_stride, batch, M, K, N, BM, BN, 0,
                                  ws_bytes > 0 ? ws.data_ptr() : nullptr, ws_bytes, stream_of(a)), "spx_matmul_split");
        return c;
    }
    // The weight gradient together with the sums of its first operand over k (the bias gradient).
    Tensor run_with_colsum(const Tensor& a, const Tensor& b, at::IntArrayRef out_shape, Tensor* colsum) const {
        if (a.scalar_type() != b.scalar_type()) assertion("operand dtypes differ: ", a.dtype(), " vs ", b.dtype());
        require_numel("spx_matmul_split", "A", a, numel_a);
        require_numel("spx_matmul_split", "B", b, numel_b);
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        const int code = dtype_code(a);
        *colsum = at::empty({batch, M}, a.options());
        return run_split(code, a.contiguous(), b.contiguous(), colsum, split_workspace(code, true), out_shape);
    }
    // (a configured tile variant is what the tuner timed: the product is its own launch then)
    bool gives_colsum() const { return mode == SPX_DDS && trans_a && !nnz_dev.has_value() && !has_tile_cfg(); }
    bool has_tile_cfg() const { return (tile_cfg.load(std::memory_order_relaxed) & 0xffff) != 0; }

    c10::SmallVector<int64_t, 3> shape() const {
        if (sparse_out()) return {batch, sparse_stride};
        return {batch, M, N};
    }

    // Gradient of the bias [batch, N] from the gradient of the result.
    Tensor bias_grad(const Tensor& grad, at::IntArrayRef out_shape) const {
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        if (!sparse_out()) return grad.view({batch, M, N}).sum(1).view(out_shape);
        const Tensor vals = grad.contiguous();
        Tensor sum = at::empty({batch, N}, vals.options().dtype(at::kFloat));
        check_rc(spx_bcs_sum(device_ptr(vals), device_ptr(sum), device_ptr(idx), idx_kind, nnz, batch, M, N, BM, BN,
                             dtype_code(vals), 1, sparse_stride, stream_of(vals)), "spx_bcs_sum");
        return sum.to(vals.scalar_type()).view(out_shape);
    }
};
typedef std::shared_ptr<const MatmulPlan> MatmulPlanPtr;

// The launch object of one kernel: the plan it is bound to at the moment.
class MatmulKernel {
public:
    void bind(int mode, int trans_a, int trans_b, int compressed, int biased, int batch, int M, int K, int N, int BM, int BK,
              int BN, std::optional<Tensor> ptr, std::optional<Tensor> idx, int idx_kind, std::optional<Tensor> sched, int nnz,
              std::optional<Tensor> nnz_dev, int64_t sparse_stride, int64_t numel_a, int64_t numel_b, int tile_cfg) {
        auto p = std::make_shared<MatmulPlan>();
        p->mode = mode; p->trans_a = trans_a; p->trans_b = trans_b; p->compressed = compressed; p->biased = biased;
        p->batch = batch; p->M = M; p->K = K; p->N = N; p->BM = BM; p->BK = BK; p->BN = BN;
        p->ptr = std::move(ptr); p->idx = std::move(idx); p->idx_kind = idx_kind; p->sched = std::move(sched);
        p->nnz = nnz; p->nnz_dev = std::move(nnz_dev); p->sparse_stride = sparse_stride;
        p->tile_cfg = tile_cfg;
        p->numel_a = numel_a; p->numel_b = numel_b;
        plan_ = std::move(p);
    }
    void unbind() { plan_.reset(); }
    void set_strict(bool strict) { if (plan_) plan_->strict = strict; }
    const MatmulPlanPtr& plan() const { return plan_; }   // null: not bound
    const MatmulPlanPtr& bound_plan() const { require_bound(plan_); return plan_; }
    static void require_bound(const MatmulPlanPtr& p) {
        if (!p) throw ValueFailure("The kernel is not compiled.");
    }
    Tensor call(const Tensor& a, const Tensor& b, const std::optional<Tensor>& bias) const {
        const MatmulPlanPtr p = bound_plan();
        py::gil_scoped_release nogil;
        return p->run(a, b, bias.has_value() ? &*bias : nullptr, p->shape());
    }

private:
    MatmulPlanPtr plan_;
};

// C = op(A) op(B) (+ bias) and its gradients, over the plans of one forward pass: its masks, its layout.
struct MatmulStep {
    MatmulPlanPtr fwd, bwd_a, bwd_b;
    bool have_a, have_b;                // the operator was built with these kernels
    bool trans_a, trans_b, relu, drop_batch;

    Tensor forward(const Tensor& a, const Tensor& b, const Tensor* bias) const {
        const auto shape = fwd->shape();
        return fwd->run(a, b, bias, drop_batch ? at::IntArrayRef(shape).slice(1) : at::IntArrayRef(shape));
    }
    // Gradients of A, B and the bias where `need` asks for them.  gate: the output, where a fused relu decided which
    // gradients pass.
    std::array<Tensor, 3> gradients(const Tensor& grad_out, const Tensor& A, const Tensor& B, const Tensor& gate,
                                    std::array<bool, 3> need, at::IntArrayRef bias_shape) const {
        std::array<Tensor, 3> out;
        at::AutoGradMode no_grad(false);
        Tensor grad = grad_out.contiguous();
        if (relu) grad = at::threshold_backward(grad, gate, 0);
        if (need[0]) {
            require_built(have_a, bwd_a, "backward_A");
            out[0] = trans_a ? bwd_a->run(B, grad, nullptr, A.sizes()) : bwd_a->run(grad, B, nullptr, A.sizes());
        }
        if (need[1]) {
            require_built(have_b, bwd_b, "backward_B");
            if (need[2] && trans_b && !fwd->sparse_out() && bwd_b->gives_colsum()) {
                Tensor bias_grad;
                out[1] = bwd_b->run_with_colsum(grad, A, B.sizes(), &bias_grad);
                out[2] = bias_grad.view(bias_shape);
                return out;
            }
            out[1] = trans_b ? bwd_b->run(grad, A, nullptr, B.sizes()) : bwd_b->run(A, grad, nullptr, B.sizes());
        }
        if (need[2]) out[2] = fwd->bias_grad(grad, bias_shape);
        return out;
    }

private:
    static void require_built(bool have, const MatmulPlanPtr& plan, const char* name) {
        if (!have) throw AttributeFailure(c10::str("the operator was built without its ", name, " kernel"));
        MatmulKernel::require_bound(plan);
    }
};

struct MatmulBackward : public Node {
    MatmulStep step;
    SavedVariable a, b, gate;
    std::vector<int64_t> bias_shape;

    variable_list apply(variable_list&& grads) override {
        return with_python_errors([&]() -> variable_list {
            variable_list out(num_outputs());
            if (!grads[0].defined()) return out;
            std::lock_guard<std::mutex> lock(mutex_);
            const Tensor A = a.unpack(), B = b.unpack();
            const Tensor saved_out = step.relu ? gate.unpack(shared_from_this()) : Tensor();
            const auto got = step.gradients(grads[0], A, B, saved_out,
                                            {task_should_compute_output(0), task_should_compute_output(1),
                                             num_outputs() > 2 && task_should_compute_output(2)}, bias_shape);
            for (size_t i = 0; i < out.size(); ++i) out[i] = got[i];
            return out;
        });
    }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        a.reset_data();
        b.reset_data();
        gate.reset_data();
    }
    std::string name() const override { return "SparseMatmulBackward"; }
};

class MatmulOp {
public:
    // `general`: the Python autograd.Function of the operator (its apply), called as general(this, A, B[, bias])
    MatmulOp(std::shared_ptr<MatmulKernel> fwd, std::shared_ptr<MatmulKernel> bwd_a, std::shared_ptr<MatmulKernel> bwd_b,
             bool trans_a, bool trans_b, bool relu, bool drop_batch, py::object general)
        : fwd_(std::move(fwd)), bwd_a_(std::move(bwd_a)), bwd_b_(std::move(bwd_b)), trans_a_(trans_a), trans_b_(trans_b),
          relu_(relu), drop_batch_(drop_batch), general_(std::move(general)) {}

    MatmulStep step() const {
        return {fwd_->bound_plan(), bwd_a_ ? bwd_a_->plan() : nullptr, bwd_b_ ? bwd_b_->plan() : nullptr,
                (bool)bwd_a_, (bool)bwd_b_, trans_a_, trans_b_, relu_, drop_batch_};
    }
    Tensor call(const Tensor& a, const Tensor& b, const std::optional<Tensor>& bias) const {
        const Tensor* bias_p = bias.has_value() ? &*bias : nullptr;
        if (!plain_call({&a, &b, bias_p})) {
            const py::object self = py::cast(this, py::return_value_policy::reference);
            return (bias_p ? general_(self, a, b, *bias_p) : general_(self, a, b)).cast<Tensor>();
        }
        MatmulStep now = step();
        py::gil_scoped_release nogil;
        Tensor out = now.forward(a, b, bias_p);
        if (!records({&a, &b, bias_p})) return out;
        auto node = std::shared_ptr<MatmulBackward>(new MatmulBackward(), torch::autograd::deleteNode);
        node->set_next_edges(bias_p ? torch::autograd::collect_next_edges(a, b, *bias_p) : torch::autograd::collect_next_edges(a, b));
        node->step = std::move(now);
        node->a = SavedVariable(a, false);
        node->b = SavedVariable(b, false);
        if (bias_p) node->bias_shape = bias_p->sizes().vec();
        torch::autograd::set_history(out, node);
        if (relu_) node->gate = SavedVariable(out, true);
        return out;
    }

    // a copy launches through the copies of the kernels (which copy.deepcopy finds in `memo`)
    std::unique_ptr<MatmulOp> deepcopy(const py::object& memo) const {
        const py::object copy = py::module_::import("copy").attr("deepcopy");
        auto kernel = [&](const std::shared_ptr<MatmulKernel>& k) {
            return k ? copy(py::cast(k), memo).cast<std::shared_ptr<MatmulKernel>>() : nullptr;
        };
        return std::make_unique<MatmulOp>(kernel(fwd_), kernel(bwd_a_), kernel(bwd_b_), trans_a_, trans_b_, relu_, drop_batch_,
                                          general_);
    }

private:
    std::shared_ptr<MatmulKernel> fwd_, bwd_a_, bwd_b_;
    bool trans_a_, trans_b_, relu_, drop_batch_;
    py::object general_;
};

// ---- masked block softmax ----------------------------------------------------------------------
struct SoftmaxPlan {
    bool backward;
    int compressed, batch, H, W, BH, BW;
    int64_t stride;
    Tensor row_ptr, idx;
    std::optional<Tensor> mask;
    mutable std::atomic<int> tile_cfg;
    mutable std::atomic<bool> strict{false};

    const char* what() const { return backward ? "spx_softmax_backward" : "spx_softmax_forward"; }

    // forward: a = x; backward: a = gradient of y, y
    Tensor run(const Tensor& a_in, const Tensor* y_in, double T, at::IntArrayRef out_shape) const {
        require_numel(what(), backward ? "grad_y" : "x", a_in, batch * stride);
        if (backward) {
            require_numel(what(), "y", *y_in, batch * stride);
            if (a_in.scalar_type() != y_in->scalar_type())
                assertion("operand dtypes differ: ", a_in.dtype(), " vs ", y_in->dtype());
        }
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        Tensor out = compressed ? at::empty(out_shape, a_in.options()) : at::zeros(out_shape, a_in.options());
        if (out.numel() == 0) return out;   // no live block: nothing to compute
        const int code = dtype_code(a_in);
        const Tensor a = a_in.contiguous();
        const Tensor y = backward ? y_in->contiguous() : Tensor();
        const int32_t *rp = (const int32_t*)device_ptr(row_ptr), *ix = (const int32_t*)device_ptr(idx);
        const uint8_t* m = (const uint8_t*)device_ptr(mask);
        int cfg = tile_cfg.load(std::memory_order_relaxed), rc;
        while (true) {
            rc = backward ? spx_softmax_backward(code, compressed, device_ptr(a), device_ptr(y), out.data_ptr(), rp, ix, m, (float)T,
                                                 batch, H, W, BH, BW, stride, cfg, stream_of(a))
                          : spx_softmax_forward(code, compressed, device_ptr(a), out.data_ptr(), rp, ix, m, (float)T,
                                                batch, H, W, BH, BW, stride, cfg, stream_of(a));
            if (rc == SPX_E_CONFIG && cfg && !strict) {   // the configured variant does not take this dtype / block width
                cfg = 0;
                tile_cfg.store(0, std::memory_order_relaxed);
                continue;
            }
            break;
        }
        check_rc(rc, what());
        return out;
    }
    c10::SmallVector<int64_t, 3> shape() const {
        if (compressed) return {batch, stride};
        return {batch, H, W};
    }
};
typedef std::shared_ptr<const SoftmaxPlan> SoftmaxPlanPtr;

class SoftmaxKernel {
public:
    void bind(bool backward, int compressed, int batch, int H, int W, int BH, int BW, int64_t stride, Tensor row_ptr, Tensor idx,
              std::optional<Tensor> mask, int tile_cfg) {
        auto p = std::make_shared<SoftmaxPlan>();
        p->backward = backward; p->compressed = compressed; p->batch = batch; p->H = H; p->W = W; p->BH = BH; p->BW = BW;
        p->stride = stride; p->row_ptr = std::move(row_ptr); p->idx = std::move(idx); p->mask = std::move(mask);
        p->tile_cfg = tile_cfg;
        if (p->mask.has_value()) require_numel(p->what(), "mask", *p->mask, stride);
        plan_ = std::move(p);
    }
    void unbind() { plan_.reset(); }
    void set_strict(bool strict) { if (plan_) plan_->strict = strict; }
    const SoftmaxPlanPtr& plan() const { return plan_; }
    static void require_bound(const SoftmaxPlanPtr& p) {
        if (!p) throw ValueFailure("The kernel is not compiled.");
    }
    Tensor forward(const Tensor& x, double T) const {
        const SoftmaxPlanPtr p = plan_;
        require_bound(p);
        py::gil_scoped_release nogil;
        return p->run(x, nullptr, T, p->shape());
    }
    Tensor backward(const Tensor& grad, const Tensor& y, double T) const {
        const SoftmaxPlanPtr p = plan_;
        require_bound(p);
        py::gil_scoped_release nogil;
        return p->run(grad, &y, T, p->shape());
    }

private:
    SoftmaxPlanPtr plan_;
};

// y = masked softmax of x and its gradient, over the plans and the factor of one forward pass.
struct SoftmaxStep {
    SoftmaxPlanPtr fwd, bwd;
    bool have;                          // the operator was built with its backward kernel
    double T;

    Tensor forward(const Tensor& x) const { return fwd->run(x, nullptr, T, fwd->shape()); }
    Tensor gradient(const Tensor& grad, const Tensor& y, at::IntArrayRef x_shape) const {
        if (!have) throw AttributeFailure("the operator was built without its backward kernel");
        SoftmaxKernel::require_bound(bwd);
        at::AutoGradMode no_grad(false);
        return bwd->run(grad, &y, T, x_shape);
    }
};

struct SoftmaxBackward : public Node {
    SoftmaxStep step;
    SavedVariable y;
    std::vector<int64_t> x_shape;

    variable_list apply(variable_list&& grads) override {
        return with_python_errors([&]() -> variable_list {
            variable_list out(1);
            if (!grads[0].defined() || !task_should_compute_output(0)) return out;
            std::lock_guard<std::mutex> lock(mutex_);
            out[0] = step.gradient(grads[0], y.unpack(shared_from_this()), x_shape);
            return out;
        });
    }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        y.reset_data();
    }
    std::string name() const override { return "SparseSoftmaxBackward"; }
};

class SoftmaxOp {
public:
    // T: what the kernels multiply by; `general`: as in MatmulOp, called as general(this, x)
    SoftmaxOp(std::shared_ptr<SoftmaxKernel> fwd, std::shared_ptr<SoftmaxKernel> bwd, double T, py::object general)
        : fwd_(std::move(fwd)), bwd_(std::move(bwd)), T_(T), general_(std::move(general)) {}
    void set_temperature(double T) { T_ = T; }
    SoftmaxStep step() const {
        SoftmaxKernel::require_bound(fwd_->plan());
        return {fwd_->plan(), bwd_ ? bwd_->plan() : nullptr, (bool)bwd_, T_};
    }
    Tensor call(const Tensor& x) const {
        if (!plain_call({&x})) return general_(py::cast(this, py::return_value_policy::reference), x).cast<Tensor>();
        SoftmaxStep now = step();
        py::gil_scoped_release nogil;
        Tensor y = now.forward(x);
        if (!records({&x})) return y;
        auto node = std::shared_ptr<SoftmaxBackward>(new SoftmaxBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(x));
        node->step = std::move(now);
        node->x_shape = x.sizes().vec();
        torch::autograd::set_history(y, node);
        node->y = SavedVariable(y, true);
        return y;
    }
    std::unique_ptr<SoftmaxOp> deepcopy(const py::object& memo) const {
        const py::object copy = py::module_::import("copy").attr("deepcopy");
        auto kernel = [&](const std::shared_ptr<SoftmaxKernel>& k) {
            return k ? copy(py::cast(k), memo).cast<std::shared_ptr<SoftmaxKernel>>() : nullptr;
        };
        return std::make_unique<SoftmaxOp>(kernel(fwd_), kernel(bwd_), T_, general_);
    }

private:
    std::shared_ptr<SoftmaxKernel> fwd_, bwd_;
    double T_;
    py::object general_;
};

// ---- fused attention -------------------------------------------------------------------------------
// The fused kernels over one index: launches with their operand checks and allocations.
class AttentionKernel {
public:
    AttentionKernel(Tensor row_ptr, Tensor bcsr, std::optional<Tensor> col_ptr, std::optional<Tensor> bcsc,
                    std::optional<Tensor> mask, double inv_temperature, int Nt, int Ns, int BH, int BW)
        : row_ptr_(std::move(row_ptr)), bcsr_(std::move(bcsr)), col_ptr_(std::move(col_ptr)), bcsc_(std::move(bcsc)),
          mask_(std::move(mask)), inv_t_((float)inv_temperature), Nt_(Nt), Ns_(Ns), BH_(BH), BW_(BW) {}

    // (output, tile configuration that ran)
    std::pair<Tensor, int> forward(const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, int tile_cfg, bool strict) const {
        py::gil_scoped_release nogil;
        const Dims d = dims("spx_attention_forward", q_in, k_in, v_in);
        device_ptr(q_in);   // refuses CPU tensors ahead of the allocations and the look-up of the stream
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        const Tensor q = q_in.contiguous(), k = k_in.contiguous(), v = v_in.contiguous();
        Tensor out = at::empty(q.sizes(), q.options());
        int rc;
        while (true) {
            rc = spx_attention_forward(d.code, device_ptr(q), device_ptr(k), device_ptr(v), out.data_ptr(), rows(), entries(),
                                       (const uint8_t*)device_ptr(mask_), inv_t_, d.batch, Nt_, Ns_, d.E, BH_, BW_, tile_cfg, stream_of(q));
            if (rc == SPX_E_CONFIG && tile_cfg && !strict) {   // a tuned variant that does not take these shapes
                tile_cfg = 0;
                continue;
            }
            break;
        }
        check_rc(rc, "spx_attention_forward");
        return {out, tile_cfg};
    }
    // (output, log-sum-exp of every score row)
    std::pair<Tensor, Tensor> forward_lse(const Tensor& q, const Tensor& k, const Tensor& v) const {
        py::gil_scoped_release nogil;
        const Dims d = dims("spx_attention_forward_lse", q, k, v);
        device_ptr(q);
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        Tensor out = at::empty(q.sizes(), q.options()), lse = at::empty({d.batch, Nt_}, q.options().dtype(at::kFloat));
        check_rc(spx_attention_forward_lse(d.code, contig(q), contig(k), contig(v), out.data_ptr(), (float*)lse.data_ptr(),
                                           rows(), entries(), (const uint8_t*)device_ptr(mask_), inv_t_, d.batch, Nt_, Ns_, d.E, BH_, BW_,
                                           stream_of(q)),
                 "spx_attention_forward_lse");
        return {out, lse};
    }
    // The live blocks of the element mask, one after the other in BCSR order.
    Tensor live_mask(int64_t nnz) const {
        py::gil_scoped_release nogil;
        if (!mask_.has_value()) throw ValueFailure("there is no element mask");
        require_numel("spx_bcs_gather", "mask", *mask_, (int64_t)Nt_ * Ns_);
        require_bytes("spx_bcs_gather", *mask_);
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        Tensor live = at::empty({nnz * BH_ * BW_}, mask_->options());
        check_rc(spx_bcs_gather(contig(*mask_), live.data_ptr(), entries(), SPX_IDX_BCSR_I32, (int)nnz, nullptr, 1, Nt_, Ns_, BH_, BW_, 1,
                                nnz * BH_ * BW_, stream_of(*mask_)), "spx_bcs_gather");
        return live;
    }
    // (query gradient, row constants); `mask`: the live blocks of the forward pass's element mask, nnz of them
    std::pair<Tensor, Tensor> backward_q(const Tensor& grad, const Tensor& out, const Tensor& q, const Tensor& k, const Tensor& v,
                                         const Tensor& lse, const std::optional<Tensor>& mask, int64_t nnz) const {
        py::gil_scoped_release nogil;
        const char* what = "spx_attention_backward_q";
        const Dims d = dims(what, q, k, v);
        require_like(what, "grad_out", grad, q);
        require_like(what, "out", out, q);
        require_numel(what, "row_lse", lse, (int64_t)d.batch * Nt_);
        require_mask(what, mask, nnz);
        device_ptr(q);
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        Tensor grad_q = at::empty(q.sizes(), q.options()), dot = at::empty({d.batch, Nt_}, q.options().dtype(at::kFloat));
        check_rc(spx_attention_backward_q_live_mask(
                     d.code, contig(grad), contig(out), contig(q), contig(k), contig(v), (const float*)contig(lse), grad_q.data_ptr(),
                     (float*)dot.data_ptr(), rows(), entries(), (const uint8_t*)(mask ? contig(*mask) : nullptr), inv_t_, d.batch, Nt_, Ns_,
                     d.E, BH_, BW_, stream_of(q)), what);
        return {grad_q, dot};
    }
    // (key gradient, value gradient)
    std::pair<Tensor, Tensor> backward_kv(const Tensor& grad, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& lse,
                                          const Tensor& dot, const std::optional<Tensor>& mask, int64_t nnz) const {
        py::gil_scoped_release nogil;
        const char* what = "spx_attention_backward_kv_recompute";
        const Dims d = dims(what, q, k, v);
        require_like(what, "grad_out", grad, q);
        require_numel(what, "row_lse", lse, (int64_t)d.batch * Nt_);
        require_numel(what, "row_dot", dot, (int64_t)d.batch * Nt_);
        require_mask(what, mask, nnz);
        if (!col_ptr_.has_value() || !bcsc_.has_value()) throw ValueFailure("the column-side kernel needs the BCSC index");
        device_ptr(q);
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        Tensor grad_k = at::empty(k.sizes(), k.options()), grad_v = at::empty(k.sizes(), k.options());
        check_rc(spx_attention_backward_kv_live_mask(
                     d.code, contig(grad), contig(q), contig(k), contig(v), (const float*)contig(lse), (const float*)contig(dot),
                     grad_k.data_ptr(), grad_v.data_ptr(), (const int32_t*)device_ptr(col_ptr_), device_ptr(bcsc_),
                     bcsc_->scalar_type() == at::kLong ? SPX_IDX_BCSC_I64 : SPX_IDX_BCSC_I32, (const uint8_t*)(mask ? contig(*mask) : nullptr),
                     inv_t_, d.batch, Nt_, Ns_, d.E, BH_, BW_, stream_of(q)), what);
        return {grad_k, grad_v};
    }

private:
    struct Dims {
        int code, batch, E;
    };
    // the tensors behind the pointers against what a kernel walks; AssertionError before any launch
    Dims dims(const char* what, const Tensor& q, const Tensor& k, const Tensor& v) const {
        if (q.dim() < 2) assertion(what, ": query of shape ", q.sizes());
        const int64_t E = q.size(-1);
        const int64_t per = (int64_t)Nt_ * E;
        int64_t batch = 1;
        for (int64_t i = 0; i < q.dim() - 2; ++i) batch *= q.size(i);
        require_numel(what, "q", q, batch * per);
        require_numel(what, "k", k, batch * Ns_ * E);
        require_numel(what, "v", v, batch * Ns_ * E);
        if (k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type())
            assertion(what, ": operand dtypes differ: ", q.dtype(), ", ", k.dtype(), ", ", v.dtype());
        return {dtype_code(q), (int)batch, (int)E};
    }
    static void require_like(const char* what, const char* name, const Tensor& t, const Tensor& q) {
        require_numel(what, name, t, q.numel());
        if (t.scalar_type() != q.scalar_type()) assertion(what, ": operand dtypes differ: ", name, " is ", t.dtype());
    }
    void require_mask(const char* what, const std::optional<Tensor>& mask, int64_t nnz) const {
        if (!mask) return;
        require_numel(what, "mask", *mask, nnz * BH_ * BW_);
        require_bytes(what, *mask);
    }
    static void require_bytes(const char* what, const Tensor& mask) {
        if (mask.element_size() != 1) assertion(what, ": the element mask holds ", mask.dtype(), ", bytes are expected");
    }
    static void* contig(const Tensor& t) {
        if (!t.is_contiguous()) throw ValueFailure("sparta_amd kernels need contiguous tensors");
        return device_ptr(t);
    }
    const int32_t* rows() const { return (const int32_t*)device_ptr(row_ptr_); }
    const int32_t* entries() const { return (const int32_t*)device_ptr(bcsr_); }

    Tensor row_ptr_, bcsr_;
    std::optional<Tensor> col_ptr_, bcsc_, mask_;
    float inv_t_;
    int Nt_, Ns_, BH_, BW_;
};

Tensor seqlen_attention(const Tensor& q_in, const Tensor& k_in, const Tensor& v_in, const Tensor& lens_in) {
    py::gil_scoped_release nogil;
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    const Tensor q = q_in.contiguous(), k = k_in.contiguous(), v = v_in.contiguous(), lens = lens_in.contiguous();
    Tensor out = at::empty(q.sizes(), q.options());
    check_rc(spx_attention_seqlen_forward(dtype_code(q), device_ptr(q), device_ptr(k), device_ptr(v), out.data_ptr(),
                                          (const int32_t*)device_ptr(lens), 1.0f, (int)q.size(0), (int)q.size(1), (int)q.size(2),
                                          (int)q.size(3), 0, stream_of(q)), "spx_attention_seqlen_forward");
    return out;
}

// ---- mixture of experts ----------------------------------------------------------------------------
// Token index and gathered product of one call: (output, tile configuration that ran).  The caller
// has checked the sizes.
std::pair<Tensor, int> moe_forward(const Tensor& tokens_in, const Tensor& ids_in, const Tensor& weight_in, const Tensor& count, const Tensor& offset,
                   const Tensor& perm, const Tensor& workspace, int tile_cfg, bool strict) {
    py::gil_scoped_release nogil;
    at::AutoDispatchBelowADInplaceOrView below_autograd;
    const Tensor tokens = tokens_in.contiguous(), ids = ids_in.to(at::kInt).contiguous();
    const Tensor weight = weight_in.to(tokens.scalar_type()).contiguous();
    const int n_tok = (int)tokens.size(0), E = (int)weight.size(0), in = (int)weight.size(1), out_dim = (int)weight.size(2);
    const int32_t *off = (const int32_t*)device_ptr(offset), *pm = (const int32_t*)device_ptr(perm);
    check_rc(spx_moe_index((const int32_t*)device_ptr(ids), n_tok, E, (int32_t*)device_ptr(count), (int32_t*)off, (int32_t*)pm,
                           device_ptr(workspace), workspace.numel(), stream_of(tokens)), "spx_moe_index");
    Tensor out = at::empty({n_tok, out_dim}, tokens.options());
    int rc;
    while (true) {
        rc = spx_moe_forward(dtype_code(tokens), device_ptr(tokens), device_ptr(weight), 0, out.data_ptr(), off, pm, n_tok, in, out_dim, E,
                             tile_cfg, stream_of(tokens));
        if (rc == SPX_E_CONFIG && tile_cfg && !strict) {   // a tuned variant that does not take this dtype
            tile_cfg = 0;
            continue;
        }
        break;
    }
    check_rc(rc, "spx_moe_forward");
    return {out, tile_cfg};
}

// ---- index build -------------------------------------------------------------------------------------
// Buffers of several index builds and the launches that fill them.  A request: (mask as contiguous bytes,
// block height, block width, BCSR wanted, BCSC wanted, capacity or -1, scratch bytes).  An answer:
// (row_ptr, bcsr, row_order, col_ptr, bcsc, col_order, nnz), None where a format is not wanted.
typedef std::tuple<Tensor, int, int, bool, bool, int64_t, int64_t> IndexRequest;

std::vector<py::tuple> build_indexes(const std::vector<IndexRequest>& requests) {
    struct Built {
        std::optional<Tensor> row_ptr, bcsr, row_order, col_ptr, bcsc, col_order;
        Tensor nnz;
    };
    std::vector<Built> built(requests.size());
    if (!requests.empty()) {
        py::gil_scoped_release nogil;
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        const Tensor& first = std::get<0>(requests[0]);
        device_ptr(first);   // refuses CPU tensors
        c10::DeviceGuard guard(first.device());
        std::vector<spx_bcs_index_job> jobs(requests.size());
        // scratch of all builds, one after the other; given back when the call returns, in stream order
        std::vector<int64_t> scratch_at(requests.size());
        int64_t scratch_bytes = 0;
        for (size_t i = 0; i < requests.size(); ++i) {
            scratch_at[i] = scratch_bytes;
            scratch_bytes += (std::get<6>(requests[i]) + 255) / 256 * 256;
        }
        const Tensor scratch = at::empty({scratch_bytes}, first.options().dtype(at::kByte));
        for (size_t i = 0; i < requests.size(); ++i) {
            const auto& [mask, BH, BW, want_r, want_c, cap_in, ws_bytes] = requests[i];
            const int H = (int)mask.size(0), W = (int)mask.size(1), R = H / BH, C = W / BW;
            const int64_t cap = cap_in < 0 ? (int64_t)R * C : cap_in;
            const bool wide = want_r && want_c;   // int64 entries of the BCSC index
            Built& b = built[i];
            spx_bcs_index_job& job = jobs[i];
            job = spx_bcs_index_job();
            // An allocation to a tensor: they are saved, shared and kept one by one, and are of two types.  Straight from the allocator: the
            // dispatcher in front of it takes as long (two masks, host: 16.5 us through at::empty, 14.7 so).
            auto empty = [&](int64_t numel, at::ScalarType type) -> Tensor {
                return at::detail::empty_generic({numel}, scratch.storage().allocator(), c10::DispatchKeySet(c10::DispatchKey::CUDA), type, std::nullopt);
            };
            b.nnz = empty(1, at::kInt);
            if (want_r) {
                b.row_ptr = empty(R + 1, at::kInt);
                b.bcsr = empty(cap, at::kInt);
                b.row_order = empty(R, at::kInt);   // the launch orders of the matmul kernels
                job.row_ptr = (int32_t*)b.row_ptr->data_ptr();
                job.bcsr_idx = (int32_t*)b.bcsr->data_ptr();
                job.row_order = (int32_t*)b.row_order->data_ptr();
            }
            if (want_c) {
                b.col_ptr = empty(C + 1, at::kInt);
                b.bcsc = empty(cap, wide ? at::kLong : at::kInt);
                b.col_order = empty(C, at::kInt);   // come out of the same launch
                job.col_ptr = (int32_t*)b.col_ptr->data_ptr();
                job.bcsc_idx = b.bcsc->data_ptr();
                job.col_order = (int32_t*)b.col_order->data_ptr();
            }
            job.mask = (const uint8_t*)device_ptr(mask);
            job.H = H; job.W = W; job.BH = BH; job.BW = BW;
            job.bcsc_i64 = wide;
            job.nnz_dev = (int32_t*)b.nnz.data_ptr();
            job.cap = (int)cap;
            job.workspace = (char*)scratch.data_ptr() + scratch_at[i];
            job.workspace_bytes = (size_t)ws_bytes;
        }
        check_rc(spx_bcs_index_batch(jobs.data(), (int)jobs.size(), stream_of(first)), "spx_bcs_index_batch");
    }
    std::vector<py::tuple> out;
    for (Built& b : built) out.push_back(py::make_tuple(b.row_ptr, b.bcsr, b.row_order, b.col_ptr, b.bcsc, b.col_order, b.nnz));
    return out;
}

}  // namespace

PYBIND11_MODULE(_native, m) {
    m.doc() = "Native host path of the sparta_amd operators (csrc/native.cpp)";
    py::register_exception_translator([](std::exception_ptr p) {
        try {
            if (p) std::rethrow_exception(p);
        } catch (const AssertionFailure& e) {
            PyErr_SetString(PyExc_AssertionError, e.what());
        } catch (const ValueFailure& e) {
            PyErr_SetString(PyExc_ValueError, e.what());
        } catch (const AttributeFailure& e) {
            PyErr_SetString(PyExc_AttributeError, e.what());
        }
    });
    py::class_<MatmulKernel, std::shared_ptr<MatmulKernel>>(m, "MatmulKernel")
        .def(py::init<>())
        .def("bind", &MatmulKernel::bind)
        .def("unbind", &MatmulKernel::unbind)
        .def("set_strict", &MatmulKernel::set_strict)
        .def("__deepcopy__", [](const MatmulKernel& k, const py::object&) { return std::make_shared<MatmulKernel>(k); })
        .def("__call__", &MatmulKernel::call, py::arg("A"), py::arg("B"), py::arg("bias") = py::none());
    py::class_<MatmulStep>(m, "MatmulStep")
        .def_readonly("relu", &MatmulStep::relu)
        .def("forward", [](const MatmulStep& s, const Tensor& a, const Tensor& b, const std::optional<Tensor>& bias) {
            py::gil_scoped_release nogil;
            return s.forward(a, b, bias.has_value() ? &*bias : nullptr);
        })
        .def("gradients", [](const MatmulStep& s, const Tensor& grad, const Tensor& a, const Tensor& b,
                             const std::optional<Tensor>& gate, std::array<bool, 3> need, const std::vector<int64_t>& bias_shape) {
            py::gil_scoped_release nogil;
            return s.gradients(grad, a, b, gate.value_or(Tensor()), need, bias_shape);   // undefined: None
        });
    py::class_<MatmulOp>(m, "MatmulOp")
        .def(py::init<std::shared_ptr<MatmulKernel>, std::shared_ptr<MatmulKernel>, std::shared_ptr<MatmulKernel>, bool, bool, bool, bool,
                      py::object>())
        .def("step", &MatmulOp::step)
        .def("__call__", &MatmulOp::call, py::arg("A"), py::arg("B"), py::arg("bias") = py::none())
        .def("__deepcopy__", &MatmulOp::deepcopy);
    py::class_<SoftmaxKernel, std::shared_ptr<SoftmaxKernel>>(m, "SoftmaxKernel")
        .def(py::init<>())
        .def("bind", &SoftmaxKernel::bind)
        .def("unbind", &SoftmaxKernel::unbind)
        .def("set_strict", &SoftmaxKernel::set_strict)
        .def("__deepcopy__", [](const SoftmaxKernel& k, const py::object&) { return std::make_shared<SoftmaxKernel>(k); })
        .def("__call__", &SoftmaxKernel::forward, py::arg("x"), py::arg("T"))
        .def("__call__", &SoftmaxKernel::backward, py::arg("grad_y"), py::arg("y"), py::arg("T"));
    py::class_<SoftmaxStep>(m, "SoftmaxStep")
        .def("forward", [](const SoftmaxStep& s, const Tensor& x) {
            py::gil_scoped_release nogil;
            return s.forward(x);
        })
        .def("gradient", [](const SoftmaxStep& s, const Tensor& grad, const Tensor& y, const std::vector<int64_t>& x_shape) {
            py::gil_scoped_release nogil;
            return s.gradient(grad, y, x_shape);
        });
    py::class_<SoftmaxOp>(m, "SoftmaxOp")
        .def(py::init<std::shared_ptr<SoftmaxKernel>, std::shared_ptr<SoftmaxKernel>, double, py::object>())
        .def("set_temperature", &SoftmaxOp::set_temperature)
        .def("step", &SoftmaxOp::step)
        .def("__call__", &SoftmaxOp::call, py::arg("x"))
        .def("__deepcopy__", &SoftmaxOp::deepcopy);
    py::class_<AttentionKernel, std::shared_ptr<AttentionKernel>>(m, "AttentionKernel")
        .def(py::init<Tensor, Tensor, std::optional<Tensor>, std::optional<Tensor>, std::optional<Tensor>, double, int, int, int, int>())
        .def("forward", &AttentionKernel::forward)
        .def("forward_lse", &AttentionKernel::forward_lse)
        .def("live_mask", &AttentionKernel::live_mask)
        .def("backward_q", &AttentionKernel::backward_q, py::arg("grad_out"), py::arg("out"), py::arg("q"), py::arg("k"), py::arg("v"),
             py::arg("row_lse"), py::arg("mask") = py::none(), py::arg("nnz") = 0)
        .def("backward_kv", &AttentionKernel::backward_kv, py::arg("grad_out"), py::arg("q"), py::arg("k"), py::arg("v"), py::arg("row_lse"),
             py::arg("row_dot"), py::arg("mask") = py::none(), py::arg("nnz") = 0)
        .def("__deepcopy__", [](const AttentionKernel& k, const py::object&) { return std::make_shared<AttentionKernel>(k); });
    m.def("seqlen_attention", &seqlen_attention);
    m.def("moe_forward", &moe_forward);
    m.def("build_indexes", &build_indexes);
}
