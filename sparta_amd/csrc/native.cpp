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
#include <torch/csrc/autograd/functions/utils.h>
#include <c10/hip/HIPStream.h>

#include <atomic>
#include <memory>
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
        }
        at::AutoDispatchBelowADInplaceOrView below_autograd;
        const int code = dtype_code(a_in);
        const Tensor a = a_in.contiguous(), b = b_in.contiguous();
        Tensor bias;
        if (bias_in && bias_in->defined()) bias = bias_in->to(a.scalar_type()).contiguous();
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
        const int cfg = tile_cfg.load(std::memory_order_relaxed) & 0xffff;
        if (nnz_dev.has_value() || biased || (cfg != 0 && !colsum)) return 0;
        // the whole reduction is one or two stages deep: the block-row kernels of spx_matmul
        if (!trans_a && trans_b && K * (code == SPX_F32 ? 4 : 2) <= 256) return 0;
        return spx_matmul_split_workspace_bytes(code, trans_a, trans_b, nnz, batch, M, K, N, BM, BN, 0, colsum);
    }
    // `colsum` (may be null) receives the sums of op(A) over k.  Contiguous operands.
    Tensor run_split(int code, const Tensor& a, const Tensor& b, Tensor* colsum, size_t ws_bytes, at::IntArrayRef out_shape) const {
        Tensor c = compressed ? at::empty(out_shape, a.options()) : at::zeros(out_shape, a.options());
        Tensor ws = at::empty({(int64_t)ws_bytes}, a.options().dtype(at::kByte));
        check_rc(spx_matmul_split(code, trans_a, trans_b, compressed, device_ptr(a), device_ptr(b), c.data_ptr(),
                                  colsum ? device_ptr(*colsum) : nullptr, (const int32_t*)device_ptr(ptr),
                                  (const int32_t*)device_ptr(idx), nnz, sparse_stride, batch, M, K, N, BM, BN, 0,
                                  ws.data_ptr(), ws_bytes, stream_of(a)), "spx_matmul_split");
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
    bool gives_colsum() const { return mode == SPX_DDS && trans_a && !nnz_dev.has_value(); }

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

// C = op(A) op(B) (+ bias) with its gradients, as one autograd node.
struct MatmulBackward : public Node {
    MatmulPlanPtr fwd, bwd_a, bwd_b;    // the plans of the forward pass: its masks, its layout
    bool have_a, have_b;                // the operator was built with these kernels
    bool trans_a, trans_b, relu;
    SavedVariable a, b, gate;           // gate: the output, where a fused relu decided which gradients pass
    std::vector<int64_t> bias_shape;

    static void require_built(bool have, const MatmulPlanPtr& plan, const char* name) {
        if (!have) throw AttributeFailure(c10::str("the operator was built without its ", name, " kernel"));
        MatmulKernel::require_bound(plan);
    }
    variable_list apply(variable_list&& grads) override {
        return with_python_errors([&]() -> variable_list {
            variable_list out(num_outputs());
            if (!grads[0].defined()) return out;
            at::AutoGradMode no_grad(false);
            const Tensor A = a.unpack(), B = b.unpack();
            Tensor grad = grads[0].contiguous();
            if (relu) grad = at::threshold_backward(grad, gate.unpack(shared_from_this()), 0);
            if (task_should_compute_output(0)) {
                require_built(have_a, bwd_a, "backward_A");
                out[0] = trans_a ? bwd_a->run(B, grad, nullptr, A.sizes()) : bwd_a->run(grad, B, nullptr, A.sizes());
            }
            if (task_should_compute_output(1)) {
                require_built(have_b, bwd_b, "backward_B");
                if (num_outputs() > 2 && task_should_compute_output(2) && trans_b && !fwd->sparse_out() && bwd_b->gives_colsum()) {
                    Tensor bias_grad;
                    out[1] = bwd_b->run_with_colsum(grad, A, B.sizes(), &bias_grad);
                    out[2] = bias_grad.view(bias_shape);
                    return out;
                }
                out[1] = trans_b ? bwd_b->run(grad, A, nullptr, B.sizes()) : bwd_b->run(A, grad, nullptr, B.sizes());
            }
            if (num_outputs() > 2 && task_should_compute_output(2)) out[2] = fwd->bias_grad(grad, bias_shape);
            return out;
        });
    }
    void release_variables() override {
        a.reset_data();
        b.reset_data();
        gate.reset_data();
    }
    std::string name() const override { return "SparseMatmulBackward"; }
};

class MatmulOp {
public:
    MatmulOp(std::shared_ptr<MatmulKernel> fwd, std::shared_ptr<MatmulKernel> bwd_a, std::shared_ptr<MatmulKernel> bwd_b,
             bool trans_a, bool trans_b, bool relu, bool drop_batch)
        : fwd_(std::move(fwd)), bwd_a_(std::move(bwd_a)), bwd_b_(std::move(bwd_b)), trans_a_(trans_a), trans_b_(trans_b),
          relu_(relu), drop_batch_(drop_batch) {}

    Tensor call(const Tensor& a, const Tensor& b, const std::optional<Tensor>& bias) const {
        const MatmulPlanPtr p = fwd_->bound_plan();
        const MatmulPlanPtr pa = bwd_a_ ? bwd_a_->plan() : nullptr, pb = bwd_b_ ? bwd_b_->plan() : nullptr;
        py::gil_scoped_release nogil;
        const auto shape = p->shape();
        const Tensor* bias_p = bias.has_value() ? &*bias : nullptr;
        Tensor out = p->run(a, b, bias_p, drop_batch_ ? at::IntArrayRef(shape).slice(1) : at::IntArrayRef(shape));
        if (!records({&a, &b, bias_p})) return out;
        auto node = std::shared_ptr<MatmulBackward>(new MatmulBackward(), torch::autograd::deleteNode);
        node->set_next_edges(bias_p ? torch::autograd::collect_next_edges(a, b, *bias_p) : torch::autograd::collect_next_edges(a, b));
        node->fwd = p;
        node->bwd_a = pa;
        node->bwd_b = pb;
        node->have_a = (bool)bwd_a_;
        node->have_b = (bool)bwd_b_;
        node->trans_a = trans_a_;
        node->trans_b = trans_b_;
        node->relu = relu_;
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
        return std::make_unique<MatmulOp>(kernel(fwd_), kernel(bwd_a_), kernel(bwd_b_), trans_a_, trans_b_, relu_, drop_batch_);
    }

private:
    std::shared_ptr<MatmulKernel> fwd_, bwd_a_, bwd_b_;
    bool trans_a_, trans_b_, relu_, drop_batch_;
};

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
    py::class_<MatmulOp>(m, "MatmulOp")
        .def(py::init<std::shared_ptr<MatmulKernel>, std::shared_ptr<MatmulKernel>, std::shared_ptr<MatmulKernel>, bool, bool, bool, bool>())
        .def("__call__", &MatmulOp::call, py::arg("A"), py::arg("B"), py::arg("bias") = py::none())
        .def("__deepcopy__", &MatmulOp::deepcopy);
}
