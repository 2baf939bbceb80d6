// The operators' calls on torch tensors in native code: checks, allocation, launch and, where autograd records, the
// node of its graph.  Every function returns None for a call that is not the plain one (devices that differ, types,
// shapes or layouts that do not fit, wrapped tensors): the callers' general path takes it, which refuses it with
// its message or converts.  Host time of a call against the same steps in Python: a product 12.9 -> 7.5 us, a fresh
// operator with a product and both gradients 183 -> 70, a pattern of new points with its order check 39 -> 23.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <cstdlib>
#include <cstring>
#include <optional>
#include <vector>

#include "../../include/kernel_matmul_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

constexpr int64_t kBlock = 128;
constexpr int64_t kMaxBatchRank = 6;

// A dense tensor of this type on this device that is no wrapper of another.
bool is_plain(const Tensor& t, at::ScalarType type, c10::Device device) {
    return t.defined() && t.is_cuda() && t.device() == device && t.scalar_type() == type && t.layout() == at::kStrided &&
           !t.is_neg() && !t.is_conj() && t.has_storage() && !t.unsafeGetTensorImpl()->is_python_dispatch();
}

// The shapes of the kernel matrix' tensors, if they fit each other.
struct Matrix {
    int kernel;
    int64_t rank, m, n;
    const Tensor &x1, &x2, &params, &start, &end;

    Matrix(int64_t kernel_, const Tensor& x1_, const Tensor& x2_, const Tensor& params_, const Tensor& start_, const Tensor& end_)
        : kernel((int)kernel_), rank(-1), m(0), n(0), x1(x1_), x2(x2_), params(params_), start(start_), end(end_) {}

    c10::Device device() const { return x1.device(); }
    c10::IntArrayRef batch() const { return x1.sizes().slice(0, (size_t)rank); }

    // `trailing` dimensions behind the batch shape.
    bool has_batch(const Tensor& t, int64_t trailing) const {
        return t.dim() == rank + trailing && t.sizes().slice(0, (size_t)rank).equals(batch());
    }

    bool fits() {
        if (!x1.defined() || !x1.is_cuda() || x1.dim() < 1 || x1.dim() - 1 > kMaxBatchRank) {
            return false;
        }
        const c10::Device on = x1.device();
        if (!is_plain(x1, at::kFloat, on) || !is_plain(x2, at::kFloat, on) || !is_plain(params, at::kFloat, on) ||
            !is_plain(start, at::kInt, on) || !is_plain(end, at::kInt, on)) {
            return false;
        }
        rank = x1.dim() - 1;
        if (!has_batch(x2, 1) || !has_batch(params, 1) || !has_batch(start, 1) || !has_batch(end, 1)) {
            return false;
        }
        m = x1.size(-1);
        n = x2.size(-1);
        const int64_t blocks = (m + kBlock - 1) / kBlock;
        return params.size(-1) == km_num_params(kernel) && start.size(-1) == blocks && end.size(-1) == blocks;
    }

    bool has_vectors(const Tensor& t, int64_t rows) const {
        return is_plain(t, at::kFloat, device()) && has_batch(t, 2) && t.size(-2) == rows;
    }
};

template <class T>
const T* data(const Tensor& t) {
    return t.numel() > 0 ? static_cast<const T*>(t.data_ptr()) : nullptr;
}
const int64_t* strides(const Tensor& t) { return t.strides().data(); }

// The device of the launch is current while this lives; its stream.
class Launch {
  public:
    explicit Launch(c10::Device device) {
        if (c10::hip::current_device() != device.index()) {
            guard_.emplace(device);
        }
        stream_ = c10::hip::getCurrentHIPStream(device.index()).stream();
    }
    void* stream() const { return stream_; }

  private:
    std::optional<c10::DeviceGuard> guard_;
    hipStream_t stream_;
};

Tensor empty(c10::IntArrayRef sizes, const Tensor& like, at::ScalarType type = at::kFloat) {
    return at::empty(sizes, at::TensorOptions().dtype(type).device(like.device()));
}

std::vector<int64_t> shape(c10::IntArrayRef batch, std::initializer_list<int64_t> trailing) {
    std::vector<int64_t> s(batch.begin(), batch.end());
    s.insert(s.end(), trailing);
    return s;
}

void check(int status) { TORCH_CHECK(status == KM_OK, km_last_error()); }

Tensor workspace(size_t bytes, const Tensor& like) { return empty({(int64_t)(bytes > 0 ? bytes : 1)}, like, at::kByte); }

Tensor matmul(const Matrix& a, const Tensor& rhs, const km_launch_options* options, const Tensor* into) {
    Tensor out = into ? *into : empty(shape(a.batch(), {a.m, rhs.size(-1)}), a.x1);
    const size_t need = km_matmul_workspace_size(a.kernel, (int)a.rank, a.batch().data(), a.m, a.n, rhs.size(-1), options);
    Tensor scratch = need > 0 ? workspace(need, a.x1) : Tensor();
    Launch on(a.device());
    check(km_matmul_with_workspace(a.kernel, (int)a.rank, a.batch().data(), a.m, a.n, rhs.size(-1), data<float>(a.x1), strides(a.x1), data<float>(a.x2),
                    strides(a.x2), data<float>(rhs), strides(rhs), data<float>(a.params), strides(a.params), data<int32_t>(a.start),
                    strides(a.start), data<int32_t>(a.end), strides(a.end), const_cast<float*>(data<float>(out)), options,
                                   need > 0 ? scratch.data_ptr() : nullptr, need, on.stream()));
    return out;
}

Tensor param_grad(const Matrix& a, const Tensor& left, const Tensor& right, const Tensor* into) {
    Tensor grad = into ? *into : empty(shape(a.batch(), {a.params.size(-1)}), a.x1);
    const int64_t c = left.size(-1);
    const size_t need = km_param_grad_workspace_size(a.kernel, (int)a.rank, a.batch().data(), a.m, a.n, c);
    Tensor scratch = workspace(need, a.x1);
    Launch on(a.device());
    check(km_param_grad(a.kernel, (int)a.rank, a.batch().data(), a.m, a.n, c, data<float>(a.x1), strides(a.x1), data<float>(a.x2),
                        strides(a.x2), data<float>(left), strides(left), data<float>(right), strides(right), data<float>(a.params),
                        strides(a.params), data<int32_t>(a.start), strides(a.start), data<int32_t>(a.end), strides(a.end),
                        const_cast<float*>(data<float>(grad)), scratch.data_ptr(), need, on.stream()));
    return grad;
}

Tensor dense(const Matrix& a) {
    Tensor out = empty(shape(a.batch(), {a.m, a.n}), a.x1);
    Launch on(a.device());
    check(km_dense(a.kernel, (int)a.rank, a.batch().data(), a.m, a.n, data<float>(a.x1), strides(a.x1), data<float>(a.x2), strides(a.x2),
                   data<float>(a.params), strides(a.params), data<int32_t>(a.start), strides(a.start), data<int32_t>(a.end),
                   strides(a.end), const_cast<float*>(data<float>(out)), on.stream()));
    return out;
}

Tensor dense_bwd(const Matrix& a, const Tensor& out_grad) {
    Tensor grad = empty(shape(a.batch(), {a.params.size(-1)}), a.x1);
    const size_t need = km_param_grad_workspace_size(a.kernel, (int)a.rank, a.batch().data(), a.m, a.n, 0);
    Tensor scratch = workspace(need, a.x1);
    Launch on(a.device());
    check(km_dense_bwd(a.kernel, (int)a.rank, a.batch().data(), a.m, a.n, data<float>(a.x1), strides(a.x1), data<float>(a.x2),
                       strides(a.x2), data<float>(a.params), strides(a.params), data<int32_t>(a.start), strides(a.start),
                       data<int32_t>(a.end), strides(a.end), data<float>(out_grad), strides(out_grad),
                       const_cast<float*>(data<float>(grad)), scratch.data_ptr(), need, on.stream()));
    return grad;
}

bool fits_matrix(const Matrix& a, const Tensor& t) {
    return is_plain(t, at::kFloat, a.device()) && a.has_batch(t, 2) && t.size(-2) == a.m && t.size(-1) == a.n;
}

// Index tensors of one shape, one per batch dimension and row and column.
struct Indices {
    std::vector<Tensor> batch;
    Tensor row, col;

    bool fit(const Matrix& a) const {
        if ((int64_t)batch.size() != a.rank || !row.defined() || row.dim() < 1 || row.dim() > kMaxBatchRank + 1) {
            return false;
        }
        for (const Tensor& t : batch) {
            if (!is_plain(t, at::kInt, a.device()) || !t.sizes().equals(row.sizes())) {
                return false;
            }
        }
        return is_plain(row, at::kInt, a.device()) && is_plain(col, at::kInt, a.device()) && col.sizes().equals(row.sizes());
    }
};

struct BatchPointers {
    const int32_t* data[kMaxBatchRank];
    const int64_t* strides[kMaxBatchRank];
    explicit BatchPointers(const Indices& i) {
        for (size_t d = 0; d < i.batch.size(); d++) {
            data[d] = static_cast<const int32_t*>(i.batch[d].data_ptr());
            strides[d] = ::strides(i.batch[d]);
        }
    }
};

Tensor index(const Matrix& a, const Indices& i) {
    Tensor out = empty(i.row.sizes(), a.x1);
    const BatchPointers batch(i);
    Launch on(a.device());
    check(km_index(a.kernel, (int)a.rank, a.batch().data(), a.m, a.n, data<float>(a.x1), strides(a.x1), data<float>(a.x2), strides(a.x2),
                   data<float>(a.params), strides(a.params), data<int32_t>(a.start), strides(a.start), data<int32_t>(a.end),
                   strides(a.end), (int)i.row.dim(), i.row.sizes().data(), batch.data, batch.strides, data<int32_t>(i.row),
                   strides(i.row), data<int32_t>(i.col), strides(i.col), const_cast<float*>(data<float>(out)), on.stream()));
    return out;
}

Tensor index_bwd(const Matrix& a, const Indices& i, const Tensor& out_grad) {
    Tensor grad = empty(shape(a.batch(), {a.params.size(-1)}), a.x1);
    const size_t need = km_index_bwd_workspace_size(i.row.numel());
    Tensor scratch = workspace(need, a.x1);
    const BatchPointers batch(i);
    Launch on(a.device());
    check(km_index_bwd(a.kernel, (int)a.rank, a.batch().data(), a.m, a.n, data<float>(a.x1), strides(a.x1), data<float>(a.x2),
                       strides(a.x2), data<float>(a.params), strides(a.params), data<int32_t>(a.start), strides(a.start),
                       data<int32_t>(a.end), strides(a.end), (int)i.row.dim(), i.row.sizes().data(), batch.data, batch.strides,
                       data<int32_t>(i.row), strides(i.row), data<int32_t>(i.col), strides(i.col), data<float>(out_grad),
                       strides(out_grad), const_cast<float*>(data<float>(grad)), scratch.data_ptr(), need, on.stream()));
    return grad;
}

bool fits_indices(const Matrix& a, const Indices& i, const Tensor& t) {
    return is_plain(t, at::kFloat, a.device()) && t.sizes().equals(i.row.sizes());
}

// ---------------------------------------------------------------------------------------
// Nodes of the autograd graph, with the gradients of the autograd functions in linear_operator.py.  They are
// recorded for eager calls only; a transformed one (functorch, forward mode, tracing) keeps the Python functions.
// ---------------------------------------------------------------------------------------
struct MatmulNode : torch::autograd::Function<MatmulNode> {
    // The transpose has the same pattern (symmetric), or rhs needs no gradient.
    static Tensor forward(AutogradContext* ctx, const Tensor& x1, const Tensor& x2, const Tensor& rhs, const Tensor& params,
                          const Tensor& start, const Tensor& end, int64_t kernel) {
        ctx->save_for_backward({x1, x2, rhs, params, start, end});
        ctx->saved_data["kernel"] = kernel;
        Matrix a(kernel, x1, x2, params, start, end);
        TORCH_CHECK(a.fits(), "the kernel matrix' tensors do not fit each other");
        return matmul(a, rhs, nullptr, nullptr);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &x1 = saved[0], &x2 = saved[1], &rhs = saved[2], &params = saved[3], &start = saved[4], &end = saved[5];
        const int64_t kernel = ctx->saved_data["kernel"].toInt();
        const Tensor out_grad = grads[0].resolve_neg();
        variable_list result(7);
        Matrix a(kernel, x1, x2, params, start, end), transpose(kernel, x2, x1, params, start, end);
        TORCH_CHECK(a.fits() && a.has_vectors(out_grad, a.m) && out_grad.size(-1) == rhs.size(-1),
                    "the gradient of the product does not fit it");
        if (ctx->needs_input_grad(3)) {
            result[3] = param_grad(a, out_grad, rhs, nullptr);
        }
        if (ctx->needs_input_grad(2)) {
            TORCH_CHECK(transpose.fits(), "the pattern does not fit the transpose");
            result[2] = matmul(transpose, out_grad, nullptr, nullptr);
        }
        return result;
    }
};

struct DenseNode : torch::autograd::Function<DenseNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x1, const Tensor& x2, const Tensor& params, const Tensor& start,
                          const Tensor& end, int64_t kernel) {
        ctx->save_for_backward({x1, x2, params, start, end});
        ctx->saved_data["kernel"] = kernel;
        Matrix a(kernel, x1, x2, params, start, end);
        TORCH_CHECK(a.fits(), "the kernel matrix' tensors do not fit each other");
        return dense(a);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        Matrix a(ctx->saved_data["kernel"].toInt(), s[0], s[1], s[2], s[3], s[4]);
        const Tensor out_grad = grads[0].resolve_neg();
        TORCH_CHECK(a.fits() && fits_matrix(a, out_grad), "the gradient of the matrix does not fit it");
        variable_list result(6);
        result[2] = dense_bwd(a, out_grad);
        return result;
    }
};

struct IndexNode : torch::autograd::Function<IndexNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x1, const Tensor& x2, const Tensor& params, const Tensor& start,
                          const Tensor& end, int64_t kernel, const Tensor& row, const Tensor& col, at::TensorList batch) {
        variable_list saved = {x1, x2, params, start, end, row, col};
        saved.insert(saved.end(), batch.begin(), batch.end());
        ctx->save_for_backward(std::move(saved));
        ctx->saved_data["kernel"] = kernel;
        Matrix a(kernel, x1, x2, params, start, end);
        TORCH_CHECK(a.fits(), "the kernel matrix' tensors do not fit each other");
        return index(a, {batch.vec(), row, col});
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        Matrix a(ctx->saved_data["kernel"].toInt(), s[0], s[1], s[2], s[3], s[4]);
        const Indices i = {std::vector<Tensor>(s.begin() + 7, s.end()), s[5], s[6]};
        const Tensor out_grad = grads[0].resolve_neg();
        TORCH_CHECK(a.fits() && i.fit(a) && fits_indices(a, i, out_grad), "the gradient of the entries does not fit them");
        variable_list result(s.size() + 1);
        result[2] = index_bwd(a, i, out_grad);
        return result;
    }
};

// ---------------------------------------------------------------------------------------
// Python entry points.  Arguments: the kernel's number, then tensors in the operators' order.
// ---------------------------------------------------------------------------------------
// Modules take these from the environment; what they do then is the Python path's.
bool watched() {
    const char* debug = std::getenv("KERNEL_MATMUL_COMPILE_DEBUG");
    const char* sizes = std::getenv("KERNEL_MATMUL_COMPILE_PRINT_SIZE");
    return (debug && std::strcmp(debug, "true") == 0) || (sizes && std::strcmp(sizes, "true") == 0);
}

// (all that is asked of the interpreter is asked here, while its lock is held)
struct Arguments {
    PyObject* const* args;
    int64_t kernel;
    bool ok;

    Arguments(PyObject* const* args_, Py_ssize_t count, Py_ssize_t tensors, Py_ssize_t expected)
        : args(args_), kernel(-1), ok(count == expected && PyLong_Check(args_[0])) {
        if (ok) {
            int overflow = 0;
            kernel = PyLong_AsLongLongAndOverflow(args[0], &overflow);
            ok = overflow == 0 && km_num_params((int)kernel) > 0 && kernel == (int)kernel;
        }
        for (Py_ssize_t i = 1; ok && i <= tensors; i++) {
            ok = THPVariable_Check(args[i]);
        }
    }
    const Tensor& operator[](Py_ssize_t i) const { return THPVariable_Unpack(args[i]); }
};

PyObject* none() { Py_RETURN_NONE; }

template <class F>
PyObject* launched(F&& f) {
    Tensor out;
    {
        pybind11::gil_scoped_release no_gil;
        out = f();
    }
    return THPVariable_Wrap(std::move(out));
}

// A tensor that the result goes into, if it is one that it fits (null: none given); false if it does not fit.
bool result_tensor(PyObject* object, const Matrix& a, std::initializer_list<int64_t> trailing, const Tensor** out) {
    *out = nullptr;
    if (object == Py_None) {
        return true;
    }
    if (!THPVariable_Check(object)) {
        return false;
    }
    const Tensor& t = THPVariable_Unpack(object);
    *out = &t;
    return is_plain(t, at::kFloat, a.device()) && t.is_contiguous() && t.sizes().equals(shape(a.batch(), trailing));
}

// matmul(kernel, x1, x2, rhs, params, start, end, options' address or None, out or None)
PyObject* py_matmul(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Arguments t(args, count, 6, 9);
    if (!t.ok) {
        return none();
    }
    Matrix a(t.kernel, t[1], t[2], t[4], t[5], t[6]);
    const Tensor& rhs = t[3];
    const Tensor* into;
    if (!a.fits() || !a.has_vectors(rhs, a.n) || !result_tensor(args[8], a, {a.m, rhs.size(-1)}, &into)) {
        return none();
    }
    const auto* options = args[7] == Py_None ? nullptr : static_cast<const km_launch_options*>(PyLong_AsVoidPtr(args[7]));
    return launched([&] { return matmul(a, rhs, options, into); });
    END_HANDLE_TH_ERRORS
}

// matmul_recorded(kernel, x1, x2, rhs, params, start, end): for a symmetric pattern, or rhs without gradient
PyObject* py_matmul_recorded(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Arguments t(args, count, 6, 7);
    if (!t.ok || watched()) {
        return none();
    }
    Matrix a(t.kernel, t[1], t[2], t[4], t[5], t[6]);
    if (!a.fits() || !a.has_vectors(t[3], a.n)) {
        return none();
    }
    return launched([&] { return MatmulNode::apply(t[1], t[2], t[3], t[4], t[5], t[6], t.kernel); });
    END_HANDLE_TH_ERRORS
}

// param_grad(kernel, x1, x2, left, right, params, start, end, out or None)
PyObject* py_param_grad(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Arguments t(args, count, 7, 9);
    if (!t.ok) {
        return none();
    }
    Matrix a(t.kernel, t[1], t[2], t[5], t[6], t[7]);
    const Tensor &left = t[3], &right = t[4];
    const Tensor* into;
    if (!a.fits() || !a.has_vectors(left, a.m) || !a.has_vectors(right, a.n) || left.size(-1) != right.size(-1) ||
        !result_tensor(args[8], a, {a.params.size(-1)}, &into)) {
        return none();
    }
    return launched([&] { return param_grad(a, left, right, into); });
    END_HANDLE_TH_ERRORS
}

// dense(kernel, x1, x2, params, start, end)
template <bool RECORD>
PyObject* py_dense(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Arguments t(args, count, 5, 6);
    if (!t.ok || (RECORD && watched())) {
        return none();
    }
    Matrix a(t.kernel, t[1], t[2], t[3], t[4], t[5]);
    if (!a.fits()) {
        return none();
    }
    return launched([&] { return RECORD ? DenseNode::apply(t[1], t[2], t[3], t[4], t[5], t.kernel) : dense(a); });
    END_HANDLE_TH_ERRORS
}

// dense_bwd(kernel, x1, x2, params, start, end, out_grad)
PyObject* py_dense_bwd(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Arguments t(args, count, 6, 7);
    if (!t.ok) {
        return none();
    }
    Matrix a(t.kernel, t[1], t[2], t[3], t[4], t[5]);
    if (!a.fits() || !fits_matrix(a, t[6])) {
        return none();
    }
    return launched([&] { return dense_bwd(a, t[6]); });
    END_HANDLE_TH_ERRORS
}

bool read_indices(PyObject* batch, const Tensor& row, const Tensor& col, Indices* i) {
    if (!PyTuple_Check(batch)) {
        return false;
    }
    for (Py_ssize_t d = 0; d < PyTuple_GET_SIZE(batch); d++) {
        PyObject* item = PyTuple_GET_ITEM(batch, d);
        if (!THPVariable_Check(item)) {
            return false;
        }
        i->batch.push_back(THPVariable_Unpack(item));
    }
    i->row = row;
    i->col = col;
    return true;
}

// index(kernel, x1, x2, params, start, end, row, col, tuple of batch indices)
template <bool RECORD>
PyObject* py_index(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Arguments t(args, count, 7, 9);
    if (!t.ok || (RECORD && watched())) {
        return none();
    }
    Matrix a(t.kernel, t[1], t[2], t[3], t[4], t[5]);
    Indices i;
    if (!a.fits() || !read_indices(args[8], t[6], t[7], &i) || !i.fit(a)) {
        return none();
    }
    return launched([&] {
        return RECORD ? IndexNode::apply(t[1], t[2], t[3], t[4], t[5], t.kernel, i.row, i.col, at::TensorList(i.batch)) : index(a, i);
    });
    END_HANDLE_TH_ERRORS
}

// index_bwd(kernel, x1, x2, params, start, end, row, col, out_grad, tuple of batch indices)
PyObject* py_index_bwd(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    const Arguments t(args, count, 8, 10);
    if (!t.ok) {
        return none();
    }
    Matrix a(t.kernel, t[1], t[2], t[3], t[4], t[5]);
    Indices i;
    if (!a.fits() || !read_indices(args[9], t[6], t[7], &i) || !i.fit(a) || !fits_indices(a, i, t[8])) {
        return none();
    }
    return launched([&] { return index_bwd(a, i, t[8]); });
    END_HANDLE_TH_ERRORS
}

// views(x1, x2, start, end, batch shape): coordinates [..., 1] without gradient and last dimension, and the pattern, as
// stride-0 views of the batch shape.
PyObject* py_views(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 5 || !PyTuple_Check(args[4])) {
        return none();
    }
    std::vector<int64_t> sizes;
    for (Py_ssize_t d = 0; d < PyTuple_GET_SIZE(args[4]); d++) {
        sizes.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(args[4], d)));
    }
    sizes.push_back(0);
    PyObject* result = PyTuple_New(4);
    if (!result) {
        return nullptr;
    }
    pybind11::object owner = pybind11::reinterpret_steal<pybind11::object>(result);
    for (int i = 0; i < 4; i++) {
        if (!THPVariable_Check(args[i])) {
            return none();
        }
        Tensor t = THPVariable_Unpack(args[i]);
        if (i < 2) {
            if (i == 1 && args[1] == args[0]) {
                Py_INCREF(PyTuple_GET_ITEM(result, 0));
                PyTuple_SET_ITEM(result, 1, PyTuple_GET_ITEM(result, 0));
                continue;
            }
            t = t.detach().squeeze(-1);
        }
        sizes.back() = t.size(-1);
        PyTuple_SET_ITEM(result, i, THPVariable_Wrap(t.sizes().equals(sizes) ? t : t.expand(sizes)));
    }
    return owner.release().ptr();
    END_HANDLE_TH_ERRORS
}

// Waits for what was launched, also where a later step throws: the host's memory that it writes is given back then.
class Settled {
  public:
    explicit Settled(void* stream) : stream_(static_cast<hipStream_t>(stream)) {}
    ~Settled() {
        if (!done_) {
            (void)hipStreamSynchronize(stream_);
        }
    }
    hipError_t wait() {
        done_ = true;
        return hipStreamSynchronize(stream_);
    }

  private:
    hipStream_t stream_;
    bool done_ = false;
};

// make_ranges(cutoff, x1, x2 or None, block size, align) -> (start, end) of contiguous float32 device tensors [n] or
// [batch, n] that ascend; None for all others.  The check's words are written to host memory, and one wait covers check
// and builder.
PyObject* py_make_ranges(PyObject*, PyObject* const* args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 5 || !PyFloat_Check(args[0]) || !THPVariable_Check(args[1]) || !PyLong_Check(args[3]) || !PyBool_Check(args[4])) {
        return none();
    }
    const float cutoff = (float)PyFloat_AS_DOUBLE(args[0]);
    const Tensor& x1 = THPVariable_Unpack(args[1]);
    const bool symmetric = args[2] == Py_None;
    if (!symmetric && !THPVariable_Check(args[2])) {
        return none();
    }
    const Tensor& x2 = symmetric ? x1 : THPVariable_Unpack(args[2]);
    int overflow = 0;
    const int64_t block = PyLong_AsLongLongAndOverflow(args[3], &overflow);  // (-1 where it does not fit)
    const bool align = args[4] == Py_True;
    if (!x1.is_cuda() || !is_plain(x1, at::kFloat, x1.device()) || !is_plain(x2, at::kFloat, x1.device()) || !x1.is_contiguous() ||
        !x2.is_contiguous() || x1.dim() < 1 || x1.dim() > 2 || x2.dim() != x1.dim() || x1.numel() == 0 || x2.numel() == 0 ||
        block < 1 || block > INT32_MAX || (x1.dim() == 2 && x1.size(0) != x2.size(0))) {
        return none();
    }
    const int64_t batch = x1.dim() == 2 ? x1.size(0) : 1, n1 = x1.size(-1), n2 = x2.size(-1);
    Tensor start, end;
    bool ascending = true;
    {
        pybind11::gil_scoped_release no_gil;
        const std::vector<int64_t> sizes = shape(x1.sizes().slice(0, x1.dim() - 1), {(n1 + block - 1) / block});
        start = empty(sizes, x1, at::kInt);
        end = empty(sizes, x1, at::kInt);
        Tensor words = at::empty({KM_SORTED_FLAGS}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
        int32_t* descents = static_cast<int32_t*>(words.data_ptr());
        Launch on(x1.device());
        Settled settled(on.stream());
        int32_t *s = static_cast<int32_t*>(start.data_ptr()), *e = static_cast<int32_t*>(end.data_ptr());
        if (symmetric) {
            check(km_check_sorted_device(data<float>(x1), batch, n1, nullptr, 0, 0, descents, on.stream()));
            check(km_make_ranges_symmetric_device(data<float>(x1), batch, n1, cutoff, (int)block, s, e, on.stream()));
        } else {
            check(km_make_ranges_checked_device(data<float>(x1), data<float>(x2), batch, n1, n2, cutoff, (int)block, align, s, e,
                                                descents, on.stream()));
        }
        const hipError_t error = settled.wait();
        TORCH_CHECK(error == hipSuccess, "make_ranges: ", hipGetErrorString(error));
        for (int i = 0; i < KM_SORTED_FLAGS; i++) {
            ascending = ascending && descents[i] == 0;
        }
    }
    if (!ascending) {
        return none();
    }
    pybind11::object first = pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(start));
    pybind11::object second = pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(end));
    return PyTuple_Pack(2, first.ptr(), second.ptr());
    END_HANDLE_TH_ERRORS
}

PyObject* py_watched(PyObject*, PyObject* const*, Py_ssize_t) { return PyBool_FromLong(watched()); }

#define KM_METHOD(name, function) {name, (PyCFunction)(void (*)(void))(function), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    KM_METHOD("matmul", py_matmul),
    KM_METHOD("matmul_recorded", py_matmul_recorded),
    KM_METHOD("param_grad", py_param_grad),
    KM_METHOD("dense", py_dense<false>),
    KM_METHOD("dense_recorded", py_dense<true>),
    KM_METHOD("dense_bwd", py_dense_bwd),
    KM_METHOD("index", py_index<false>),
    KM_METHOD("index_recorded", py_index<true>),
    KM_METHOD("index_bwd", py_index_bwd),
    KM_METHOD("views", py_views),
    KM_METHOD("watched", py_watched),
    KM_METHOD("make_ranges", py_make_ranges),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_km_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__km_torch(void) { return PyModule_Create(&module); }
