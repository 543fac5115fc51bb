// The host path of the operators in C++: argument checks, allocations and the calls into libnq_gfx950.so.
//
// A decode call of a small linear takes 7 us on the GPU and a prefill group of a decoder layer 100; checked, allocated
// and launched from Python they took 20 us and 28 us per group of the host.  This file registers the device implementations
// of torch.ops.binary_kernels.* (schemas and shape-only implementations are in ops.py) and is the extension module
// nanoquant_amd._host for the calls beyond the operators.  It holds no state, and allocates and launches without the interpreter
// lock: a launch waits while the stream's queue is full, maybe for a host function that needs the lock.
//
// Checks and messages are those of the reference's host wrappers:
//   nanoquant_dyn_forward     src/nanoquant/kernel/cuda/gemv_kernel.cu:308-346, cuda/meta_utils.h:14-38
//   marlin_onebit_forward     src/nanoquant/kernel/cuda/gemm.cpp:36-98
//   marlin_nanoquant_forward  src/nanoquant/kernel/cuda/gemm.cpp:112-122
#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>

#include <algorithm>
#include <array>
#include <initializer_list>
#include <numeric>
#include <string>
#include <vector>

#include "../../include/nq_gfx950.h"

namespace py = pybind11;
using at::Tensor;
using MaybeTensor = std::optional<Tensor>;

namespace {

constexpr int64_t kMarlinMinMaxPar = 32;

// A status of the C ABI as the exception that the reference's wrappers raise.
void check_status(int status) {
    if (status == NQ_OK) return;
    std::string msg = nq_status_string(status);
    if (status == NQ_ERR_HIP) msg += " (hipError " + std::to_string(nq_last_hip_error()) + ")";
    TORCH_CHECK(false, msg);
}

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
const void* data(const Tensor& t) { return t.const_data_ptr(); }
const void* data(const MaybeTensor& t) { return t ? t->const_data_ptr() : nullptr; }
Tensor empty(std::initializer_list<int64_t> sizes, const Tensor& like) {
    return Tensor(at::detail::empty_cuda(at::IntArrayRef(sizes.begin(), sizes.size()), like.scalar_type(), like.device(), std::nullopt));
}
std::string sizes_text(const Tensor& t) {
    std::string s = "[";
    for (int64_t i = 0; i < t.dim(); ++i) s += (i ? ", " : "") + std::to_string(t.size(i));
    return s + "]";
}

// ---- decode -----------------------------------------------------------------------------------
void check_dev_cont(const Tensor& t, const char* name, at::ScalarType dtype, const char* what) {
    TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
    TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
    TORCH_CHECK(t.scalar_type() == dtype, name, " ", what);
}

struct GemvDims {
    int64_t n, r, m;
};

GemvDims check_gemv_args(const Tensor& x, const Tensor& scale_g, const Tensor& Ubits, const MaybeTensor& scale_l, const Tensor& Vbits,
                         const Tensor& scale_h) {
    const auto dt = x.scalar_type();
    TORCH_CHECK(dt == at::kHalf || dt == at::kBFloat16, "Support only Half or BFloat16");
    const char* what = dt == at::kHalf ? "must be float16 tensor" : "must be bfloat16 tensor";
    check_dev_cont(x, "x", dt, what);
    check_dev_cont(scale_g, "scale_g", dt, what);
    check_dev_cont(scale_h, "scale_h", dt, what);
    check_dev_cont(Ubits, "Ubits", at::kInt, "tensor dtype must be int32");
    check_dev_cont(Vbits, "Vbits", at::kInt, "tensor dtype must be int32");
    if (scale_l) {
        check_dev_cont(*scale_l, "(*scale_l)", dt, what);
        TORCH_CHECK(scale_l->size(0) == Ubits.size(0), "scale_l size mismatch");
    }
    TORCH_CHECK(x.dim() >= 1, "x must have at least one dimension");
    const GemvDims d{x.size(-1), Ubits.size(0), scale_h.size(0)};
    // The reference trusts these and indexes out of bounds otherwise; the launch needs them to hold.
    TORCH_CHECK(Ubits.dim() == 2 && Vbits.dim() == 2, "Ubits and Vbits must be 2-D packed word matrices");
    TORCH_CHECK(Ubits.size(1) == (d.n + 31) / 32, "Ubits has ", Ubits.size(1), " words per row, expected ", (d.n + 31) / 32, " for ", d.n,
                " input columns");
    TORCH_CHECK(scale_g.numel() == d.n, "scale_g size mismatch");
    TORCH_CHECK(Vbits.size(0) == d.m && Vbits.size(1) == (d.r + 31) / 32, "Vbits must be [", d.m, ", ", (d.r + 31) / 32, "], got ",
                sizes_text(Vbits));
    return d;
}

void check_bias(const MaybeTensor& bias, int64_t m, const Tensor& x) {
    if (!bias) return;
    check_dev_cont(*bias, "bias", x.scalar_type(), "Bias");
    TORCH_CHECK(bias->dim() == 1 && bias->size(0) == m, "bias must be [", m, "], got ", sizes_text(*bias));
}

int dtype_id(const Tensor& x) { return x.scalar_type() == at::kHalf ? NQ_F16 : NQ_BF16; }

Tensor gemv_launch(const GemvDims& d, const Tensor& x, const Tensor& scale_g, const Tensor& Ubits, const MaybeTensor& scale_l,
                   const Tensor& Vbits, const Tensor& scale_h, const MaybeTensor& bias) {
    const auto shape = x.sizes();
    const int64_t batch = std::accumulate(shape.begin(), shape.end() - 1, (int64_t)1, std::multiplies<int64_t>());
    const c10::DeviceGuard guard(x.device());
    Tensor y = empty({batch, d.m}, x);
    if (batch > 0 && d.m > 0) {
        const Tensor h(at::detail::empty_cuda({batch, std::max<int64_t>(d.r, 1)}, at::kFloat, x.device(), std::nullopt));
        check_status(nq_gemv_forward_bias(data(x), data(scale_g), (const uint32_t*)data(Ubits), data(scale_l), (const uint32_t*)data(Vbits),
                                          data(scale_h), data(bias), (float*)h.mutable_data_ptr(), y.mutable_data_ptr(), (int)batch, (int)d.n,
                                          (int)d.r, (int)d.m, dtype_id(x), stream_of(x)));
    }
    if (x.dim() == 2) return y;
    std::vector<int64_t> out(shape.begin(), shape.end());
    out.back() = d.m;
    return y.reshape(out);
}

Tensor gemv_bias(const Tensor& x, const Tensor& scale_g, const Tensor& Ubits, const MaybeTensor& scale_l, const Tensor& Vbits,
                 const Tensor& scale_h, const MaybeTensor& bias) {
    const GemvDims d = check_gemv_args(x, scale_g, Ubits, scale_l, Vbits, scale_h);
    check_bias(bias, d.m, x);
    return gemv_launch(d, x, scale_g, Ubits, scale_l, Vbits, scale_h, bias);
}

// Legal values of the CUDA tuning hints (gemv_kernel.cu:351-354).  They select template instances in the reference; here they
// are validated and otherwise ignored.  4 is added to the accumulator set because it is the schema's own default.
void check_hint(const char* name, int64_t value, std::initializer_list<int64_t> legal) {
    if (std::find(legal.begin(), legal.end(), value) != legal.end()) return;
    std::string choices;
    for (int64_t v : legal) choices += (choices.empty() ? "" : ", ") + std::to_string(v);
    TORCH_CHECK_VALUE(false, name, " should be one of [", choices, "], but ", value, " was given");
}
void check_hint_by_name(const std::string& name, int64_t value) {
    const std::string kind = name.substr(0, name.find_last_not_of("12") + 1);
    if (kind == "n_th") check_hint(name.c_str(), value, {64, 128, 256});
    else if (kind == "n_rpw") check_hint(name.c_str(), value, {1, 2, 4, 8});
    else if (kind == "n_acc") check_hint(name.c_str(), value, {1, 2, 4});
    else if (kind == "n_pipe") check_hint(name.c_str(), value, {1, 2, 4, 8, 16});
    else TORCH_CHECK_VALUE(false, "unknown tuning hint ", name);
}

Tensor nanoquant_dyn_forward(const Tensor& x, const Tensor& scale_g, const Tensor& Ubits, const MaybeTensor& scale_l, const Tensor& Vbits,
                             const Tensor& scale_h, int64_t th1, int64_t th2, int64_t rpw1, int64_t rpw2, int64_t acc1, int64_t acc2,
                             int64_t pipe1, int64_t pipe2) {
    const GemvDims d = check_gemv_args(x, scale_g, Ubits, scale_l, Vbits, scale_h);
    check_hint("n_th1", th1, {64, 128, 256});
    check_hint("n_rpw1", rpw1, {1, 2, 4, 8});
    check_hint("n_acc1", acc1, {1, 2, 4});
    check_hint("n_pipe1", pipe1, {1, 2, 4, 8, 16});
    check_hint("n_th2", th2, {64, 128, 256});
    check_hint("n_rpw2", rpw2, {1, 2, 4, 8});
    check_hint("n_acc2", acc2, {1, 2, 4});
    check_hint("n_pipe2", pipe2, {1, 2, 4, 8, 16});
    return gemv_launch(d, x, scale_g, Ubits, scale_l, Vbits, scale_h, std::nullopt);
}

// ---- prefill ----------------------------------------------------------------------------------
// marlin_onebit_check_and_alloc (gemm.cpp:36-56) for k input columns: the rows of the matrix.
int64_t onebit_check(int64_t k, const Tensor& B, const MaybeTensor& s_in, const MaybeTensor& s_out, const Tensor& workspace) {
    const int64_t rows = B.size(1) * 2;
    TORCH_CHECK(k == B.size(0) * 16, "k dimension mismatch");
    TORCH_CHECK(!s_in || s_in->size(0) == k, "s_in size mismatch");
    TORCH_CHECK(!s_out || s_out->size(0) == rows, "s_out size mismatch");
    TORCH_CHECK(workspace.numel() >= rows / 128 * kMarlinMinMaxPar, "workspace too small");
    return rows;
}

int gemm_dtype(const Tensor& A) {
    if (A.scalar_type() == at::kHalf) return NQ_F16;
    if (A.scalar_type() == at::kBFloat16) return NQ_BF16;
    TORCH_CHECK(false, "Unsupported dtype: Marlin only supports Half and BFloat16");
}

void check_gemm_tensor(const Tensor& t, const char* name, at::ScalarType dtype) {
    TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
    TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
    if (t.scalar_type() != dtype) {
        const char* text = dtype == at::kInt ? "torch.int32" : dtype == at::kHalf ? "torch.float16" : "torch.bfloat16";
        TORCH_CHECK(false, name, " must have dtype ", text);
    }
}
void check_gemm_scale(const MaybeTensor& t, const char* name, const Tensor& x) {
    if (t) check_gemm_tensor(*t, name, x.scalar_type());
}

Tensor marlin_onebit_forward(const Tensor& x, const Tensor& weight, const MaybeTensor& scale_g, const MaybeTensor& scale_h,
                             const Tensor& workspace) {
    const int dt = gemm_dtype(x);
    const int64_t tokens = x.size(0), k = x.size(1), rows = onebit_check(k, weight, scale_g, scale_h, workspace);
    check_gemm_tensor(x, "x", x.scalar_type());
    check_gemm_tensor(weight, "weight", at::kInt);
    check_gemm_scale(scale_g, "scale_g", x);
    check_gemm_scale(scale_h, "scale_h", x);
    const c10::DeviceGuard guard(x.device());
    Tensor y = empty({tokens, rows}, x);
    if (tokens > 0 && rows > 0)
        check_status(nq_gemm_onebit(data(x), (const uint32_t*)data(weight), data(scale_g), data(scale_h), y.mutable_data_ptr(), nullptr, 0,
                                    (int)tokens, (int)k, (int)rows, dt, stream_of(x)));
    return y;
}

// The operands of one linear, checked; r and m of its factors.
struct GemmDims {
    int64_t tokens, n, r, m;
};
GemmDims check_gemm_args(const Tensor& x, const Tensor& weight_u, const Tensor& weight_v, const MaybeTensor& scale_g,
                         const MaybeTensor& scale_l, const MaybeTensor& scale_h, const Tensor& workspace, const MaybeTensor& bias) {
    GemmDims d;
    d.tokens = x.size(0);
    d.n = x.size(1);
    d.r = onebit_check(d.n, weight_u, scale_g, scale_l, workspace);
    check_gemm_tensor(x, "x", x.scalar_type());
    check_gemm_tensor(weight_u, "weight_u", at::kInt);
    check_gemm_tensor(weight_v, "weight_v", at::kInt);
    check_gemm_scale(scale_g, "scale_g", x);
    check_gemm_scale(scale_l, "scale_l", x);
    check_gemm_scale(scale_h, "scale_h", x);
    d.m = onebit_check(d.r, weight_v, std::nullopt, scale_h, workspace);
    check_bias(bias, d.m, x);
    return d;
}

Tensor gemm_bias(const Tensor& x, const Tensor& weight_u, const Tensor& weight_v, const MaybeTensor& scale_g, const MaybeTensor& scale_l,
                 const MaybeTensor& scale_h, const Tensor& workspace, const MaybeTensor& bias) {
    const int dt = gemm_dtype(x);
    const GemmDims d = check_gemm_args(x, weight_u, weight_v, scale_g, scale_l, scale_h, workspace, bias);
    const c10::DeviceGuard guard(x.device());
    Tensor y = empty({d.tokens, d.m}, x);
    if (d.tokens > 0 && d.m > 0) {
        const Tensor h = empty({d.tokens, d.r}, x);
        check_status(nq_gemm_nanoquant_bias(data(x), (const uint32_t*)data(weight_u), (const uint32_t*)data(weight_v), data(scale_g),
                                            data(scale_l), data(scale_h), data(bias), h.mutable_data_ptr(), y.mutable_data_ptr(), nullptr, 0,
                                            (int)d.tokens, (int)d.n, (int)d.r, (int)d.m, dt, stream_of(x)));
    }
    return y;
}

Tensor marlin_nanoquant_forward(const Tensor& x, const Tensor& weight_u, const Tensor& weight_v, const MaybeTensor& scale_g,
                                const MaybeTensor& scale_l, const MaybeTensor& scale_h, const Tensor& workspace) {
    return gemm_bias(x, weight_u, weight_v, scale_g, scale_l, scale_h, workspace, std::nullopt);
}

// ---- groups: Python lists of tensors ------------------------------------------------------------
Tensor tensor_of(PyObject* o, const char* what) {
    TORCH_CHECK_TYPE(THPVariable_Check(o), what, " must be a tensor");
    return THPVariable_Unpack(o);
}
MaybeTensor maybe_tensor_of(PyObject* o, const char* what) {
    if (o == Py_None) return std::nullopt;
    return tensor_of(o, what);
}

struct GroupTerm {
    Tensor x, weight_u, weight_v, workspace, h;
    MaybeTensor scale_g, scale_l, scale_h, bias;
    GemmDims d;
};

// Checks term i of a group against the first one; `term` is the operator's argument tuple behind x.
GroupTerm group_term(const Tensor& x, const Tensor& x0, PyObject* term, PyObject* bias) {
    GroupTerm t;
    const py::tuple f = py::reinterpret_borrow<py::object>(term);
    TORCH_CHECK_VALUE(f.size() == 6, "a term is (weight_u, weight_v, scale_g, scale_l, scale_h, workspace)");
    t.x = x;
    t.weight_u = tensor_of(f[0].ptr(), "weight_u");
    t.weight_v = tensor_of(f[1].ptr(), "weight_v");
    t.scale_g = maybe_tensor_of(f[2].ptr(), "scale_g");
    t.scale_l = maybe_tensor_of(f[3].ptr(), "scale_l");
    t.scale_h = maybe_tensor_of(f[4].ptr(), "scale_h");
    t.workspace = tensor_of(f[5].ptr(), "workspace");
    t.bias = maybe_tensor_of(bias, "bias");
    TORCH_CHECK(x.scalar_type() == x0.scalar_type() && x.dim() == 2 && x.size(0) == x0.size(0) && x.device() == x0.device(),
                "all inputs of a group must be 2-D with the same token count, dtype and device");
    t.d = check_gemm_args(x, t.weight_u, t.weight_v, t.scale_g, t.scale_l, t.scale_h, t.workspace, t.bias);
    return t;
}

std::vector<nq_gemm_term> terms_of(const std::vector<GroupTerm>& terms, const std::vector<void*>& y) {
    std::vector<nq_gemm_term> arr;
    arr.reserve(terms.size());
    for (size_t i = 0; i < terms.size(); ++i) {
        const GroupTerm& t = terms[i];
        arr.push_back({data(t.x), (const uint32_t*)data(t.weight_u), (const uint32_t*)data(t.weight_v), data(t.scale_g), data(t.scale_l),
                       data(t.scale_h), data(t.bias), t.h.mutable_data_ptr(), y[i], (int)t.d.n, (int)t.d.r, (int)t.d.m});
    }
    return arr;
}

// The workspace of the panel launches, panel_ws() (None: there is none now), asked for only where a stage takes one.  Without the
// interpreter lock.
MaybeTensor panel_workspace(const nq_gemm_term* terms, int count, int64_t tokens, int panel_mode, const py::object& panel_ws) {
    if (panel_mode == NQ_PANEL_NEVER || !nq_gemm_group_wants_panel(terms, count, (int)tokens, panel_mode)) return std::nullopt;
    const py::gil_scoped_acquire lock;
    return maybe_tensor_of(panel_ws().ptr(), "the panel workspace");
}

// The launches of checked terms; y: one output address per term.  Without the interpreter lock.
void launch_group_terms(const std::vector<GroupTerm>& terms, const std::vector<void*>& y, int dt, int panel_mode, const py::object& panel_ws) {
    const int64_t tokens = terms[0].d.tokens;
    const int most = nq_gemm_group_max();
    const std::vector<nq_gemm_term> arr = terms_of(terms, y);
    for (size_t lo = 0; lo < arr.size(); lo += most) {
        const int count = (int)std::min<size_t>(most, arr.size() - lo);
        const MaybeTensor ws = panel_workspace(arr.data() + lo, count, tokens, panel_mode, panel_ws);
        check_status(nq_gemm_nanoquant_group_ws(arr.data() + lo, count, (int)tokens, dt, nullptr, 0, ws ? ws->mutable_data_ptr() : nullptr,
                                                ws ? (size_t)ws->nbytes() : 0, panel_mode, stream_of(terms[0].x)));
    }
}

std::vector<Tensor> tensors_of(const py::sequence& s, const char* what) {
    std::vector<Tensor> out;
    out.reserve(s.size());
    for (const auto& o : s) out.push_back(tensor_of(o.ptr(), what));
    return out;
}

py::list gemm_group(const py::sequence& xs, const py::sequence& terms, const py::object& biases, const py::object& outs, int panel_mode,
                    const py::object& panel_ws) {
    const size_t count = terms.size();
    py::list result;
    if (count == 0) return result;
    TORCH_CHECK(xs.size() == count && (biases.is_none() || py::len(biases) == count) && (outs.is_none() || py::len(outs) == count),
                "one x (and one bias / output entry) per term");
    const std::vector<Tensor> x = tensors_of(xs, "x");
    const int dt = gemm_dtype(x[0]);
    const c10::DeviceGuard guard(x[0].device());
    std::vector<GroupTerm> checked;
    std::vector<Tensor> out(count);
    checked.reserve(count);
    for (size_t i = 0; i < count; ++i) {
        const py::object term = terms[i], bias = biases.is_none() ? py::object(py::none()) : py::object(py::sequence(biases)[i]);
        checked.push_back(group_term(x[i], x[0], term.ptr(), bias.ptr()));
        const GemmDims& d = checked.back().d;
        if (!outs.is_none()) {
            out[i] = tensor_of(py::object(py::sequence(outs)[i]).ptr(), "out");
            TORCH_CHECK(out[i].dim() == 2 && out[i].size(0) == d.tokens && out[i].size(1) == d.m && out[i].scalar_type() == x[0].scalar_type() &&
                            out[i].device() == x[0].device() && out[i].is_contiguous() && (uintptr_t)out[i].const_data_ptr() % 16 == 0,
                        "outs[", i, "] must be a contiguous, 16-byte aligned [", d.tokens, ", ", d.m, "] tensor of ",
                        dt == NQ_F16 ? "torch.float16" : "torch.bfloat16", " on ", x[0].device().str());
        }
    }
    {
        const py::gil_scoped_release unlocked;
        std::vector<void*> y;
        for (size_t i = 0; i < count; ++i) {
            const GemmDims& d = checked[i].d;
            if (outs.is_none()) out[i] = empty({d.tokens, d.m}, x[0]);
            checked[i].h = empty({d.tokens, d.r}, x[0]);
            y.push_back(out[i].mutable_data_ptr());
        }
        if (checked[0].d.tokens > 0) launch_group_terms(checked, y, dt, panel_mode, panel_ws);
    }
    for (const Tensor& t : out) result.append(py::reinterpret_steal<py::object>(THPVariable_Wrap(t)));
    return result;
}

// Weights that are sums of terms.  Where one call can take all terms the second GEMM adds them up; otherwise the t-th terms of all
// weights write into one flat buffer per t, weights with more terms first, so that the sums over the terms are one in-place add
// per extra term index.
py::list gemm_group_sum(const py::sequence& xs, const py::sequence& term_groups, const py::object& bias_groups, int panel_mode,
                        const py::object& panel_ws) {
    const size_t weights = term_groups.size();
    py::list result;
    if (weights == 0) return result;
    bool filled = xs.size() == weights;
    std::vector<py::sequence> groups;
    std::vector<size_t> terms_of_weight;
    for (size_t i = 0; i < weights; ++i) {
        groups.push_back(py::sequence(term_groups[i]));
        terms_of_weight.push_back(groups.back().size());
        filled = filled && terms_of_weight.back() > 0;
    }
    TORCH_CHECK(filled, "one x and at least one term per weight");
    const std::vector<Tensor> x = tensors_of(xs, "x");
    const int dt = gemm_dtype(x[0]);
    const c10::DeviceGuard guard(x[0].device());
    const int64_t tokens = x[0].size(0);
    std::vector<size_t> order(weights);
    std::iota(order.begin(), order.end(), (size_t)0);
    std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return terms_of_weight[a] > terms_of_weight[b]; });
    const size_t depth = terms_of_weight[order[0]];
    std::vector<GroupTerm> checked;
    std::vector<Tensor> firsts(weights);
    std::vector<int64_t> rows(weights), offsets, sizes;           // per weight; per checked term; per term index
    std::vector<int> next, last(weights, -1);
    for (size_t t = 0; t < depth; ++t) {
        int64_t size = 0;
        for (size_t i : order) {
            if (terms_of_weight[i] <= t) break;
            const py::object term = groups[i][t];
            py::object bias = py::none();
            if (!bias_groups.is_none()) {
                const py::object own = py::sequence(bias_groups)[i];
                if (!own.is_none()) bias = py::sequence(own)[t];
            }
            checked.push_back(group_term(x[i], x[0], term.ptr(), bias.ptr()));
            const GemmDims& d = checked.back().d;
            if (t == 0) rows[i] = d.m;
            TORCH_CHECK(rows[i] == d.m, "all terms of a weight must have the same output size");
            TORCH_CHECK(size * x[0].element_size() % 16 == 0, "tokens * out_features must keep the outputs 16-byte aligned");
            if (last[i] >= 0) next[last[i]] = (int)next.size();
            last[i] = (int)next.size();
            next.push_back(-1);
            offsets.push_back(size);
            size += tokens * d.m;
        }
        sizes.push_back(size);
    }
    {
        const py::gil_scoped_release unlocked;
        for (GroupTerm& t : checked) t.h = empty({t.d.tokens, t.d.r}, x[0]);
        Tensor sum = empty({sizes[0]}, x[0]);
        std::vector<void*> y(checked.size(), nullptr);
        for (size_t k = 0; k < weights; ++k) {                        // the first terms, in this order
            y[k] = (char*)sum.mutable_data_ptr() + offsets[k] * x[0].element_size();
            firsts[order[k]] = sum.as_strided({tokens, rows[order[k]]}, {rows[order[k]], 1}, offsets[k]);
        }
        const int count = (int)checked.size();
        std::vector<nq_gemm_term> arr;
        if (tokens > 0 && panel_mode == NQ_PANEL_AUTO && count <= nq_gemm_group_max()) arr = terms_of(checked, y);
        if (!arr.empty() && nq_gemm_sum_pays(arr.data(), next.data(), count, (int)tokens)) {
            const MaybeTensor ws = panel_workspace(arr.data(), count, tokens, panel_mode, panel_ws);
            check_status(nq_gemm_nanoquant_sum(arr.data(), next.data(), count, (int)tokens, dt, ws ? ws->mutable_data_ptr() : nullptr,
                                               ws ? (size_t)ws->nbytes() : 0, panel_mode, stream_of(x[0])));
        } else if (tokens > 0) {
            std::vector<Tensor> more;
            for (size_t t = 1, k = weights; t < depth; ++t) {
                more.push_back(empty({sizes[t]}, x[0]));
                for (size_t i = 0; i < weights && terms_of_weight[order[i]] > t; ++i, ++k)
                    y[k] = (char*)more.back().mutable_data_ptr() + offsets[k] * x[0].element_size();
            }
            launch_group_terms(checked, y, dt, panel_mode, panel_ws);
            for (size_t t = 1; t < depth; ++t) (sizes[t] == sizes[0] ? sum : sum.narrow(0, 0, sizes[t])).add_(more[t - 1]);
        }
    }
    for (const Tensor& first : firsts) result.append(py::reinterpret_steal<py::object>(THPVariable_Wrap(first)));
    return result;
}

}  // namespace

TORCH_LIBRARY_IMPL(binary_kernels, CUDA, m) {
    m.impl("nanoquant_dyn_forward", &nanoquant_dyn_forward);
    m.impl("marlin_onebit_forward", &marlin_onebit_forward);
    m.impl("marlin_nanoquant_forward", &marlin_nanoquant_forward);
}

PYBIND11_MODULE(_host, m) {
    using Unlocked = py::call_guard<py::gil_scoped_release>;
    m.def("nanoquant_dyn_forward", &nanoquant_dyn_forward, Unlocked());
    m.def("marlin_onebit_forward", &marlin_onebit_forward, Unlocked());
    m.def("marlin_nanoquant_forward", &marlin_nanoquant_forward, Unlocked());
    m.def("gemv_bias", &gemv_bias, Unlocked());
    m.def("gemm_bias", &gemm_bias, Unlocked());
    m.def("gemm_group", &gemm_group);
    m.def("gemm_group_sum", &gemm_group_sum);
    m.def("check_hint", &check_hint_by_name);
}
