// The host side of the calls that a token is made of - layer, embedding lookup, rotation - and of those that producing and
// loading a model is made of - quantising, rotating down the columns, cutting - between torch and the C ABI, in one native
// step per call: argument checks, the output's allocation and the launch.
//
// Bound by what it costs to get a launch out: at one token the kernels take 4-5 us, and the same checks in Python with
// a ctypes call of 26 arguments took 14.2 us per W4A16B16O16Linear call, 10.9 per embedding lookup and 9.6 per
// rotation; the seven cuts of a pruned decoder layer, 53 us of kernels, took 81 (58 to 60 now), quantising
// 14336 x 4096 39 (36 now; the kernel: 29).  The checks, their messages and the order in which they are made are those of uniql_amd.ops, which
// validates a layer's own tensors once (prepare_linear) and hands the functions' addresses over (bind).
// Nothing of a call is kept: no address of an input, no check, no output.  A layer's sizes -> scratch sizes map belongs to
// the layer's handle and is a pure function of its key.  The interpreter lock is given up for the whole call - copies of
// strided rows, allocations and launches may all wait for the device - but for that map and the accumulator's lookup.
#include <torch/extension.h>

#include <map>
#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>

#include "uniql_amd.h"

namespace {

namespace py = pybind11;
using at::Tensor;

decltype(&uniql_w4a16_linear) p_linear = nullptr;
decltype(&uniql_w4a16_linear_workspace) p_workspace = nullptr;
decltype(&uniql_w4_embedding_lookup) p_embedding = nullptr;
decltype(&uniql_fwht) p_fwht = nullptr;
decltype(&uniql_fwht_composite) p_composite = nullptr;
decltype(&uniql_fwht_columns) p_fwht_columns = nullptr;
decltype(&uniql_w4a16_quantize) p_quantize = nullptr;
decltype(&uniql_w4a16_cut_columns) p_cut_columns = nullptr;
decltype(&uniql_w4a16_cut_rows) p_cut_rows = nullptr;
decltype(&uniql_status_string) p_status = nullptr;

void bind(uintptr_t linear, uintptr_t workspace, uintptr_t embedding, uintptr_t fwht, uintptr_t composite, uintptr_t fwht_columns,
          uintptr_t quantize, uintptr_t cut_columns, uintptr_t cut_rows, uintptr_t status) {
    p_linear = reinterpret_cast<decltype(p_linear)>(linear);
    p_workspace = reinterpret_cast<decltype(p_workspace)>(workspace);
    p_embedding = reinterpret_cast<decltype(p_embedding)>(embedding);
    p_fwht = reinterpret_cast<decltype(p_fwht)>(fwht);
    p_composite = reinterpret_cast<decltype(p_composite)>(composite);
    p_fwht_columns = reinterpret_cast<decltype(p_fwht_columns)>(fwht_columns);
    p_quantize = reinterpret_cast<decltype(p_quantize)>(quantize);
    p_cut_columns = reinterpret_cast<decltype(p_cut_columns)>(cut_columns);
    p_cut_rows = reinterpret_cast<decltype(p_cut_rows)>(cut_rows);
    p_status = reinterpret_cast<decltype(p_status)>(status);
}

[[noreturn]] void fail(const std::string& what) { throw std::runtime_error(what); }
void check(int code, const char* what) {
    if (code != UNIQL_OK) fail(std::string(what) + ": " + p_status(code) + " (code " + std::to_string(code) + ")");
}
void require_gpu(const Tensor& t, const char* name) {
    if (!t.is_cuda()) fail(std::string(name) + " must be a GPU tensor (this package has no CPU path)");
}
Tensor new_output(at::IntArrayRef sizes, at::ScalarType type, const Tensor& like) {
    return at::empty(sizes, like.options().dtype(type).requires_grad(false).memory_format(std::nullopt));
}

struct Linear {
    Tensor B, s, workspace;   // held so that the addresses below stay valid
    std::optional<Tensor> bias;
    int size_n, size_k, n_out, groups, had_block;
    float had_scale;
    bool silu_mul;
    std::map<std::tuple<int64_t, int64_t, unsigned>, std::pair<size_t, size_t>> needs;   // (m, columns asked for, flags) -> accum, temp bytes
};

// The call on x [m, k_in]; `sizes`: the shape of a new output.  Without the interpreter lock.
Tensor run(Linear& p, Tensor x, std::optional<Tensor> residual, bool relu2, bool out_f32, std::optional<Tensor> out,
           unsigned flags, uintptr_t stream, const py::object& accumulator, std::optional<std::vector<int64_t>> sizes) {
    if (!x.is_cuda()) fail("x must be a GPU tensor (this package has no CPU path)");
    if (x.scalar_type() != at::kHalf) fail("x and s must be float16");
    if (x.dim() != 2 || x.stride(1) != 1) fail("x must be 2-D with unit stride along K");
    const int64_t m = x.size(0);
    int64_t k_in = x.size(1);
    if (!(p.size_k - 128 < k_in && k_in <= p.size_k))
        fail("x has " + std::to_string(k_in) + " columns, the packed weights cover " + std::to_string(p.size_k));
    if (m > 0x7fffffff) fail("x has more rows than a call can take");
    if (p.silu_mul && relu2) fail("silu_mul and relu2 are different epilogues: choose one");
    const int64_t n_out = p.n_out;
    const void* res_ptr = nullptr;
    int64_t ldr = 0;
    if (residual) {
        require_gpu(*residual, "residual");
        if (p.silu_mul || relu2) fail("a residual cannot be combined with an activation epilogue");
        if (residual->scalar_type() != at::kHalf || residual->dim() != 2 || residual->size(0) != m || residual->size(1) != n_out ||
            residual->stride(1) != 1)
            fail("residual must be float16 [m, out_features] with unit inner stride");
        res_ptr = residual->data_ptr();
        ldr = m > 1 ? residual->stride(0) : n_out;
    }
    if (k_in % 8 || (m > 1 && x.stride(0) % 8) || reinterpret_cast<uintptr_t>(x.data_ptr()) % 16) {
        // rare: rows that cannot be read in 16-byte pieces are copied (and padded) here
        x = at::constant_pad_nd(x, {0, p.size_k - k_in});
        k_in = p.size_k;
    }
    const c10::DeviceGuard guard(x.device());
    const at::ScalarType type = out_f32 ? at::kFloat : at::kHalf;
    Tensor y;
    int64_t ldd = n_out;
    if (!out) {
        y = sizes ? new_output(*sizes, type, x) : new_output({m, n_out}, type, x);
    } else {
        if (out->scalar_type() != type || out->dim() != 2 || out->size(0) != m || out->size(1) != n_out || out->stride(1) != 1 ||
            out->device() != x.device())
            fail("out must be a [m, out_features] view with unit inner stride on x's device");
        y = *out;
        if (m > 1) ldd = y.stride(0);
    }
    if (m == 0) return y;
    if (out_f32) flags |= UNIQL_F_OUT_F32;
    const int64_t lda = m > 1 ? x.stride(0) : std::max<int64_t>((k_in + 7) / 8 * 8, 8);
    // Rows shorter than K are read as they are, like whole ones, unless they are rotated first or too far apart for the tiled
    // kernels' offsets; only then is there a copy of them to ask scratch memory for (4000 rows of 9000: 73 MB).
    const int64_t k_asked = p.had_block == 0 && lda < (1LL << 24) ? p.size_k : k_in;
    size_t need_acc, need_tmp;
    Tensor accum, temp;
    {
        const py::gil_scoped_acquire lock;
        const auto key = std::make_tuple(m, k_asked, flags);
        auto hit = p.needs.find(key);
        if (hit == p.needs.end()) {
            size_t acc = 0, tmp = 0;
            check(p_workspace((int)m, p.size_n, p.size_k, (int)k_asked, p.had_block, flags, &acc, &tmp), "uniql_w4a16_linear_workspace");
            if (p.needs.size() > 4096) p.needs.clear();
            hit = p.needs.emplace(key, std::make_pair(acc, tmp)).first;
        }
        need_acc = hit->second.first;
        need_tmp = hit->second.second;
        if (need_acc) accum = accumulator(py::cast(x.device()), need_acc, stream).cast<Tensor>();
    }
    if (need_tmp) temp = new_output({(int64_t)need_tmp}, at::kByte, x);
    const int code = p_linear(x.data_ptr(), lda, (int)k_in, p.B.data_ptr(), p.s.data_ptr(), p.bias ? p.bias->data_ptr() : nullptr, res_ptr,
                              ldr, y.data_ptr(), ldd, (int)n_out,
                              p.silu_mul ? UNIQL_EPI_SILU_MUL : (relu2 ? UNIQL_EPI_RELU2 : UNIQL_EPI_NONE),
                              p.workspace.data_ptr<int32_t>(), p.workspace.numel(), need_acc ? accum.data_ptr() : nullptr,
                              need_acc ? (size_t)accum.numel() * 8 : 0, need_tmp ? temp.data_ptr() : nullptr, need_tmp, (int)m, p.size_n,
                              p.size_k, p.groups, p.had_block, p.had_scale, flags, reinterpret_cast<void*>(stream));
    check(code, "uniql_w4a16_linear");
    return y;
}

// rows x [..., k] as a matrix with unit inner stride (copied only where it has to be)
Tensor as_rows(const Tensor& x, int64_t columns) {
    Tensor r = x.dim() == 2 ? x : x.reshape({-1, columns});
    return r.stride(-1) == 1 ? r : r.contiguous();
}

// a layer module's forward: x [..., in_features], residual of the result's shape
Tensor forward(Linear& p, const Tensor& x, const std::optional<Tensor>& residual, bool relu2, uintptr_t stream,
               const py::object& accumulator) {
    const py::gil_scoped_release release;
    const at::NoGradGuard no_grad;
    if (x.dim() == 0) fail("x must have at least one dimension");
    std::optional<Tensor> res;
    if (residual) res = residual->reshape({-1, p.n_out});
    std::vector<int64_t> sizes = x.sizes().vec();
    sizes.back() = p.n_out;
    return run(p, as_rows(x, x.size(-1)), res, relu2, false, std::nullopt, 0, stream, accumulator, sizes);
}

Tensor prepared(Linear& p, const Tensor& x, const std::optional<Tensor>& residual, bool relu2, bool out_f32,
                const std::optional<Tensor>& out, unsigned flags, uintptr_t stream, const py::object& accumulator) {
    const py::gil_scoped_release release;
    return run(p, x, residual, relu2, out_f32, out, flags, stream, accumulator, std::nullopt);
}

Tensor embedding(const Tensor& ids_in, const Tensor& weight, const Tensor& scale, uintptr_t stream) {
    const py::gil_scoped_release release;
    const at::NoGradGuard no_grad;
    if (weight.dim() != 2) fail("weight must be 2-D");
    require_gpu(weight, "weight");
    if (weight.scalar_type() != at::kInt) fail("weight's dtype must be int32");
    const int64_t vocab = weight.size(0), dim = weight.size(1) * 8;
    if (scale.dim() != 1) fail("scale must be 1-D");
    require_gpu(scale, "scale");
    if (scale.scalar_type() != at::kHalf) fail("scale's dtype must be float16");
    if (scale.numel() != vocab) fail("scale must have one entry per vocabulary row");
    if (ids_in.dim() != 1 && ids_in.dim() != 2) fail("input must be a 1D or 2D tensor");
    require_gpu(ids_in, "input");
    if (ids_in.scalar_type() != at::kLong) fail("input's dtype must be int64");
    const Tensor ids = ids_in.contiguous();
    if (!weight.is_contiguous() || !scale.is_contiguous()) fail("weight and scale must be contiguous");
    const c10::DeviceGuard guard(ids.device());
    std::vector<int64_t> sizes = ids.sizes().vec();
    sizes.push_back(dim);
    Tensor y = new_output(sizes, at::kHalf, ids);
    const int code = p_embedding(ids.data_ptr<int64_t>(), ids.numel(), weight.data_ptr(), scale.data_ptr(), y.data_ptr(), vocab,
                                 (int)dim, reinterpret_cast<void*>(stream));
    check(code, "uniql_w4_embedding_lookup");
    return y;
}

int value_type(at::ScalarType t) { return t == at::kHalf ? UNIQL_DT_F16 : (t == at::kBFloat16 ? UNIQL_DT_BF16 : UNIQL_DT_F32); }

// base 0: blocks of `block` values; else the composite transform of width base * 2^k.  New tensor.
Tensor hadamard(const Tensor& x_in, int64_t block, int base, double scale, uintptr_t stream) {
    const py::gil_scoped_release release;
    const at::NoGradGuard no_grad;
    require_gpu(x_in, "x");
    const at::ScalarType t = x_in.scalar_type();
    if (t != at::kHalf && t != at::kBFloat16 && t != at::kFloat)
        fail("hadamard transform supports float16 / bfloat16 / float32, got " + std::string(c10::toString(t)));
    const int type = value_type(t);
    const Tensor x = x_in.contiguous();
    const int64_t dim = x.size(-1), rows = dim ? x.numel() / dim : 0;
    if (dim > 0x7fffffff || block > 0x7fffffff) fail("the last axis is too wide");
    const c10::DeviceGuard guard(x.device());
    Tensor y = at::empty_like(x);
    void* const st = reinterpret_cast<void*>(stream);
    const int code = base == 0 ? p_fwht(x.data_ptr(), y.data_ptr(), rows, (int)dim, (int)block, (float)scale, type, st)
                               : p_composite(x.data_ptr(), y.data_ptr(), rows, (int)dim, base, (float)scale, type, st);
    check(code, base == 0 ? "uniql_fwht" : "uniql_fwht_composite");
    return y;
}

// Down the columns of x [rows, cols]; nothing where the kernel does not take the matrix.  New tensor.
std::optional<Tensor> hadamard_columns(const Tensor& x, double scale, uintptr_t stream) {
    const py::gil_scoped_release release;
    const at::NoGradGuard no_grad;
    require_gpu(x, "x");
    const at::ScalarType t = x.scalar_type();
    if (x.dim() != 2 || (t != at::kHalf && t != at::kBFloat16 && t != at::kFloat) || !x.is_contiguous()) return std::nullopt;
    const int64_t rows = x.size(0), cols = x.size(1);
    if ((rows != 1024 && rows != 2048 && rows != 4096) || cols == 0 || cols % 8 || reinterpret_cast<uintptr_t>(x.data_ptr()) % 16)
        return std::nullopt;
    if (cols > 0x7fffffff) fail("the last axis is too wide");
    const c10::DeviceGuard guard(x.device());
    Tensor y = at::empty_like(x);
    check(p_fwht_columns(x.data_ptr(), y.data_ptr(), (int)rows, (int)cols, (float)scale, value_type(t), reinterpret_cast<void*>(stream)),
          "uniql_fwht_columns");
    return y;
}

// weight [out, in] and, of weights that are quantised already, their scales [k_pad / 128, out] -> packed and permuted.  New tensors.
std::pair<Tensor, Tensor> new_packed(int64_t k, int64_t n, const Tensor& like) {
    return {new_output({k / 16, 2 * n}, at::kInt, like), new_output({k / 128, n}, at::kHalf, like)};
}
std::pair<Tensor, Tensor> quantize(const Tensor& weight, const std::optional<Tensor>& given, int64_t pad_out, uintptr_t stream) {
    const py::gil_scoped_release release;
    const at::NoGradGuard no_grad;
    require_gpu(weight, "weight");
    if (weight.scalar_type() != at::kHalf || weight.dim() != 2 || weight.stride(1) != 1)
        fail("weight must be float16 [out_features, in_features] with unit inner stride");
    const int64_t n = weight.size(0), k = weight.size(1), k_pad = (k + 127) / 128 * 128, n_pad = n + pad_out;
    if (given) {
        require_gpu(*given, "given_scale");
        if (given->scalar_type() != at::kHalf || given->dim() != 2 || given->size(0) != k_pad / 128 || given->size(1) != n ||
            !given->is_contiguous())
            fail("given_scale must be contiguous float16 [k_pad/128, out_features]");
    }
    if (n > 0x7fffffff || n_pad < 0 || n_pad > 0x7fffffff || k_pad > 0x7fffffff) fail("weight is larger than a call can take");
    const c10::DeviceGuard guard(weight.device());
    auto out = new_packed(k_pad, n_pad, weight);
    check(p_quantize(weight.data_ptr(), weight.stride(0), given ? given->data_ptr() : nullptr, out.first.data_ptr(), out.second.data_ptr(),
                     (int)n, (int)k, (int)n_pad, (int)k_pad, reinterpret_cast<void*>(stream)),
          "uniql_w4a16_quantize");
    return out;
}

// A packed group-128 matrix [k / 16, 2 n] with its scales [groups, n].
void require_packed(const Tensor& B, const Tensor& s, int64_t n, int64_t k) {
    require_gpu(B, "B");
    require_gpu(s, "s");
    if (B.scalar_type() != at::kInt || s.scalar_type() != at::kHalf || !B.is_contiguous() || !s.is_contiguous())
        fail("B must be contiguous int32 and s contiguous float16");
    if (k < 0 || B.dim() != 2 || B.size(0) != k / 16 || B.size(1) != 2 * n || s.dim() != 2 || s.size(1) != n)
        fail("B / s shapes do not match size_k, size_n");
}

// runs: six values each.  New tensors.
std::pair<Tensor, Tensor> cut_columns(const Tensor& B, const Tensor& s, int n, int k, const std::vector<int>& runs,
                                      std::optional<int> k_real, std::optional<int> n_scaled, int64_t pad_out, uintptr_t stream) {
    const py::gil_scoped_release release;
    const at::NoGradGuard no_grad;
    require_packed(B, s, n, k);
    if (s.size(0) != k / 128) fail("scales must be [k/128, n]");
    if (runs.size() % 6) fail("runs must have six values each");
    int64_t n_pad = pad_out;
    for (size_t i = 0; i < runs.size(); i += 6) n_pad += (int64_t)runs[i + 1] * runs[i + 3];
    if (n_pad < 0 || n_pad > 0x7fffffff) fail("the kept width is not one that a call can take");
    const c10::DeviceGuard guard(B.device());
    auto out = new_packed(k, n_pad, B);
    check(p_cut_columns(B.data_ptr(), s.data_ptr(), n, k, k_real.value_or(k), runs.data(), (int)(runs.size() / 6),
                        n_scaled.value_or((int)n_pad), out.first.data_ptr(), out.second.data_ptr(), (int)n_pad,
                        reinterpret_cast<void*>(stream)),
          "uniql_w4a16_cut_columns");
    return out;
}

std::pair<Tensor, Tensor> cut_rows(const Tensor& B, const Tensor& s, int n, int k, int units, int full, int kept, int n_real,
                                   int64_t pad_out, uintptr_t stream) {
    const py::gil_scoped_release release;
    const at::NoGradGuard no_grad;
    require_packed(B, s, n, k);
    const int64_t k_pad = ((int64_t)units * kept + 127) / 128 * 128, n_pad = n_real + pad_out;
    if (k_pad < 0 || n_pad < 0 || n_pad > 0x7fffffff) fail("the kept sizes are not ones that a call can take");
    const c10::DeviceGuard guard(B.device());
    auto out = new_packed(k_pad, n_pad, B);
    check(p_cut_rows(B.data_ptr(), s.data_ptr(), n, k, (int)s.size(0), units, full, kept, n_real, out.first.data_ptr(),
                     out.second.data_ptr(), (int)n_pad, reinterpret_cast<void*>(stream)),
          "uniql_w4a16_cut_rows");
    return out;
}

}  // namespace

PYBIND11_MODULE(_host, module) {
    py::class_<Linear>(module, "Linear")
        .def(py::init([](Tensor B, Tensor s, Tensor workspace, std::optional<Tensor> bias, int size_n, int size_k, int n_out,
                         int had_block, double had_scale, bool silu_mul) {
            const int groups = (int)s.size(0);
            return Linear{std::move(B), std::move(s), std::move(workspace), std::move(bias), size_n, size_k, n_out, groups,
                          had_block, (float)had_scale, silu_mul, {}};
        }))
        .def_readonly("B", &Linear::B)
        .def_readonly("s", &Linear::s)
        .def_readonly("workspace", &Linear::workspace)
        .def_readonly("bias", &Linear::bias)
        .def_readonly("size_n", &Linear::size_n)
        .def_readonly("size_k", &Linear::size_k)
        .def_readonly("n_out", &Linear::n_out)
        .def_readonly("groups", &Linear::groups)
        .def_readonly("had_block", &Linear::had_block)
        .def_readonly("had_scale", &Linear::had_scale)
        .def_readonly("silu_mul", &Linear::silu_mul)
        .def("forward", &forward)
        .def("prepared", &prepared);
    module.def("bind", &bind);
    module.def("embedding", &embedding);
    module.def("hadamard", &hadamard);
    module.def("hadamard_columns", &hadamard_columns);
    module.def("quantize", &quantize);
    module.def("cut_columns", &cut_columns);
    module.def("cut_rows", &cut_rows);
}
