// The operators of torch.ops.ops_rec as native dispatcher kernels (device key CUDA = HIP tensors, and AutogradCUDA).
//
// What bounds a small call is the host: the Python implementations (ops_rec/_ops.py, _activation.py) take 13 .. 24 us per
// forward and 150 .. 300 us per forward + backward through a Python autograd formula, for kernels of 5 .. 40 us.  Here a call
// in canonical form -- contiguous tensors of one device, index tensors of one type, shapes that agree -- is described to the
// C ABI (include/hstu_mi355.h) and launched without entering Python, in the backward on the autograd engine's own thread.
// Every other call (something to convert, an argument to refuse, an empty output) goes to the Python implementation, which
// holds the checks, their messages and the conversions; so nothing is accepted or refused here that is not there.

#include <ATen/Context.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/native/TensorFactories.h>
#include <ATen/ops/mm.h>
#include <ATen/ops/zeros.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>

#include <cstring>
#include <optional>
#include <tuple>

#include "../../include/hstu_mi355.h"
#include "../../include/ops_rec_activation_mi355.h"

namespace py = pybind11;

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The Python implementations by name, set once by set_fallbacks(); never released (calls may come during interpreter exit).
struct Fallbacks {
    PyObject* forward = nullptr;          // _ops._forward_impl
    PyObject* backward = nullptr;         // _ops._backward_impl
    PyObject* paged = nullptr;            // _ops.hstu_paged
    PyObject* ln_mul = nullptr;           // _activation.ln_mul
    PyObject* in_linear_silu = nullptr;   // _activation.distance_in_linear_silu
    PyObject* in_linear_silu_backward = nullptr;
} fallbacks;

template <typename R, typename... A>
R in_python(PyObject* fn, const A&... args)
{
    py::gil_scoped_acquire gil;
    TORCH_CHECK(fn != nullptr, "ops_rec: the Python implementations have not been attached");
    return py::reinterpret_borrow<py::object>(fn)(args...).template cast<R>();
}

int dtype_code(at::ScalarType t)
{
    switch (t) {
    case at::kBFloat16: return HSTU_DT_BF16;
    case at::kHalf: return HSTU_DT_FP16;
    case at::kFloat: return HSTU_DT_FP32;
    case at::kFloat8_e4m3fn: return HSTU_DT_FP8_E4M3;
    default: return -1;
    }
}

// torch.empty without its way through the dispatcher: memory nobody has written yet holds NaN (all ones) when the program has asked
// for that (torch.use_deterministic_algorithms with torch.utils.deterministic.fill_uninitialized_memory)
Tensor empty(at::IntArrayRef size, at::ScalarType dtype, const at::Device& device)
{
    Tensor t(at::detail::empty_cuda(size, dtype, device, std::nullopt));
    const at::Context& context = at::globalContext();
    if (context.deterministicAlgorithms() && context.deterministicFillUninitializedMemory()) {
        at::native::fill_empty_deterministic_(t);
    }
    return t;
}

// A workspace a call can do without: none (undefined) when the allocator has no room for it.
Tensor empty_or_none(uint64_t bytes, const at::Device& device)
{
    if (bytes != 0) {
        try {
            return empty({static_cast<int64_t>(bytes)}, at::kByte, device);
        } catch (const c10::OutOfMemoryError&) {
        }
    }
    return Tensor();
}

void* ptr(const Tensor& t) { return t.defined() && t.numel() != 0 ? t.data_ptr() : nullptr; }
void* ptr(const OptTensor& t) { return t.has_value() ? ptr(*t) : nullptr; }

bool is_set(const OptTensor& t) { return t.has_value() && t->defined(); }

// an optional tensor as the library reads it: absent, or on the device, contiguous and of the type and 1-D size given
bool absent_or_vector(const OptTensor& t, at::ScalarType dtype, int64_t n, const at::Device& device)
{
    return !is_set(t) || (t->device() == device && t->scalar_type() == dtype && t->dim() == 1 && t->size(0) == n && t->is_contiguous());
}

bool absent_or_plane(const OptTensor& t, const Tensor& q, int64_t batch, int64_t max_q, int64_t max_k)
{
    return !is_set(t) || (t->device() == q.device() && t->scalar_type() == q.scalar_type() && t->dim() == 4 && t->size(0) == batch &&
                          t->size(1) == q.size(1) && t->size(2) == max_q && t->size(3) == max_k && t->is_contiguous());
}

hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// The arguments of one attention call, in the order of the operators' schemas.
struct Call {
    const Tensor& q;
    const Tensor& k;
    const Tensor& v;
    const OptTensor& mask;
    const OptTensor& bias;
    int64_t mask_type, max_q, max_k;
    double silu_scale;
    const Tensor& offs_q;
    const Tensor& offs_k;
    const OptTensor& ctx;
    const OptTensor& tgt;
    std::optional<int64_t> group;
    std::optional<double> alpha;
};

constexpr int64_t kMaxSeqLen = HSTU_MAX_SEQ_LEN;

// Fills the C-ABI description (all but `out`); false when the call is not in canonical form.  q, k and v are contiguous.
bool describe(const Call& c, hstu_jagged_fwd_params& p)
{
    const Tensor &q = c.q, &k = c.k, &v = c.v, &oq = c.offs_q, &ok = c.offs_k;
    if (q.dim() != 3 || k.dim() != 3 || v.dim() != 3 || !oq.defined() || !ok.defined()) {
        return false;
    }
    const at::Device device = q.device();
    const at::ScalarType dtype = q.scalar_type(), index = oq.scalar_type();
    const int code = dtype_code(dtype);
    const bool same = &oq == &ok || ok.is_same(oq);
    if (!device.is_cuda() || code < 0 || k.scalar_type() != dtype || v.scalar_type() != dtype || k.device() != device || v.device() != device ||
        !q.is_contiguous() || !k.is_contiguous() || !v.is_contiguous() || k.size(0) != v.size(0) || k.size(1) != v.size(1) ||
        q.size(2) != k.size(2)) {
        return false;
    }
    if ((index != at::kInt && index != at::kLong) || oq.dim() != 1 || oq.size(0) < 2 || oq.device() != device || !oq.is_contiguous()) {
        return false;
    }
    const int64_t batch = oq.size(0) - 1;
    if (!same && (ok.scalar_type() != index || ok.dim() != 1 || ok.size(0) != oq.size(0) || ok.device() != device || !ok.is_contiguous())) {
        return false;
    }
    if (c.max_q < 1 || c.max_q > kMaxSeqLen || c.max_k < 1 || c.max_k > kMaxSeqLen || c.mask_type < 0 || c.mask_type > 3 || c.mask_type == 1 ||
        (c.mask_type == HSTU_MASK_CUSTOM) != is_set(c.mask)) {
        return false;  // (a mask beside another mask_type is only checked for its device: left to Python)
    }
    if (!absent_or_vector(c.ctx, index, batch, device) || !absent_or_vector(c.tgt, index, batch, device) ||
        !absent_or_plane(c.bias, q, batch, c.max_q, c.max_k) || !absent_or_plane(c.mask, q, batch, c.max_q, c.max_k)) {
        return false;
    }
    std::memset(&p, 0, sizeof p);
    p.struct_size = sizeof p;
    p.dtype = code;
    p.out_dtype = code == HSTU_DT_FP8_E4M3 ? HSTU_DT_FP16 : code;
    p.index_dtype = index == at::kLong ? HSTU_IDX_I64 : HSTU_IDX_I32;
    p.q = ptr(q);
    p.k = ptr(k);
    p.v = ptr(v);
    p.mask = ptr(c.mask);
    p.attn_bias = ptr(c.bias);
    p.seq_offset_q = oq.data_ptr();
    p.seq_offset_k = ok.data_ptr();
    p.num_context = ptr(c.ctx);
    p.num_target = ptr(c.tgt);
    p.total_q = q.size(0);
    p.total_k = k.size(0);
    p.num_heads_q = q.size(1);
    p.num_heads_k = k.size(1);
    p.head_dim_qk = q.size(2);
    p.head_dim_v = v.size(2);
    p.n_offsets = batch + 1;
    p.mask_type = c.mask_type;
    p.max_seq_len_q = c.max_q;
    p.max_seq_len_k = c.max_k;
    p.target_group_size = c.group.value_or(0);
    p.silu_scale = c.silu_scale == 0.0 ? 1.0 / static_cast<double>(c.max_q) : c.silu_scale;
    p.alpha = c.alpha.value_or(1.0);
    return true;
}

// Output allocated, workspace asked for and the kernel launched; an undefined tensor when the library refuses the description
// (the Python implementation then says so in its words).
Tensor launch_forward(hstu_jagged_fwd_params& p, const Tensor& q, at::ScalarType out_dtype)
{
    const c10::DeviceGuard guard(q.device());
    uint64_t ws_bytes = 0;
    if (p.total_q * p.num_heads_q * p.head_dim_v == 0) {
        return Tensor();
    }
    Tensor out = empty({p.total_q, p.num_heads_q, p.head_dim_v}, out_dtype, q.device());
    p.out = out.data_ptr();
    if (hstu_jagged_fwd_workspace_size(&p, &ws_bytes) != HSTU_OK) {
        return Tensor();
    }
    Tensor ws;
    if (ws_bytes != 0) {
        ws = empty({static_cast<int64_t>(ws_bytes)}, at::kByte, q.device());
    }
    const int rc = hstu_jagged_fwd(&p, ptr(ws), ws_bytes, stream_of(q));
    TORCH_CHECK(rc == HSTU_OK, "hstu_jagged_fwd failed (", rc, "): ", hstu_last_error());
    return out;
}

Tensor forward(const Call& c, bool deterministic)
{
    hstu_jagged_fwd_params p;
    if (describe(c, p)) {
        const bool fp8 = p.dtype == HSTU_DT_FP8_E4M3;
        p.deterministic = deterministic ? 1 : 0;
        p.fp8_scaled_p = fp8 ? 1 : 0;  // e4m3 tensors through the reference's entry point: its rounding point of P
        Tensor out = launch_forward(p, c.q, fp8 ? at::kHalf : c.q.scalar_type());
        if (out.defined()) {
            return out;
        }
    }
    return in_python<Tensor>(fallbacks.forward, c.q, c.k, c.v, c.mask, c.bias, c.mask_type, c.max_q, c.max_k, c.silu_scale, c.offs_q, c.offs_k,
                             c.ctx, c.tgt, c.group, c.alpha, deterministic);
}

using Gradients = std::tuple<Tensor, Tensor, Tensor, Tensor>;

Gradients backward(const Tensor& grad_in, const Call& c)
{
    const Tensor& q = c.q;
    const at::ScalarType dtype = q.scalar_type();
    // (a gradient may come as an expanded view: from a sum, for instance)
    const Tensor grad = grad_in.defined() && !grad_in.is_contiguous() ? grad_in.contiguous() : grad_in;
    hstu_jagged_bwd_params p;
    if (dtype != at::kFloat8_e4m3fn && is_set(c.ctx) == is_set(c.tgt) && grad.defined() &&
        describe(c, p.fwd) && grad.dim() == 3 && grad.scalar_type() == dtype && grad.device() == q.device() && grad.size(0) == q.size(0) &&
        grad.size(1) == q.size(1) && grad.size(2) == c.v.size(2) && (q.numel() != 0 || c.k.numel() != 0)) {
        const c10::DeviceGuard guard(q.device());
        Tensor dq = empty(q.sizes(), dtype, q.device()), dk = empty(c.k.sizes(), dtype, q.device()), dv = empty(c.v.sizes(), dtype, q.device());
        Tensor dbias;
        if (is_set(c.bias)) {
            dbias = empty(c.bias->sizes(), dtype, q.device());
        }
        p.struct_size = sizeof p;
        p.reserved0 = 0;
        p.grad = ptr(grad);
        p.grad_q = ptr(dq);
        p.grad_k = ptr(dk);
        p.grad_v = ptr(dv);
        p.grad_attn_bias = ptr(dbias);
        uint64_t ws_bytes = 0;
        if (hstu_jagged_bwd_best_workspace_size(&p, &ws_bytes) == HSTU_OK) {
            Tensor ws = empty_or_none(ws_bytes, q.device());
            // no room: the workspace of the other launch orders where that is a smaller one, and none for the order that needs none
            uint64_t less = 0;
            if (!ws.defined() && hstu_jagged_bwd_workspace_size(&p, &less) == HSTU_OK && less < ws_bytes) {
                ws_bytes = less;
                ws = empty_or_none(ws_bytes, q.device());
            }
            const int rc = hstu_jagged_bwd(&p, ptr(ws), ws.defined() ? ws_bytes : 0, stream_of(q));
            TORCH_CHECK(rc == HSTU_OK, "hstu_jagged_bwd failed (", rc, "): ", hstu_last_error());
            return {dq, dk, dv, dbias};
        }
    }
    py::gil_scoped_acquire gil;
    const auto r = in_python<std::tuple<Tensor, Tensor, Tensor, OptTensor>>(fallbacks.backward, grad_in, c.q, c.k, c.v, c.mask, c.bias, c.mask_type,
                                                                            c.max_q, c.max_k, c.silu_scale, c.offs_q, c.offs_k, c.ctx, c.tgt,
                                                                            c.group, c.alpha);
    return {std::get<0>(r), std::get<1>(r), std::get<2>(r), std::get<3>(r).value_or(Tensor())};
}

// q, k, v as the kernels read them (a view that is not contiguous is copied, as the Python implementation does)
const Tensor contiguous(const Tensor& t) { return t.is_contiguous() ? t : t.contiguous(); }

Tensor jagged_equal(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& mask, const OptTensor& bias, int64_t mask_type,
                    int64_t max_seq_len, double silu_scale, const Tensor& offs, const OptTensor& ctx, const OptTensor& tgt,
                    std::optional<int64_t> group, std::optional<double> alpha, bool deterministic)
{
    const Tensor qc = contiguous(q), kc = contiguous(k), vc = contiguous(v);
    return forward({qc, kc, vc, mask, bias, mask_type, max_seq_len, max_seq_len, silu_scale, offs, offs, ctx, tgt, group, alpha}, deterministic);
}

Tensor jagged_delta(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& mask, const OptTensor& bias, int64_t mask_type,
                    int64_t max_seq_len, int64_t max_seq_len_k, double silu_scale, const Tensor& offs, const Tensor& offs_k, const OptTensor& ctx,
                    const OptTensor& tgt, std::optional<int64_t> group, std::optional<double> alpha, bool deterministic)
{
    const Tensor qc = contiguous(q), kc = contiguous(k), vc = contiguous(v);
    return forward({qc, kc, vc, mask, bias, mask_type, max_seq_len, max_seq_len_k, silu_scale, offs, offs_k, ctx, tgt, group, alpha}, deterministic);
}

Gradients jagged_backward_delta(const Tensor& grad, const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& mask, const OptTensor& bias,
                                int64_t mask_type, int64_t max_seq_len, int64_t max_seq_len_k, double silu_scale, const Tensor& offs,
                                const Tensor& offs_k, const OptTensor& ctx, const OptTensor& tgt, std::optional<int64_t> group,
                                std::optional<double> alpha)
{
    const Tensor qc = contiguous(q), kc = contiguous(k), vc = contiguous(v);
    return backward(grad, {qc, kc, vc, mask, bias, mask_type, max_seq_len, max_seq_len_k, silu_scale, offs, offs_k, ctx, tgt, group, alpha});
}

Gradients jagged_backward_equal(const Tensor& grad, const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& mask, const OptTensor& bias,
                                int64_t mask_type, int64_t max_seq_len, double silu_scale, const Tensor& offs, const OptTensor& ctx,
                                const OptTensor& tgt, std::optional<int64_t> group, std::optional<double> alpha)
{
    return jagged_backward_delta(grad, q, k, v, mask, bias, mask_type, max_seq_len, max_seq_len, silu_scale, offs, offs, ctx, tgt, group, alpha);
}

// hstu_jagged_fp8 (a Python function, not a dispatcher operator): None when the call is not in canonical form.
OptTensor fp8_forward(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& q_descale, const OptTensor& k_descale,
                      const OptTensor& v_descale, const OptTensor& mask, const OptTensor& bias, int64_t mask_type, int64_t max_seq_len,
                      int64_t max_seq_len_k, double silu_scale, const Tensor& offs, const Tensor& offs_k, const OptTensor& ctx,
                      const OptTensor& tgt, std::optional<int64_t> group, std::optional<double> alpha, bool half_out)
{
    hstu_jagged_fwd_params p;
    if (!describe({q, k, v, mask, bias, mask_type, max_seq_len, max_seq_len_k, silu_scale, offs, offs_k, ctx, tgt, group, alpha}, p) ||
        p.dtype != HSTU_DT_FP8_E4M3 || !absent_or_vector(q_descale, at::kFloat, q.size(1), q.device()) ||
        !absent_or_vector(k_descale, at::kFloat, k.size(1), q.device()) || !absent_or_vector(v_descale, at::kFloat, k.size(1), q.device())) {
        return std::nullopt;
    }
    p.out_dtype = half_out ? HSTU_DT_FP16 : HSTU_DT_BF16;
    p.q_descale = static_cast<const float*>(ptr(q_descale));
    p.k_descale = static_cast<const float*>(ptr(k_descale));
    p.v_descale = static_cast<const float*>(ptr(v_descale));
    Tensor out = launch_forward(p, q, half_out ? at::kHalf : at::kBFloat16);
    return out.defined() ? OptTensor(out) : std::nullopt;
}

Tensor paged(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cache, const OptTensor& mask, const OptTensor& bias, int64_t mask_type,
             int64_t max_seq_len, int64_t max_seq_len_k, double silu_scale, const Tensor& offs, const Tensor& offs_k, const Tensor& offs_t,
             const Tensor& page_offsets, const Tensor& page_ids, const Tensor& last_page_len, const Tensor& num_target, int64_t group,
             std::optional<double> alpha, bool deterministic)
{
    hstu_paged_fwd_params p;
    const OptTensor tgt = num_target.defined() ? OptTensor(num_target) : std::nullopt;
    if (cache.defined() && page_ids.defined() && last_page_len.defined() && offs_t.defined() &&
        page_offsets.defined() && describe({q, k, v, mask, bias, mask_type, max_seq_len, max_seq_len_k, silu_scale, offs, offs_k, std::nullopt, tgt, group, alpha}, p.fwd)) {
        const at::ScalarType index = offs.scalar_type();
        const auto vector = [&](const Tensor& t) {
            return t.dim() == 1 && t.size(0) > 0 && t.scalar_type() == index && t.device() == q.device() && t.is_contiguous();
        };
        if (p.fwd.dtype != HSTU_DT_FP8_E4M3 && (group > 0 || !tgt) && k.size(0) == q.size(0) && v.size(2) == k.size(2) && cache.dim() == 5 &&
            cache.size(1) == 2 && cache.numel() != 0 && cache.scalar_type() == q.scalar_type() && cache.device() == q.device() &&
            cache.size(3) == k.size(1) && cache.size(4) == k.size(2) && cache.is_contiguous() && vector(offs_t) && offs_t.size(0) >= 2 &&
            vector(page_offsets) && page_offsets.size(0) == offs.size(0) && vector(page_ids) && vector(last_page_len) && q.numel() != 0) {
            const c10::DeviceGuard guard(q.device());
            p.struct_size = sizeof p;
            p.reserved0 = 0;
            p.fwd.deterministic = deterministic ? 1 : 0;
            // an upper bound on the end of the key ranges that needs no device read: every page full plus every input row
            p.fwd.total_k = page_ids.numel() * cache.size(2) + q.size(0);
            p.kv_cache = cache.data_ptr();
            p.page_offsets = page_offsets.data_ptr();
            p.page_ids = page_ids.data_ptr();
            p.last_page_len = last_page_len.data_ptr();
            p.seq_offset_t = offs_t.data_ptr();
            p.num_pages = cache.size(0);
            p.page_size = cache.size(2);
            p.n_page_ids = page_ids.numel();
            Tensor out = empty({q.size(0), q.size(1), v.size(2)}, q.scalar_type(), q.device());
            p.fwd.out = out.data_ptr();
            uint64_t ws_bytes = 0;
            if (hstu_paged_fwd_workspace_size(&p, &ws_bytes) == HSTU_OK) {
                const Tensor ws = empty({static_cast<int64_t>(ws_bytes != 0 ? ws_bytes : 1)}, at::kByte, q.device());
                const int rc = hstu_paged_fwd(&p, ws.data_ptr(), ws_bytes, stream_of(q));
                TORCH_CHECK(rc == HSTU_OK, "hstu_paged_fwd failed (", rc, "): ", hstu_last_error());
                return out;
            }
        }
    }
    const auto maybe = [](const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; };
    return in_python<Tensor>(fallbacks.paged, q, k, v, maybe(cache), mask, bias, mask_type, max_seq_len, max_seq_len_k, silu_scale, maybe(offs),
                             maybe(offs_k), maybe(offs_t), maybe(page_offsets), maybe(page_ids), maybe(last_page_len), tgt, group, alpha,
                             deterministic);
}

// ------------------------------------------------------------------------------------------------ layer operators ----

Tensor ln_mul(const Tensor& x, const Tensor& u, const Tensor& gamma, const Tensor& beta)
{
    const at::ScalarType dtype = x.scalar_type(), affine = gamma.scalar_type();
    const at::Device device = x.device();
    if (device.is_cuda() && x.dim() == 2 && u.dim() == 2 && gamma.dim() == 1 && beta.dim() == 1 &&
        x.numel() != 0 && x.sizes() == u.sizes() && (dtype == at::kFloat || dtype == at::kBFloat16 || dtype == at::kHalf) && u.scalar_type() == dtype &&
        beta.scalar_type() == affine && (affine == at::kFloat || affine == dtype) && gamma.size(0) == x.size(1) && beta.size(0) == x.size(1) &&
        u.device() == device && gamma.device() == device && beta.device() == device && x.is_contiguous() && u.is_contiguous() &&
        gamma.is_contiguous() && beta.is_contiguous()) {
        const c10::DeviceGuard guard(device);
        Tensor out = empty(x.sizes(), dtype, device);
        ln_mul_params p;
        std::memset(&p, 0, sizeof p);
        p.struct_size = sizeof p;
        p.x = x.data_ptr();
        p.u = u.data_ptr();
        p.gamma = gamma.data_ptr();
        p.beta = beta.data_ptr();
        p.out = out.data_ptr();
        p.rows = x.size(0);
        p.cols = x.size(1);
        p.dtype = dtype_code(dtype);
        p.affine_dtype = dtype_code(affine);
        p.epsilon = 1e-5f;  // fixed by the reference's host tiling (ascendc/activation/ln_mul/op_host/ln_mul.cpp:75)
        const int rc = ln_mul_fwd(&p, stream_of(x));
        TORCH_CHECK(rc == HSTU_OK, "ln_mul failed (", rc, "): ", hstu_last_error());
        return out;
    }
    return in_python<Tensor>(fallbacks.ln_mul, x, u, gamma, beta);
}

// shapes, types and layout of x, weight, bias and the split as in_linear_silu takes them (_activation._in_linear_silu_shapes)
bool in_linear_silu_canonical(const Tensor& x, const Tensor& weight, const OptTensor& bias, at::IntArrayRef split)
{
    constexpr int64_t lo = 16, hi = 512 * 16;
    if (x.dim() != 2 || weight.dim() != 2 || x.numel() == 0 || weight.numel() == 0 || split.size() != 4 || !x.device().is_cuda() ||
        weight.device() != x.device() || (x.scalar_type() != at::kBFloat16 && x.scalar_type() != at::kHalf) || weight.scalar_type() != x.scalar_type() ||
        !x.is_contiguous() || !weight.is_contiguous()) {
        return false;
    }
    const int64_t k = x.size(1), n = weight.size(0);
    int64_t sum = 0;
    for (const int64_t s : split) {
        if (s < lo || s > hi || s % lo != 0) {
            return false;
        }
        sum += s;
    }
    return k >= lo && k <= hi && k % lo == 0 && n >= 4 * lo && n <= 4 * hi && n % lo == 0 && sum == n && weight.size(1) == k && n % (4 * k) == 0 &&
           absent_or_vector(bias, at::kFloat, n, x.device());
}

using Projection = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor>;

Projection in_linear_silu(const Tensor& x, const Tensor& weight, const Tensor& bias_in, at::IntArrayRef split)
{
    const OptTensor bias = bias_in.defined() ? OptTensor(bias_in) : std::nullopt;
    if (in_linear_silu_canonical(x, weight, bias, split)) {
        const c10::DeviceGuard guard(x.device());
        const int64_t m = x.size(0), n = weight.size(0);
        const auto rows = [&](int64_t cols) { return empty({m, cols}, x.scalar_type(), x.device()); };
        Projection out{rows(split[0]), rows(split[1]), rows(split[2]), rows(split[3]), rows(n)};
        in_linear_silu_params p;
        std::memset(&p, 0, sizeof p);
        p.struct_size = sizeof p;
        p.x = x.data_ptr();
        p.weight = weight.data_ptr();
        p.bias = static_cast<decltype(p.bias)>(ptr(bias));
        p.user = std::get<0>(out).data_ptr();
        p.value = std::get<1>(out).data_ptr();
        p.query = std::get<2>(out).data_ptr();
        p.key = std::get<3>(out).data_ptr();
        p.linear_output = std::get<4>(out).data_ptr();
        p.m = m;
        p.n = n;
        p.k = x.size(1);
        for (int i = 0; i < 4; ++i) {
            p.split[i] = split[i];
        }
        p.dtype = dtype_code(x.scalar_type());
        const int rc = in_linear_silu_fwd(&p, stream_of(x));
        TORCH_CHECK(rc == HSTU_OK, "in_linear_silu failed (", rc, "): ", hstu_last_error());
        return out;
    }
    return in_python<Projection>(fallbacks.in_linear_silu, x, weight, bias, split.vec());
}

Gradients in_linear_silu_backward(const Tensor& x, const Tensor& weight, const OptTensor& bias, const Tensor& user_grad, const Tensor& value_grad,
                                  const Tensor& query_grad, const Tensor& key_grad, const Tensor& linear_output, at::IntArrayRef split)
{
    const Tensor* const grads[4] = {&user_grad, &value_grad, &query_grad, &key_grad};
    bool ok = in_linear_silu_canonical(x, weight, bias, split) && linear_output.dim() == 2 &&
              linear_output.size(0) == x.size(0) && linear_output.size(1) == weight.size(0) && linear_output.scalar_type() == x.scalar_type() &&
              linear_output.device() == x.device() && linear_output.is_contiguous();
    for (int i = 0; ok && i < 4; ++i) {
        const Tensor& g = *grads[i];
        ok = g.dim() == 2 && g.size(0) == x.size(0) && g.size(1) == split[i] && g.scalar_type() == x.scalar_type() && g.device() == x.device();
    }
    if (ok) {
        const c10::DeviceGuard guard(x.device());
        const int64_t m = x.size(0), n = weight.size(0);
        const Tensor g[4] = {contiguous(user_grad), contiguous(value_grad), contiguous(query_grad), contiguous(key_grad)};
        Tensor d_mixed = empty({m, n}, x.scalar_type(), x.device()), weight_grad, bias_grad;
        if (is_set(bias)) {
            bias_grad = empty({n}, at::kFloat, x.device());
        }
        in_linear_silu_bwd_weight_params p;
        std::memset(&p, 0, sizeof p);
        p.struct_size = sizeof p;
        p.x = x.data_ptr();
        p.k = x.size(1);
        in_linear_silu_bwd_params& s = p.stage;
        s.struct_size = sizeof s;
        s.linear_output = linear_output.data_ptr();
        s.user_grad = g[0].data_ptr();
        s.value_grad = g[1].data_ptr();
        s.query_grad = g[2].data_ptr();
        s.key_grad = g[3].data_ptr();
        s.d_mixed = d_mixed.data_ptr();
        s.bias_grad = static_cast<float*>(ptr(bias_grad));
        s.m = m;
        s.n = n;
        for (int i = 0; i < 4; ++i) {
            s.split[i] = split[i];
        }
        s.dtype = dtype_code(x.scalar_type());
        uint64_t ws_bytes = 0;
        int rc = HSTU_OK;
        bool library = in_linear_silu_bwd_weight_pays(&p) == 0;
        if (!library) {
            weight_grad = empty({n, x.size(1)}, x.scalar_type(), x.device());
            p.weight_grad = weight_grad.data_ptr();
            rc = in_linear_silu_bwd_weight_workspace_size(&p, &ws_bytes);
            if (rc == HSTU_OK) {
                if (const Tensor ws = empty_or_none(ws_bytes, x.device()); ws.defined()) {
                    rc = in_linear_silu_bwd_weight(&p, ws.data_ptr(), ws_bytes, stream_of(x));
                } else {  // no room for the partial weight gradients: the library product needs none
                    library = true;
                }
            }
        }
        if (library) {
            rc = in_linear_silu_bwd_dmixed_workspace_size(&s, &ws_bytes);
            if (rc == HSTU_OK) {
                const Tensor ws = ws_bytes != 0 ? empty({static_cast<int64_t>(ws_bytes)}, at::kByte, x.device()) : Tensor();
                rc = in_linear_silu_bwd_dmixed(&s, ptr(ws), ws_bytes, stream_of(x));
            }
        }
        TORCH_CHECK(rc == HSTU_OK, "in_linear_silu_backward failed (", rc, "): ", hstu_last_error());
        if (library) {
            weight_grad = at::mm(d_mixed.t(), x);
        }
        return {at::mm(d_mixed, weight), weight_grad, bias_grad, Tensor()};
    }
    py::gil_scoped_acquire gil;
    const auto r = in_python<std::tuple<Tensor, Tensor, OptTensor, OptTensor>>(fallbacks.in_linear_silu_backward, x, weight, bias, user_grad,
                                                                               value_grad, query_grad, key_grad, linear_output, split.vec());
    return {std::get<0>(r), std::get<1>(r), std::get<2>(r).value_or(Tensor()), Tensor()};
}

// ------------------------------------------------------------------------------------------------------- autograd ----
// The formulas of ops_rec/autograd/hstu_v1_autograd.py and _activation.py as C++ nodes: what is saved, what is refused and which
// inputs get gradients are the same (ascendc/attention/hstu_v1/torch_extension/hstu_v1_autograd.py:53-374).  Both directions go
// through the dispatcher below autograd, so tracing and functionalisation see the operators.

template <typename F>
auto operator_handle(const char* name, const char* overload)
{
    return c10::Dispatcher::singleton().findSchemaOrThrow(name, overload).typed<F>();
}

bool needs_grad(const Tensor& t) { return t.defined() && t.requires_grad(); }
bool needs_grad(const OptTensor& t) { return t.has_value() && needs_grad(*t); }

Tensor unwrap(const OptTensor& t) { return t.value_or(Tensor()); }
OptTensor wrap(const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; }

template <bool DELTA>
Tensor call_forward(const Call& c, bool deterministic)
{
    if constexpr (DELTA) {
        static const auto op = operator_handle<decltype(jagged_delta)>("ops_rec::hstu_jagged", "delta");
        return op.call(c.q, c.k, c.v, c.mask, c.bias, c.mask_type, c.max_q, c.max_k, c.silu_scale, c.offs_q, c.offs_k, c.ctx, c.tgt, c.group, c.alpha,
                       deterministic);
    } else {
        static const auto op = operator_handle<decltype(jagged_equal)>("ops_rec::hstu_jagged", "equal");
        return op.call(c.q, c.k, c.v, c.mask, c.bias, c.mask_type, c.max_q, c.silu_scale, c.offs_q, c.ctx, c.tgt, c.group, c.alpha, deterministic);
    }
}

template <bool DELTA>
struct JaggedFunction : torch::autograd::Function<JaggedFunction<DELTA>> {
    static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& bias, const Call* call,
                          bool deterministic)
    {
        const at::AutoDispatchBelowADInplaceOrView below;
        const Call& c = *call;
        // offsets that serve both sides are saved once: saved-tensor hooks (offloading, for one) hand back a tensor per saved one, and
        // the library tells self-attention, whose pair plane takes half the room, by the two being the same
        const Tensor offs_k = c.offs_k.is_same(c.offs_q) ? Tensor() : c.offs_k;
        ctx->save_for_backward({q, k, v, unwrap(c.mask), unwrap(bias), c.offs_q, offs_k, unwrap(c.ctx), unwrap(c.tgt)});
        ctx->saved_data["ints"] = std::vector<int64_t>{c.mask_type, c.max_q, c.max_k, c.group.has_value() ? 1 : 0, c.group.value_or(0),
                                                       c.alpha.has_value() ? 1 : 0};
        ctx->saved_data["reals"] = std::vector<double>{c.silu_scale, c.alpha.value_or(1.0)};
        return call_forward<DELTA>(c, deterministic);
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        static const auto op = operator_handle<decltype(jagged_backward_delta)>("ops_rec::hstu_jagged_backward", "delta");
        const variable_list s = ctx->get_saved_variables();
        const auto ints = ctx->saved_data["ints"].toIntVector();
        const auto reals = ctx->saved_data["reals"].toDoubleVector();
        const auto group = ints[3] != 0 ? std::optional<int64_t>(ints[4]) : std::nullopt;
        const auto alpha = ints[5] != 0 ? std::optional<double>(reals[1]) : std::nullopt;
        const auto [dq, dk, dv, dbias] = op.call(grads[0], s[0], s[1], s[2], wrap(s[3]), wrap(s[4]), ints[0], ints[1], ints[2], reals[0], s[5],
                                                 s[6].defined() ? s[6] : s[5], wrap(s[7]), wrap(s[8]), group, alpha);
        return {dq, dk, dv, dbias, Tensor(), Tensor()};
    }
};

template <bool DELTA>
Tensor with_autograd(const Call& c, bool deterministic)
{
    if (!at::GradMode::is_enabled() ||
        !(needs_grad(c.q) || needs_grad(c.k) || needs_grad(c.v) || needs_grad(c.bias) || needs_grad(c.mask))) {
        const at::AutoDispatchBelowADInplaceOrView below;
        return call_forward<DELTA>(c, deterministic);
    }
    // (only a call that records a gradient is refused: under no_grad the mask is an input like any other)
    TORCH_CHECK_NOT_IMPLEMENTED(!needs_grad(c.mask), DELTA ? "hstu_jagged.delta" : "hstu_jagged.equal",
                                ": mask is a non-differentiable input (the backward op returns no mask gradient); "
                                "do not pass a mask with requires_grad=True");
    return JaggedFunction<DELTA>::apply(c.q, c.k, c.v, c.bias, &c, deterministic);
}

Tensor jagged_equal_autograd(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& mask, const OptTensor& bias, int64_t mask_type,
                             int64_t max_seq_len, double silu_scale, const Tensor& offs, const OptTensor& ctx, const OptTensor& tgt,
                             std::optional<int64_t> group, std::optional<double> alpha, bool deterministic)
{
    return with_autograd<false>({q, k, v, mask, bias, mask_type, max_seq_len, max_seq_len, silu_scale, offs, offs, ctx, tgt, group, alpha},
                                deterministic);
}

Tensor jagged_delta_autograd(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& mask, const OptTensor& bias, int64_t mask_type,
                             int64_t max_seq_len, int64_t max_seq_len_k, double silu_scale, const Tensor& offs, const Tensor& offs_k,
                             const OptTensor& ctx, const OptTensor& tgt, std::optional<int64_t> group, std::optional<double> alpha,
                             bool deterministic)
{
    return with_autograd<true>({q, k, v, mask, bias, mask_type, max_seq_len, max_seq_len_k, silu_scale, offs, offs_k, ctx, tgt, group, alpha},
                               deterministic);
}

variable_list as_list(const Projection& p)
{
    return {std::get<0>(p), std::get<1>(p), std::get<2>(p), std::get<3>(p), std::get<4>(p)};
}

struct InLinearSiluFunction : torch::autograd::Function<InLinearSiluFunction> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& weight, const OptTensor& bias, at::IntArrayRef split)
    {
        static const auto op = operator_handle<decltype(in_linear_silu)>("ops_rec::distance_in_linear_silu", "");
        const at::AutoDispatchBelowADInplaceOrView below;
        variable_list out = as_list(op.call(x, weight, unwrap(bias), split));
        // outputs nobody differentiates come back undefined: no [m, n] of zeros is made for linear_output, whose gradient the
        // formula does not take (torch_extension/_autograd.py:55-86)
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({x, weight, unwrap(bias), out[4]});
        ctx->saved_data["split"] = split.vec();
        return out;
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads)
    {
        static const auto op = operator_handle<decltype(in_linear_silu_backward)>("ops_rec::in_linear_silu_backward", "");
        const variable_list s = ctx->get_saved_variables();
        const auto split = ctx->saved_data["split"].toIntVector();
        for (size_t i = 0; i < 4; ++i) {
            if (!grads[i].defined()) {
                grads[i] = at::zeros_symint({s[0].sym_size(0), c10::SymInt(split[i])}, s[0].options());
            }
        }
        const auto r = op.call(s[0], s[1], wrap(s[2]), grads[0], grads[1], grads[2], grads[3], s[3], split);
        return {std::get<0>(r), std::get<1>(r), std::get<2>(r), Tensor()};
    }
};

Projection in_linear_silu_autograd(const Tensor& x, const Tensor& weight, const Tensor& bias, at::IntArrayRef split)
{
    if (!at::GradMode::is_enabled() || !(needs_grad(x) || needs_grad(weight) || needs_grad(bias))) {
        static const auto op = operator_handle<decltype(in_linear_silu)>("ops_rec::distance_in_linear_silu", "");
        const at::AutoDispatchBelowADInplaceOrView below;
        return op.call(x, weight, bias, split);
    }
    const variable_list out = InLinearSiluFunction::apply(x, weight, wrap(bias), split);
    return {out[0], out[1], out[2], out[3], out[4]};
}

}  // namespace

TORCH_LIBRARY_IMPL(ops_rec, CUDA, m)
{
    m.impl("hstu_jagged.equal", jagged_equal);
    m.impl("hstu_jagged.delta", jagged_delta);
    m.impl("hstu_jagged_backward.equal", jagged_backward_equal);
    m.impl("hstu_jagged_backward.delta", jagged_backward_delta);
    m.impl("hstu_paged", paged);
    m.impl("ln_mul", ln_mul);
    m.impl("distance_in_linear_silu", in_linear_silu);
    m.impl("in_linear_silu_backward", in_linear_silu_backward);
}

TORCH_LIBRARY_IMPL(ops_rec, AutogradCUDA, m)
{
    m.impl("hstu_jagged.equal", jagged_equal_autograd);
    m.impl("hstu_jagged.delta", jagged_delta_autograd);
    m.impl("distance_in_linear_silu", in_linear_silu_autograd);
}

PYBIND11_MODULE(_torch_binding, m)
{
    m.def("set_fallbacks", [](py::object forward, py::object backward, py::object paged_fn, py::object ln_mul_fn, py::object projection,
                              py::object projection_backward) {
        fallbacks.forward = forward.release().ptr();
        fallbacks.backward = backward.release().ptr();
        fallbacks.paged = paged_fn.release().ptr();
        fallbacks.ln_mul = ln_mul_fn.release().ptr();
        fallbacks.in_linear_silu = projection.release().ptr();
        fallbacks.in_linear_silu_backward = projection_backward.release().ptr();
    });
    m.def("fp8_forward", &fp8_forward, py::call_guard<py::gil_scoped_release>());
}
