// PyTorch-ROCm dispatcher registration for the cudaforge:: operators.
//
// Same namespace, the same ten schemas, the same Autograd guard list and the
// same CPU (ATen) implementations as the reference's extension
// (cpp/src/bindings.cpp:342-404), so code written against
// torch.ops.cudaforge.* runs unchanged. On ROCm a GPU tensor carries the CUDA
// dispatch key, so the GPU implementations register under CUDA; they call the
// C ABI of libcudaforge_hip.so on PyTorch's current HIP stream and never
// synchronise (bindings.cpp:56-63 does the same with the CUDA stream).
//
// Differences from the reference, all widening:
//   * the GPU implementations accept float32, bfloat16 and float16 where the
//     reference's accept float32 only (bindings.cpp:45-48); lora_linear takes
//     float32 and bfloat16;
//   * a few extra operators the Python layer uses: dequantize_int8_to (half
//     outputs), quantize_dequantize, softmax_as (output dtype),
//     softmax_scaled (scaled, causally masked attention scores), row_sum,
//     lora_linear_fwd / lora_linear_bwd / lora_linear_bwd_input for the adapter
//     autograd path, and
//     attention_scores_causal / attention_pv_causal, the two causal attention
//     products of the transformer block.
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/record_function.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/autograd_not_implemented_fallback.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <limits>
#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "cudaforge_hip.h"

namespace cudaforge_amd {
namespace {

// ---- shared checks ---------------------------------------------------------

void check_contiguous(const torch::Tensor& t, const char* name) {
    TORCH_CHECK(t.is_contiguous(), name, " must be contiguous; call .contiguous() first. ",
                "The kernels index rows as `base + row * cols`, which is only "
                "valid for a contiguous row-major layout.");
}

void check_2d(const torch::Tensor& t, const char* name) {
    TORCH_CHECK(t.dim() == 2, name, " must be 2-D, got ", t.dim(), " dimensions");
}

cf_dtype to_cf(const torch::Tensor& t, const char* name) {
    switch (t.scalar_type()) {
        case torch::kFloat32:
            return CF_F32;
        case torch::kBFloat16:
            return CF_BF16;
        case torch::kFloat16:
            return CF_F16;
        default:
            TORCH_CHECK(false, name, " has dtype ", t.scalar_type(),
                        ", which has no HIP kernel (float32, bfloat16 or float16)");
    }
}

cf_dtype to_cf(torch::ScalarType type) {
    switch (type) {
        case torch::kFloat32:
            return CF_F32;
        case torch::kBFloat16:
            return CF_BF16;
        case torch::kFloat16:
            return CF_F16;
        default:
            TORCH_CHECK(false, "dtype ", type, " has no HIP kernel (float32, bfloat16 or float16)");
    }
}

void check_same_device(const torch::Tensor& a, const torch::Tensor& b, const char* name) {
    TORCH_CHECK(a.device() == b.device(), name, " is on ", b.device(), " but the input is on ",
                a.device());
}

/// PyTorch's current stream on the tensor's device, as the C ABI's void*.
void* stream_for(const torch::Tensor& t) {
    return static_cast<void*>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

void check_status(cf_status status) {
    TORCH_CHECK(status == CF_OK, "cudaforge HIP kernel failed: ", cf_last_error());
}

// ---- GPU implementations -----------------------------------------------------

torch::Tensor rmsnorm_hip(const torch::Tensor& input, const torch::Tensor& weight, double eps) {
    check_2d(input, "input");
    check_contiguous(input, "input");
    check_contiguous(weight, "weight");
    check_same_device(input, weight, "weight");
    TORCH_CHECK(weight.dim() == 1, "weight must be 1-D, got ", weight.dim(), " dimensions");
    TORCH_CHECK(weight.size(0) == input.size(1), "weight length ", weight.size(0),
                " does not match the input's last dimension ", input.size(1));
    TORCH_CHECK(weight.scalar_type() == input.scalar_type(), "weight dtype ",
                weight.scalar_type(), " must match the input's ", input.scalar_type());
    const at::DeviceGuard guard(input.device());
    torch::Tensor output = torch::empty_like(input);
    check_status(cf_rmsnorm(input.data_ptr(), weight.data_ptr(), output.data_ptr(),
                            to_cf(input, "input"), input.size(0), input.size(1),
                            static_cast<float>(eps), stream_for(input)));
    return output;
}

torch::Tensor softmax_as_hip(const torch::Tensor& input, torch::ScalarType out_dtype) {
    check_2d(input, "input");
    check_contiguous(input, "input");
    const at::DeviceGuard guard(input.device());
    torch::Tensor output = torch::empty(input.sizes(), input.options().dtype(out_dtype));
    check_status(cf_softmax(input.data_ptr(), to_cf(input, "input"), output.data_ptr(),
                            to_cf(out_dtype), input.size(0), input.size(1), stream_for(input)));
    return output;
}

torch::Tensor softmax_hip(const torch::Tensor& input) {
    return softmax_as_hip(input, input.scalar_type());
}

torch::Tensor softmax_scaled_hip(const torch::Tensor& input, double scale, int64_t causal_period,
                                 torch::ScalarType out_dtype) {
    check_2d(input, "input");
    check_contiguous(input, "input");
    TORCH_CHECK(causal_period >= 0, "causal_period must be >= 0, got ", causal_period);
    const at::DeviceGuard guard(input.device());
    torch::Tensor output = torch::empty(input.sizes(), input.options().dtype(out_dtype));
    check_status(cf_softmax_scaled(input.data_ptr(), to_cf(input, "input"), output.data_ptr(),
                                   to_cf(out_dtype), input.size(0), input.size(1),
                                   static_cast<float>(scale), causal_period, stream_for(input)));
    return output;
}

// Causal attention products: q, k, v [batch, seq, heads * head_dim],
// probs [batch, heads, seq, seq].
void check_attention(const torch::Tensor& rows, int64_t heads, const char* name) {
    TORCH_CHECK(rows.dim() == 3, name, " must be [batch, seq, hidden], got ", rows.dim(), " dims");
    TORCH_CHECK(heads > 0 && rows.size(2) % heads == 0, "hidden ", rows.size(2), " is not divisible by heads ",
                heads);
}

torch::Tensor attention_scores_causal_hip(const torch::Tensor& q, const torch::Tensor& k, int64_t heads) {
    check_attention(q, heads, "q");
    TORCH_CHECK(k.sizes() == q.sizes(), "q and k differ in shape");
    TORCH_CHECK(k.scalar_type() == q.scalar_type(), "q and k differ in dtype");
    check_same_device(q, k, "k");
    check_contiguous(q, "q");
    check_contiguous(k, "k");
    const at::DeviceGuard guard(q.device());
    const int64_t batch = q.size(0), seq = q.size(1);
    torch::Tensor scores = torch::empty({batch, heads, seq, seq}, q.options());
    check_status(cf_attention_scores_causal(q.data_ptr(), k.data_ptr(), scores.data_ptr(), to_cf(q, "q"), batch,
                                            seq, heads, q.size(2) / heads, stream_for(q)));
    return scores;
}

torch::Tensor attention_pv_causal_hip(const torch::Tensor& probs, const torch::Tensor& v, int64_t heads) {
    check_attention(v, heads, "v");
    const int64_t batch = v.size(0), seq = v.size(1);
    TORCH_CHECK(probs.dim() == 4 && probs.size(0) == batch && probs.size(1) == heads && probs.size(2) == seq &&
                    probs.size(3) == seq,
                "probs must be [batch, heads, seq, seq] = [", batch, ", ", heads, ", ", seq, ", ", seq, "]");
    TORCH_CHECK(probs.scalar_type() == v.scalar_type(), "probs and v differ in dtype");
    check_same_device(v, probs, "probs");
    check_contiguous(probs, "probs");
    check_contiguous(v, "v");
    const at::DeviceGuard guard(v.device());
    torch::Tensor out = torch::empty(v.sizes(), v.options());
    check_status(cf_attention_pv_causal(probs.data_ptr(), v.data_ptr(), out.data_ptr(), to_cf(v, "v"), batch, seq,
                                        heads, v.size(2) / heads, stream_for(v)));
    return out;
}

std::tuple<torch::Tensor, torch::Tensor> lora_linear_fwd_hip(const torch::Tensor& x,
                                                             const torch::Tensor& w,
                                                             const torch::Tensor& a,
                                                             const torch::Tensor& b,
                                                             double scale) {
    check_2d(x, "x");
    check_2d(w, "w");
    check_2d(a, "a");
    check_2d(b, "b");
    for (const auto& [tensor, name] : {std::pair<const torch::Tensor*, const char*>{&x, "x"},
                                       {&w, "w"}, {&a, "a"}, {&b, "b"}}) {
        check_contiguous(*tensor, name);
        check_same_device(x, *tensor, name);
        TORCH_CHECK(tensor->scalar_type() == x.scalar_type(), name, " has dtype ",
                    tensor->scalar_type(), " but x has ", x.scalar_type());
    }
    TORCH_CHECK(x.scalar_type() == torch::kFloat32 || x.scalar_type() == torch::kBFloat16,
                "lora_linear has HIP kernels for float32 and bfloat16, got ", x.scalar_type());
    const int64_t batch = x.size(0);
    const int64_t in_features = x.size(1);
    const int64_t out_features = w.size(1);
    const int64_t rank = a.size(1);
    TORCH_CHECK(w.size(0) == in_features, "w must be [in_features, out_features]; got [",
                w.size(0), ", ", w.size(1), "] for in_features=", in_features);
    TORCH_CHECK(a.size(0) == in_features, "a must be [in_features, rank]; got [", a.size(0), ", ",
                a.size(1), "] for in_features=", in_features);
    TORCH_CHECK(b.size(0) == rank && b.size(1) == out_features,
                "b must be [rank, out_features] = [", rank, ", ", out_features, "]; got [",
                b.size(0), ", ", b.size(1), "]");
    const at::DeviceGuard guard(x.device());
    torch::Tensor output = torch::empty({batch, out_features}, x.options());
    torch::Tensor xa = torch::empty({batch, rank}, x.options().dtype(torch::kFloat32));
    // Partial sums go through a workspace from torch's caching allocator (no
    // synchronising hipMalloc).
    const size_t ws_bytes =
        cf_lora_forward_workspace_bytes(to_cf(x, "x"), batch, in_features, out_features, rank);
    torch::Tensor workspace =
        torch::empty({static_cast<int64_t>(ws_bytes > 0 ? ws_bytes : 1)}, x.options().dtype(torch::kUInt8));
    check_status(cf_lora_forward(x.data_ptr(), w.data_ptr(), a.data_ptr(), b.data_ptr(),
                                 output.data_ptr(), xa.data_ptr<float>(), to_cf(x, "x"), batch,
                                 in_features, out_features, rank, static_cast<float>(scale),
                                 ws_bytes > 0 ? workspace.data_ptr() : nullptr, ws_bytes,
                                 stream_for(x)));
    return {output, xa};
}

torch::Tensor lora_linear_hip(const torch::Tensor& x, const torch::Tensor& w,
                              const torch::Tensor& a, const torch::Tensor& b, double scale) {
    return std::get<0>(lora_linear_fwd_hip(x, w, a, b, scale));
}

bool aligned16(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// Adapter gradients; with w and a also the input gradient: the plain GEMM
// dy @ w^T through the vendor BLAS, the adapter's part added in place (by the
// BLAS too where the library says that is the faster way).
std::tuple<torch::Tensor, torch::Tensor, torch::Tensor> lora_backward_hip(
    const torch::Tensor& x, const torch::Tensor& dy, const torch::Tensor* w, const torch::Tensor* a,
    const torch::Tensor& b, const torch::Tensor& xa, double scale) {
    check_2d(x, "x");
    check_2d(dy, "dy");
    check_2d(b, "b");
    check_2d(xa, "xa");
    for (const auto& [tensor, name] : {std::pair<const torch::Tensor*, const char*>{&x, "x"},
                                       {&dy, "dy"}, {&b, "b"}, {&xa, "xa"}}) {
        check_contiguous(*tensor, name);
        check_same_device(x, *tensor, name);
    }
    TORCH_CHECK(dy.scalar_type() == x.scalar_type() && b.scalar_type() == x.scalar_type(),
                "x, dy and b must share a dtype");
    TORCH_CHECK(xa.scalar_type() == torch::kFloat32, "xa must be float32");
    const int64_t batch = x.size(0);
    const int64_t in_features = x.size(1);
    const int64_t rank = b.size(0);
    const int64_t out_features = b.size(1);
    TORCH_CHECK(dy.size(0) == batch && dy.size(1) == out_features, "dy must be [", batch, ", ",
                out_features, "]");
    TORCH_CHECK(xa.size(0) == batch && xa.size(1) == rank, "xa must be [", batch, ", ", rank, "]");
    if (w != nullptr) {
        for (const auto& [tensor, name] : {std::pair<const torch::Tensor*, const char*>{w, "w"}, {a, "a"}}) {
            check_2d(*tensor, name);
            check_contiguous(*tensor, name);
            check_same_device(x, *tensor, name);
            TORCH_CHECK(tensor->scalar_type() == x.scalar_type(), "x and ", name, " must share a dtype");
        }
        TORCH_CHECK(w->size(0) == in_features && w->size(1) == out_features, "w must be [", in_features,
                    ", ", out_features, "]");
        TORCH_CHECK(a->size(0) == in_features && a->size(1) == rank, "a must be [", in_features, ", ",
                    rank, "]");
    }
    const at::DeviceGuard guard(x.device());
    torch::Tensor grad_x;
    bool own_update = false;
    if (w != nullptr) {
        // A backward inside an autocast block runs here with its keys on: mm
        // would then return another dtype than the kernel below is told.
        const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
        grad_x = at::mm(dy, w->t());
        TORCH_CHECK(grad_x.scalar_type() == x.scalar_type() && grad_x.is_contiguous() &&
                        grad_x.sizes() == x.sizes(),
                    "dy @ w^T is not a contiguous ", x.scalar_type(), " tensor of x's shape");
        own_update = aligned16(x) && aligned16(dy) && aligned16(b) &&
                     cf_lora_backward_updates_input(to_cf(x, "x"), batch, in_features, out_features, rank) != 0;
        if (!own_update) {
            const torch::Tensor g = at::mm(dy, b.t());
            // A GEMM with alpha = 0 reads nothing, and 0 * inf is NaN.
            scale != 0.0 ? grad_x.addmm_(g, a->t(), 1, scale) : grad_x.add_(at::mm(g, a->t()), scale);
        }
    }
    torch::Tensor grad_a = torch::empty({in_features, rank}, x.options());
    torch::Tensor grad_b = torch::empty({rank, out_features}, x.options());
    const size_t bytes =
        cf_lora_backward_dtype_workspace_bytes(to_cf(x, "x"), batch, in_features, out_features, rank);
    torch::Tensor workspace =
        torch::empty({static_cast<int64_t>(bytes > 0 ? bytes : 1)}, x.options().dtype(torch::kUInt8));
    check_status(cf_lora_backward_input(
        x.data_ptr(), dy.data_ptr(), a != nullptr ? a->data_ptr() : nullptr, b.data_ptr(),
        xa.data_ptr<float>(), grad_a.data_ptr(), grad_b.data_ptr(),
        own_update ? grad_x.data_ptr() : nullptr, to_cf(x, "x"), batch, in_features, out_features, rank,
        static_cast<float>(scale), workspace.data_ptr(), bytes, stream_for(x)));
    return {grad_x, grad_a, grad_b};
}

std::tuple<torch::Tensor, torch::Tensor> lora_linear_bwd_hip(const torch::Tensor& x,
                                                             const torch::Tensor& dy,
                                                             const torch::Tensor& b,
                                                             const torch::Tensor& xa,
                                                             double scale) {
    auto [grad_x, grad_a, grad_b] = lora_backward_hip(x, dy, nullptr, nullptr, b, xa, scale);
    return {grad_a, grad_b};
}

std::tuple<torch::Tensor, torch::Tensor, torch::Tensor> lora_linear_bwd_input_hip(
    const torch::Tensor& x, const torch::Tensor& dy, const torch::Tensor& w, const torch::Tensor& a,
    const torch::Tensor& b, const torch::Tensor& xa, double scale) {
    return lora_backward_hip(x, dy, &w, &a, b, xa, scale);
}

std::vector<torch::Tensor> fused_residual_rmsnorm_hip(const torch::Tensor& x,
                                                      const torch::Tensor& residual,
                                                      const torch::Tensor& weight, double eps) {
    check_2d(x, "x");
    check_contiguous(x, "x");
    check_contiguous(residual, "residual");
    check_contiguous(weight, "weight");
    check_same_device(x, residual, "residual");
    check_same_device(x, weight, "weight");
    TORCH_CHECK(x.sizes() == residual.sizes(), "x and residual must have the same shape, got ",
                x.sizes(), " and ", residual.sizes());
    TORCH_CHECK(weight.dim() == 1 && weight.size(0) == x.size(1), "weight must be 1-D of length ",
                x.size(1), ", got ", weight.sizes());
    TORCH_CHECK(residual.scalar_type() == x.scalar_type() &&
                    weight.scalar_type() == x.scalar_type(),
                "x, residual and weight must share a dtype");
    const at::DeviceGuard guard(x.device());
    torch::Tensor output = torch::empty_like(x);
    torch::Tensor residual_out = torch::empty_like(x);
    check_status(cf_fused_residual_rmsnorm(x.data_ptr(), residual.data_ptr(), weight.data_ptr(),
                                           output.data_ptr(), residual_out.data_ptr(),
                                           to_cf(x, "x"), x.size(0), x.size(1),
                                           static_cast<float>(eps), stream_for(x)));
    return {output, residual_out};
}

torch::Tensor silu_hip(const torch::Tensor& input) {
    check_contiguous(input, "input");
    const at::DeviceGuard guard(input.device());
    torch::Tensor output = torch::empty_like(input);
    check_status(cf_silu(input.data_ptr(), output.data_ptr(), to_cf(input, "input"),
                         input.numel(), stream_for(input)));
    return output;
}

torch::Tensor gelu_hip(const torch::Tensor& input) {
    check_contiguous(input, "input");
    const at::DeviceGuard guard(input.device());
    torch::Tensor output = torch::empty_like(input);
    check_status(cf_gelu(input.data_ptr(), output.data_ptr(), to_cf(input, "input"),
                         input.numel(), stream_for(input)));
    return output;
}

torch::Tensor swiglu_hip(const torch::Tensor& gate, const torch::Tensor& up) {
    check_contiguous(gate, "gate");
    check_contiguous(up, "up");
    check_same_device(gate, up, "up");
    TORCH_CHECK(gate.sizes() == up.sizes(), "gate and up must have the same shape, got ",
                gate.sizes(), " and ", up.sizes());
    TORCH_CHECK(gate.scalar_type() == up.scalar_type(), "gate and up must have the same dtype");
    const at::DeviceGuard guard(gate.device());
    torch::Tensor output = torch::empty_like(gate);
    check_status(cf_swiglu(gate.data_ptr(), up.data_ptr(), output.data_ptr(),
                           to_cf(gate, "gate"), gate.numel(), stream_for(gate)));
    return output;
}

torch::Tensor sum_hip(const torch::Tensor& input) {
    check_contiguous(input, "input");
    const at::DeviceGuard guard(input.device());
    const cf_dtype dtype = to_cf(input, "input");
    // accumulate = 0: the kernel writes the sum, so no fill is needed (and
    // none is recorded when the op is captured into a graph).
    const int64_t count = input.numel();
    if (count == 0) return torch::zeros({}, input.options());
    torch::Tensor out = torch::empty({1}, input.options().dtype(torch::kFloat32));
    {
        const size_t bytes = cf_reduce_sum_workspace_bytes(count);
        torch::Tensor workspace =
            torch::empty({static_cast<int64_t>(bytes)}, input.options().dtype(torch::kUInt8));
        check_status(cf_reduce_sum(input.data_ptr(), dtype, out.data_ptr<float>(), count,
                                   workspace.data_ptr(), bytes, /*accumulate=*/0,
                                   stream_for(input)));
    }
    return out.squeeze().to(input.scalar_type());
}

torch::Tensor row_sum_hip(const torch::Tensor& input) {
    check_2d(input, "input");
    check_contiguous(input, "input");
    const at::DeviceGuard guard(input.device());
    torch::Tensor out = torch::empty({input.size(0)}, input.options().dtype(torch::kFloat32));
    check_status(cf_row_sum(input.data_ptr(), to_cf(input, "input"), out.data_ptr<float>(),
                            input.size(0), input.size(1), stream_for(input)));
    return out;
}

std::vector<torch::Tensor> quantize_int8_hip(const torch::Tensor& input) {
    check_contiguous(input, "input");
    const at::DeviceGuard guard(input.device());
    const int64_t count = input.numel();
    torch::Tensor quantised = torch::empty({count}, input.options().dtype(torch::kInt8));
    torch::Tensor scales =
        torch::empty({cf_quant_scale_count(count)}, input.options().dtype(torch::kFloat32));
    check_status(cf_quantize_int8(input.data_ptr(), to_cf(input, "input"),
                                  quantised.data_ptr<int8_t>(), scales.data_ptr<float>(), count,
                                  stream_for(input)));
    return {quantised.view(input.sizes()), scales};
}

torch::Tensor dequantize_int8_to_hip(const torch::Tensor& quantised, const torch::Tensor& scales,
                                     torch::ScalarType out_dtype) {
    TORCH_CHECK(quantised.scalar_type() == torch::kInt8, "quantised must be int8");
    TORCH_CHECK(scales.scalar_type() == torch::kFloat32, "scales must be float32, got ",
                scales.scalar_type());
    check_contiguous(quantised, "quantised");
    check_contiguous(scales, "scales");
    check_same_device(quantised, scales, "scales");
    const int64_t count = quantised.numel();
    TORCH_CHECK(scales.numel() == cf_quant_scale_count(count), "expected ",
                cf_quant_scale_count(count), " block scales, got ", scales.numel());
    const at::DeviceGuard guard(quantised.device());
    torch::Tensor output = torch::empty(quantised.sizes(), scales.options().dtype(out_dtype));
    check_status(cf_dequantize_int8(quantised.data_ptr<int8_t>(), scales.data_ptr<float>(),
                                    output.data_ptr(), to_cf(out_dtype), count,
                                    stream_for(quantised)));
    return output;
}

torch::Tensor dequantize_int8_hip(const torch::Tensor& quantised, const torch::Tensor& scales) {
    return dequantize_int8_to_hip(quantised, scales, scales.scalar_type());
}

torch::Tensor quantize_dequantize_hip(const torch::Tensor& input) {
    check_contiguous(input, "input");
    const at::DeviceGuard guard(input.device());
    torch::Tensor output = torch::empty_like(input);
    check_status(cf_quantize_dequantize(input.data_ptr(), output.data_ptr(),
                                        to_cf(input, "input"), input.numel(),
                                        stream_for(input)));
    return output;
}

// ---- CPU implementations (ATen), as the reference's ----------------------------

torch::Tensor rmsnorm_cpu(const torch::Tensor& input, const torch::Tensor& weight, double eps) {
    check_2d(input, "input");
    TORCH_CHECK(weight.size(0) == input.size(1), "weight length ", weight.size(0),
                " does not match the input's last dimension ", input.size(1));
    const torch::Tensor promoted = input.to(torch::kFloat32);
    const torch::Tensor variance = promoted.pow(2).mean(-1, /*keepdim=*/true);
    const torch::Tensor normalised = promoted * torch::rsqrt(variance + eps);
    return (normalised * weight.to(torch::kFloat32)).to(input.scalar_type());
}

torch::Tensor softmax_cpu(const torch::Tensor& input) {
    check_2d(input, "input");
    return torch::softmax(input, /*dim=*/-1);
}

torch::Tensor softmax_as_cpu(const torch::Tensor& input, torch::ScalarType out_dtype) {
    check_2d(input, "input");
    return torch::softmax(input.to(torch::kFloat32), /*dim=*/-1).to(out_dtype);
}

torch::Tensor softmax_scaled_cpu(const torch::Tensor& input, double scale, int64_t causal_period,
                                 torch::ScalarType out_dtype) {
    check_2d(input, "input");
    TORCH_CHECK(causal_period >= 0, "causal_period must be >= 0, got ", causal_period);
    torch::Tensor logits = input.to(torch::kFloat32) * scale;
    if (causal_period > 0) {
        const auto options = torch::TensorOptions().dtype(torch::kLong).device(input.device());
        const torch::Tensor cols = torch::arange(input.size(1), options).unsqueeze(0);
        const torch::Tensor rows =
            torch::remainder(torch::arange(input.size(0), options), causal_period).unsqueeze(1);
        logits = logits.masked_fill(cols > rows, -std::numeric_limits<float>::infinity());
    }
    return torch::softmax(logits, /*dim=*/-1).to(out_dtype);
}

// The same products on the CPU: heads split out, the full q k^T (the
// kernel leaves the entries above the diagonal unspecified; these hold their
// dot products) and the lower triangle of probs times v.
torch::Tensor attention_scores_causal_cpu(const torch::Tensor& q, const torch::Tensor& k, int64_t heads) {
    check_attention(q, heads, "q");
    TORCH_CHECK(k.sizes() == q.sizes(), "q and k differ in shape");
    const int64_t batch = q.size(0), seq = q.size(1), d = q.size(2) / heads;
    const torch::Tensor qh = q.view({batch, seq, heads, d}).transpose(1, 2).to(torch::kFloat32);
    const torch::Tensor kh = k.view({batch, seq, heads, d}).transpose(1, 2).to(torch::kFloat32);
    return torch::matmul(qh, kh.transpose(-2, -1)).to(q.scalar_type());
}

torch::Tensor attention_pv_causal_cpu(const torch::Tensor& probs, const torch::Tensor& v, int64_t heads) {
    check_attention(v, heads, "v");
    const int64_t batch = v.size(0), seq = v.size(1), d = v.size(2) / heads;
    TORCH_CHECK(probs.dim() == 4 && probs.size(0) == batch && probs.size(1) == heads && probs.size(2) == seq &&
                    probs.size(3) == seq,
                "probs must be [batch, heads, seq, seq] = [", batch, ", ", heads, ", ", seq, ", ", seq, "]");
    const torch::Tensor vh = v.view({batch, seq, heads, d}).transpose(1, 2).to(torch::kFloat32);
    const torch::Tensor out = torch::matmul(torch::tril(probs.to(torch::kFloat32)), vh);
    return out.transpose(1, 2).reshape({batch, seq, heads * d}).to(v.scalar_type());
}

torch::Tensor lora_linear_cpu(const torch::Tensor& x, const torch::Tensor& w,
                              const torch::Tensor& a, const torch::Tensor& b, double scale) {
    return torch::matmul(x, w) + scale * torch::matmul(torch::matmul(x, a), b);
}

std::tuple<torch::Tensor, torch::Tensor> lora_linear_fwd_cpu(const torch::Tensor& x,
                                                             const torch::Tensor& w,
                                                             const torch::Tensor& a,
                                                             const torch::Tensor& b,
                                                             double scale) {
    const torch::Tensor xa = torch::matmul(x.to(torch::kFloat32), a.to(torch::kFloat32));
    const torch::Tensor y =
        torch::matmul(x, w) + scale * torch::matmul(xa.to(x.scalar_type()), b);
    return {y, xa};
}

std::tuple<torch::Tensor, torch::Tensor> lora_linear_bwd_cpu(const torch::Tensor& x,
                                                             const torch::Tensor& dy,
                                                             const torch::Tensor& b,
                                                             const torch::Tensor& xa,
                                                             double scale) {
    const auto type = x.scalar_type();
    const torch::Tensor xf = x.to(torch::kFloat32);
    const torch::Tensor dyf = dy.to(torch::kFloat32);
    const torch::Tensor g = torch::matmul(dyf, b.to(torch::kFloat32).t()).to(type).to(torch::kFloat32);
    const torch::Tensor grad_a = (scale * torch::matmul(xf.t(), g)).to(type);
    const torch::Tensor grad_b =
        (scale * torch::matmul(xa.to(type).to(torch::kFloat32).t(), dyf)).to(type);
    return {grad_a, grad_b};
}

std::tuple<torch::Tensor, torch::Tensor, torch::Tensor> lora_linear_bwd_input_cpu(
    const torch::Tensor& x, const torch::Tensor& dy, const torch::Tensor& w, const torch::Tensor& a,
    const torch::Tensor& b, const torch::Tensor& xa, double scale) {
    // As on the GPU: the operands' dtype, whatever autocast is on.
    const c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
    const torch::Tensor grad_x =
        torch::matmul(dy, w.t()) + scale * torch::matmul(torch::matmul(dy, b.t()), a.t());
    auto [grad_a, grad_b] = lora_linear_bwd_cpu(x, dy, b, xa, scale);
    return {grad_x, grad_a, grad_b};
}

torch::Tensor sum_cpu(const torch::Tensor& input) { return input.sum(); }

torch::Tensor row_sum_cpu(const torch::Tensor& input) {
    check_2d(input, "input");
    return input.to(torch::kFloat32).sum(-1);
}

std::vector<torch::Tensor> fused_residual_rmsnorm_cpu(const torch::Tensor& x,
                                                      const torch::Tensor& residual,
                                                      const torch::Tensor& weight, double eps) {
    TORCH_CHECK(x.sizes() == residual.sizes(), "x and residual must have the same shape, got ",
                x.sizes(), " and ", residual.sizes());
    const torch::Tensor summed = x + residual;
    return {rmsnorm_cpu(summed, weight, eps), summed};
}

torch::Tensor silu_cpu(const torch::Tensor& input) { return torch::silu(input); }

torch::Tensor gelu_cpu(const torch::Tensor& input) { return torch::gelu(input, "tanh"); }

torch::Tensor swiglu_cpu(const torch::Tensor& gate, const torch::Tensor& up) {
    TORCH_CHECK(gate.sizes() == up.sizes(), "gate and up must have the same shape, got ",
                gate.sizes(), " and ", up.sizes());
    if (gate.scalar_type() == torch::kHalf || gate.scalar_type() == torch::kBFloat16) {
        return (torch::silu(gate.to(torch::kFloat32)) * up.to(torch::kFloat32))
            .to(gate.scalar_type());
    }
    return torch::silu(gate) * up;
}

std::vector<torch::Tensor> quantize_int8_cpu(const torch::Tensor& input) {
    const int64_t count = input.numel();
    const int64_t block = 64;
    const int64_t blocks = (count + block - 1) / block;
    const torch::Tensor flat = input.reshape({-1}).to(torch::kFloat32);
    const torch::Tensor padded = torch::constant_pad_nd(flat, {0, blocks * block - count}, 0.0);
    const torch::Tensor grouped = padded.reshape({blocks, block});
    torch::Tensor scales = std::get<0>(grouped.abs().max(/*dim=*/1)) / 127.0;
    scales = torch::where(scales > 0, scales, torch::ones_like(scales));
    const torch::Tensor quantised =
        torch::clamp(torch::round(grouped / scales.unsqueeze(1)), -127, 127)
            .reshape({-1})
            .slice(0, 0, count)
            .to(torch::kInt8);
    return {quantised.view_as(input), scales};
}

torch::Tensor dequantize_int8_cpu(const torch::Tensor& quantised, const torch::Tensor& scales) {
    const int64_t count = quantised.numel();
    const int64_t block = 64;
    const int64_t blocks = (count + block - 1) / block;
    const torch::Tensor flat = quantised.reshape({-1}).to(torch::kFloat32);
    const torch::Tensor padded = torch::constant_pad_nd(flat, {0, blocks * block - count}, 0.0);
    const torch::Tensor grouped = padded.reshape({blocks, block});
    return (grouped * scales.unsqueeze(1)).reshape({-1}).slice(0, 0, count).view_as(quantised);
}

torch::Tensor dequantize_int8_to_cpu(const torch::Tensor& quantised, const torch::Tensor& scales,
                                     torch::ScalarType out_dtype) {
    return dequantize_int8_cpu(quantised, scales).to(out_dtype);
}

torch::Tensor quantize_dequantize_cpu(const torch::Tensor& input) {
    const auto parts = quantize_int8_cpu(input);
    return dequantize_int8_cpu(parts[0], parts[1]).to(input.scalar_type());
}

bool cuda_kernels_available() { return true; }

// ---- direct entry for ordinary GPU calls ---------------------------------------
//
// A call from Python through torch.ops costs 4-5 us of host time (schema
// parsing, boxing, the autograd fallback) on top of the checks in ops.py, more
// than the smallest kernels take. The try_* functions below are what ops.py
// asks first: when a call is an ordinary one they run the HIP implementation
// directly, otherwise they return None and ops.py goes its general way
// (validation messages, copies of non-contiguous inputs, fallbacks, the
// dispatcher). A call is ordinary when every tensor is a plain dense GPU tensor
// (exact type, no dispatch key beyond CUDA and its autograd), nothing is
// tracing, profiling, transforming or overriding it, no gradient is needed,
// and the arguments are ones the general way would pass to the same HIP
// implementation unchanged.

bool ordinary_context() {
    // Dispatch keys switched on for the thread: beyond these two, a mode
    // (tracing, functorch, Python dispatch) is active; autocast's key is always
    // on a tensor and excluded for the thread unless autocast is on.
    static const c10::DispatchKeySet usual({c10::DispatchKey::BackendSelect, c10::DispatchKey::ADInplaceOrView});
    const c10::impl::LocalDispatchKeySet local = c10::impl::tls_local_dispatch_key_set();
    return (local.included_.raw_repr() & ~usual.raw_repr()) == 0 &&
           local.excluded_.has(c10::DispatchKey::AutocastCUDA) && !at::impl::torch_function_mode_enabled() && !at::hasCallbacks();
}

/// Dense GPU storage, no dispatch key beyond CUDA and its autograd, and no
/// forward-mode tangent.
bool plain_gpu(const at::Tensor& t) {
    static const c10::DispatchKeySet usual(
        {c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA,
         c10::DispatchKey::ADInplaceOrView});
    return t.defined() && t.key_set().has(c10::DispatchKey::CUDA) &&
           (t.key_set().raw_repr() & ~usual.raw_repr()) == 0 && !t._fw_grad(0).defined();
}

/// The tensor behind `object`, or null when it is not a plain GPU tensor that
/// is contiguous and not empty.
const at::Tensor* ordinary(py::handle object) {
    if (!THPVariable_CheckTypeExact(Py_TYPE(object.ptr()))) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(object.ptr());
    return plain_gpu(t) && t.is_contiguous() && t.numel() > 0 ? &t : nullptr;
}

// The other arguments come as Python objects: a value that is not plainly a
// number or a dtype (a tensor, a NumPy type, a bool, an int out of range) is
// left to the general way, whose conversions and errors stand.

std::optional<double> plain_double(py::handle object) {
    if (PyFloat_Check(object.ptr())) return PyFloat_AS_DOUBLE(object.ptr());
    if (!PyLong_CheckExact(object.ptr())) return std::nullopt;
    const double value = PyLong_AsDouble(object.ptr());
    if (value == -1.0 && PyErr_Occurred() != nullptr) {
        PyErr_Clear();
        return std::nullopt;
    }
    return value;
}

std::optional<int64_t> plain_int(py::handle object) {
    if (!PyLong_CheckExact(object.ptr())) return std::nullopt;
    int overflow = 0;
    const long long value = PyLong_AsLongLongAndOverflow(object.ptr(), &overflow);
    return overflow == 0 ? std::optional<int64_t>(value) : std::nullopt;
}

/// The dtype given, `otherwise` for None, nothing for any other object or a
/// dtype without kernels.
std::optional<at::ScalarType> plain_dtype(py::handle object, at::ScalarType otherwise) {
    if (!object.is_none() && !THPDtype_Check(object.ptr())) return std::nullopt;
    const at::ScalarType t = object.is_none() ? otherwise : reinterpret_cast<THPDtype*>(object.ptr())->scalar_type;
    return t == torch::kFloat32 || t == torch::kBFloat16 || t == torch::kFloat16 ? std::optional<at::ScalarType>(t)
                                                                                 : std::nullopt;
}

bool kernel_dtype(at::ScalarType t) {
    return t == torch::kFloat32 || t == torch::kBFloat16 || t == torch::kFloat16;
}

bool grad_needed(std::initializer_list<const at::Tensor*> tensors) {
    if (!at::GradMode::is_enabled()) return false;
    for (const at::Tensor* t : tensors) {
        if (t->requires_grad()) return true;
    }
    return false;
}

/// Plain, same dtype and device, a dtype with kernels, no gradient needed.
bool ordinary_set(std::initializer_list<const at::Tensor*> tensors) {
    const at::Tensor* first = *tensors.begin();
    for (const at::Tensor* t : tensors) {
        if (t == nullptr || t->scalar_type() != first->scalar_type() || t->device() != first->device()) return false;
    }
    return kernel_dtype(first->scalar_type()) && !grad_needed(tensors);
}

py::object wrap(const at::Tensor& t) { return py::reinterpret_steal<py::object>(THPVariable_Wrap(t)); }

/// `fn` on x as [rows, last dim], the result in x's shape.
template <typename Fn>
py::object by_rows(const at::Tensor& x, Fn fn) {
    at::Tensor y;
    {
        py::gil_scoped_release no_gil;
        if (x.dim() == 2) {
            y = fn(x);
        } else {
            y = fn(x.view({-1, x.size(-1)})).view(x.sizes());
        }
    }
    return wrap(y);
}

py::object try_rmsnorm(py::handle x_, py::handle weight_, py::handle eps_) {
    const at::Tensor* x = ordinary(x_);
    const at::Tensor* w = ordinary(weight_);
    const std::optional<double> eps = plain_double(eps_);
    if (x == nullptr || w == nullptr || !eps || !ordinary_context() || !ordinary_set({x, w})) return py::none();
    if (x->dim() < 1 || w->dim() != 1 || x->size(-1) != w->size(0)) return py::none();
    return by_rows(*x, [&](const at::Tensor& rows) { return rmsnorm_hip(rows, *w, *eps); });
}

py::object try_fused_residual_rmsnorm(py::handle x_, py::handle residual_, py::handle weight_, py::handle eps_) {
    const at::Tensor* x = ordinary(x_);
    const at::Tensor* r = ordinary(residual_);
    const at::Tensor* w = ordinary(weight_);
    const std::optional<double> eps = plain_double(eps_);
    if (x == nullptr || r == nullptr || w == nullptr || !eps || !ordinary_context() || !ordinary_set({x, r, w})) {
        return py::none();
    }
    if (x->dim() != 2 || r->sizes() != x->sizes() || w->dim() != 1 || x->size(1) != w->size(0)) return py::none();
    std::vector<at::Tensor> out;
    {
        py::gil_scoped_release no_gil;
        out = fused_residual_rmsnorm_hip(*x, *r, *w, *eps);
    }
    return py::make_tuple(wrap(out[0]), wrap(out[1]));
}

py::object try_softmax(py::handle x_, py::handle dtype_) {
    const at::Tensor* x = ordinary(x_);
    if (x == nullptr || !ordinary_context() || !ordinary_set({x}) || x->dim() < 1) return py::none();
    const std::optional<at::ScalarType> out = plain_dtype(dtype_, x->scalar_type());
    if (!out) return py::none();
    return by_rows(*x, [&](const at::Tensor& rows) { return softmax_as_hip(rows, *out); });
}

py::object try_softmax_scaled(py::handle x_, py::handle scale_, py::handle causal_period_, py::handle dtype_) {
    const at::Tensor* x = ordinary(x_);
    if (x == nullptr || !ordinary_context() || !ordinary_set({x}) || x->dim() < 1) return py::none();
    const std::optional<double> scale = plain_double(scale_);
    const std::optional<int64_t> period = plain_int(causal_period_);
    const std::optional<at::ScalarType> out = plain_dtype(dtype_, x->scalar_type());
    if (!scale || !period || !out || *period < 0) return py::none();
    return by_rows(*x, [&](const at::Tensor& rows) { return softmax_scaled_hip(rows, *scale, *period, *out); });
}

template <at::Tensor (*kFn)(const at::Tensor&)>
py::object try_unary(py::handle x_) {
    const at::Tensor* x = ordinary(x_);
    if (x == nullptr || !ordinary_context() || !ordinary_set({x})) return py::none();
    at::Tensor y;
    {
        py::gil_scoped_release no_gil;
        y = kFn(*x);
    }
    return wrap(y);
}

py::object try_swiglu(py::handle gate_, py::handle up_) {
    const at::Tensor* gate = ordinary(gate_);
    const at::Tensor* up = ordinary(up_);
    if (gate == nullptr || up == nullptr || !ordinary_context() || !ordinary_set({gate, up})) return py::none();
    if (gate->sizes() != up->sizes()) return py::none();
    at::Tensor y;
    {
        py::gil_scoped_release no_gil;
        y = swiglu_hip(*gate, *up);
    }
    return wrap(y);
}

py::object try_quantize_int8(py::handle x_) {
    const at::Tensor* x = ordinary(x_);
    if (x == nullptr || !ordinary_context() || !ordinary_set({x})) return py::none();
    std::vector<at::Tensor> out;
    {
        py::gil_scoped_release no_gil;
        out = quantize_int8_hip(*x);
    }
    return py::make_tuple(wrap(out[0]), wrap(out[1]));
}

py::object try_dequantize_int8(py::handle codes_, py::handle scales_, py::handle dtype_) {
    const at::Tensor* codes = ordinary(codes_);
    const at::Tensor* scales = ordinary(scales_);
    if (codes == nullptr || scales == nullptr || !ordinary_context()) return py::none();
    const std::optional<at::ScalarType> out = plain_dtype(dtype_, torch::kFloat32);
    if (codes->scalar_type() != torch::kInt8 || scales->scalar_type() != torch::kFloat32 ||
        codes->device() != scales->device() || !out || grad_needed({scales}) ||
        scales->numel() != cf_quant_scale_count(codes->numel())) {
        return py::none();
    }
    at::Tensor y;
    {
        py::gil_scoped_release no_gil;
        y = dequantize_int8_to_hip(*codes, *scales, *out);
    }
    return wrap(y);
}

/// [batch, seq, hidden] rows of bf16 that the causal attention kernels take.
bool attention_rows(const at::Tensor& t, int64_t heads) {
    if (t.scalar_type() != torch::kBFloat16 || t.dim() != 3 || heads <= 0 || t.size(2) % heads != 0) return false;
    const int64_t d = t.size(2) / heads;
    return (d == 32 || d == 64 || d == 96 || d == 128) && t.size(1) % 8 == 0;
}

py::object try_attention_scores(py::handle q_, py::handle k_, py::handle heads_) {
    const at::Tensor* q = ordinary(q_);
    const at::Tensor* k = ordinary(k_);
    const std::optional<int64_t> heads = plain_int(heads_);
    if (q == nullptr || k == nullptr || !heads || !ordinary_context() || !ordinary_set({q, k})) return py::none();
    if (!attention_rows(*q, *heads) || k->sizes() != q->sizes() || !aligned16(*q) || !aligned16(*k)) return py::none();
    at::Tensor y;
    {
        py::gil_scoped_release no_gil;
        y = attention_scores_causal_hip(*q, *k, *heads);
    }
    return wrap(y);
}

py::object try_attention_pv(py::handle probs_, py::handle v_, py::handle heads_) {
    const at::Tensor* probs = ordinary(probs_);
    const at::Tensor* v = ordinary(v_);
    const std::optional<int64_t> heads = plain_int(heads_);
    if (probs == nullptr || v == nullptr || !heads || !ordinary_context() || !ordinary_set({probs, v})) return py::none();
    if (!attention_rows(*v, *heads) || probs->dim() != 4 || probs->size(0) != v->size(0) ||
        probs->size(1) != *heads || probs->size(2) != v->size(1) || probs->size(3) != v->size(1) ||
        !aligned16(*probs) || !aligned16(*v)) {
        return py::none();
    }
    at::Tensor y;
    {
        py::gil_scoped_release no_gil;
        y = attention_pv_causal_hip(*probs, *v, *heads);
    }
    return wrap(y);
}

// ---- the LoRA linear, with its autograd node ------------------------------------

/// The autograd function of cuda_force_amd/autograd.py as a native node: the
/// same saved tensors, kernels and composed path under create_graph, without
/// the interpreter in either direction.
struct LoraLinear : public torch::autograd::Function<LoraLinear> {
    static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& x, const at::Tensor& w,
                              const at::Tensor& a, const at::Tensor& b, double scale) {
        auto [y, xa] = lora_linear_fwd_hip(x, w, a, b, scale);
        ctx->save_for_backward({x, w, a, b, xa});
        ctx->saved_data["scale"] = scale;
        return y;
    }

    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                   torch::autograd::variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const at::Tensor &x = saved[0], &w = saved[1], &a = saved[2], &b = saved[3], &xa = saved[4];
        const double scale = ctx->saved_data["scale"].toDouble();
        const at::Tensor dy = grads[0].contiguous();
        at::Tensor grad_x, grad_w, grad_a, grad_b;
        const bool adapter = ctx->needs_input_grad(2) || ctx->needs_input_grad(3);
        const bool recorded = at::GradMode::is_enabled();
        const bool fused_x = adapter && ctx->needs_input_grad(0) && !recorded;
        // The gradient and what saved-tensor hooks return need not be as plain
        // as the operands were, nor the context as it was in the forward: a
        // batched gradient (is_grads_batched) has no storage, a mode or a
        // profiler may have been entered since. Those calls go through the
        // dispatcher, and so does a recorded one, whose autograd entry refuses
        // to differentiate the adapter gradients.
        const bool direct = !recorded && ordinary_context() && plain_gpu(dy) && plain_gpu(x) && plain_gpu(w) &&
                            plain_gpu(a) && plain_gpu(b) && plain_gpu(xa);
        if (adapter && direct) {
            std::tie(grad_x, grad_a, grad_b) =
                lora_backward_hip(x, dy, fused_x ? &w : nullptr, fused_x ? &a : nullptr, b, xa, scale);
        } else if (fused_x) {
            static const auto op = c10::Dispatcher::singleton()
                                       .findSchemaOrThrow("cudaforge::lora_linear_bwd_input", "")
                                       .typed<std::tuple<at::Tensor, at::Tensor, at::Tensor>(
                                           const at::Tensor&, const at::Tensor&, const at::Tensor&,
                                           const at::Tensor&, const at::Tensor&, const at::Tensor&, double)>();
            std::tie(grad_x, grad_a, grad_b) = op.call(x, dy, w, a, b, xa, scale);
        } else if (adapter) {
            static const auto op = c10::Dispatcher::singleton()
                                       .findSchemaOrThrow("cudaforge::lora_linear_bwd", "")
                                       .typed<std::tuple<at::Tensor, at::Tensor>(
                                           const at::Tensor&, const at::Tensor&, const at::Tensor&,
                                           const at::Tensor&, double)>();
            std::tie(grad_a, grad_b) = op.call(x, dy, b, xa, scale);
        }
        if (ctx->needs_input_grad(0) && !fused_x) {
            grad_x = at::matmul(dy, w.t()) + scale * at::matmul(at::matmul(dy, b.t()), a.t());
        }
        if (ctx->needs_input_grad(1)) grad_w = at::matmul(x.t(), dy);
        return {grad_x, grad_w, grad_a, grad_b, at::Tensor()};
    }
};

py::object try_lora_linear(py::handle x_, py::handle w_, py::handle a_, py::handle b_, py::handle scale_) {
    const at::Tensor* x = ordinary(x_);
    const at::Tensor* w = ordinary(w_);
    const at::Tensor* a = ordinary(a_);
    const at::Tensor* b = ordinary(b_);
    const std::optional<double> scale = plain_double(scale_);
    if (x == nullptr || w == nullptr || a == nullptr || b == nullptr || !scale || !ordinary_context()) {
        return py::none();
    }
    const at::ScalarType dtype = x->scalar_type();
    if (dtype != torch::kFloat32 && dtype != torch::kBFloat16) return py::none();
    for (const at::Tensor* t : {w, a, b}) {
        if (t->scalar_type() != dtype || t->device() != x->device() || t->dim() != 2) return py::none();
    }
    if (x->dim() < 2 || x->size(-1) != w->size(0) || a->size(0) != w->size(0) || b->size(0) != a->size(1) ||
        b->size(1) != w->size(1)) {
        return py::none();
    }
    const bool grad = grad_needed({x, w, a, b});
    at::Tensor y;
    {
        py::gil_scoped_release no_gil;
        const at::Tensor rows = x->dim() == 2 ? *x : x->view({-1, x->size(-1)});
        y = grad ? LoraLinear::apply(rows, *w, *a, *b, *scale) : lora_linear_hip(rows, *w, *a, *b, *scale);
        if (x->dim() != 2) {
            std::vector<int64_t> shape = x->sizes().vec();
            shape.back() = w->size(1);
            y = y.view(shape);
        }
    }
    return wrap(y);
}

}  // namespace
}  // namespace cudaforge_amd

TORCH_LIBRARY(cudaforge, m) {
    // The reference's ten schemas, verbatim (cpp/src/bindings.cpp:342-355).
    m.def("rmsnorm(Tensor input, Tensor weight, float eps) -> Tensor");
    m.def("softmax(Tensor input) -> Tensor");
    m.def("lora_linear(Tensor x, Tensor w, Tensor a, Tensor b, float scale) -> Tensor");
    m.def("sum(Tensor input) -> Tensor");
    m.def("silu(Tensor input) -> Tensor");
    m.def("gelu(Tensor input) -> Tensor");
    m.def("swiglu(Tensor gate, Tensor up) -> Tensor");
    m.def(
        "fused_residual_rmsnorm(Tensor x, Tensor residual, Tensor weight, float eps) "
        "-> Tensor[]");
    m.def("quantize_int8(Tensor input) -> Tensor[]");
    m.def("dequantize_int8(Tensor quantised, Tensor scales) -> Tensor");
    // Extensions used by the Python layer.
    m.def("dequantize_int8_to(Tensor quantised, Tensor scales, ScalarType dtype) -> Tensor");
    m.def("quantize_dequantize(Tensor input) -> Tensor");
    m.def("softmax_as(Tensor input, ScalarType dtype) -> Tensor");
    m.def("softmax_scaled(Tensor input, float scale, int causal_period, ScalarType dtype) -> Tensor");
    m.def("row_sum(Tensor input) -> Tensor");
    m.def(
        "lora_linear_fwd(Tensor x, Tensor w, Tensor a, Tensor b, float scale) "
        "-> (Tensor, Tensor)");
    m.def(
        "lora_linear_bwd(Tensor x, Tensor dy, Tensor b, Tensor xa, float scale) "
        "-> (Tensor, Tensor)");
    m.def(
        "lora_linear_bwd_input(Tensor x, Tensor dy, Tensor w, Tensor a, Tensor b, Tensor xa, float scale) "
        "-> (Tensor, Tensor, Tensor)");
    m.def("attention_scores_causal(Tensor q, Tensor k, int heads) -> Tensor");
    m.def("attention_pv_causal(Tensor probs, Tensor v, int heads) -> Tensor");
}

// Inference-only operators raise on differentiation instead of silently
// producing wrong gradients; the same per-operator registration as the
// reference (bindings.cpp:369-377), extended to the extra operators.
// fused_residual_rmsnorm is left out, as it is there.
TORCH_LIBRARY_IMPL(cudaforge, Autograd, m) {
    for (const char* name :
         {"rmsnorm", "softmax", "lora_linear", "sum", "silu", "gelu", "swiglu", "quantize_int8",
          "dequantize_int8", "dequantize_int8_to", "quantize_dequantize", "softmax_as",
          "softmax_scaled", "row_sum", "lora_linear_fwd", "lora_linear_bwd", "lora_linear_bwd_input",
          "attention_scores_causal", "attention_pv_causal"}) {
        m.impl(name, torch::autograd::autogradNotImplementedFallback());
    }
}

TORCH_LIBRARY_IMPL(cudaforge, CPU, m) {
    using namespace cudaforge_amd;
    m.impl("rmsnorm", &rmsnorm_cpu);
    m.impl("softmax", &softmax_cpu);
    m.impl("lora_linear", &lora_linear_cpu);
    m.impl("sum", &sum_cpu);
    m.impl("silu", &silu_cpu);
    m.impl("gelu", &gelu_cpu);
    m.impl("swiglu", &swiglu_cpu);
    m.impl("fused_residual_rmsnorm", &fused_residual_rmsnorm_cpu);
    m.impl("quantize_int8", &quantize_int8_cpu);
    m.impl("dequantize_int8", &dequantize_int8_cpu);
    m.impl("dequantize_int8_to", &dequantize_int8_to_cpu);
    m.impl("quantize_dequantize", &quantize_dequantize_cpu);
    m.impl("softmax_as", &softmax_as_cpu);
    m.impl("softmax_scaled", &softmax_scaled_cpu);
    m.impl("row_sum", &row_sum_cpu);
    m.impl("lora_linear_fwd", &lora_linear_fwd_cpu);
    m.impl("lora_linear_bwd", &lora_linear_bwd_cpu);
    m.impl("lora_linear_bwd_input", &lora_linear_bwd_input_cpu);
    m.impl("attention_scores_causal", &attention_scores_causal_cpu);
    m.impl("attention_pv_causal", &attention_pv_causal_cpu);
}

TORCH_LIBRARY_IMPL(cudaforge, CUDA, m) {
    using namespace cudaforge_amd;
    m.impl("rmsnorm", &rmsnorm_hip);
    m.impl("softmax", &softmax_hip);
    m.impl("lora_linear", &lora_linear_hip);
    m.impl("sum", &sum_hip);
    m.impl("silu", &silu_hip);
    m.impl("gelu", &gelu_hip);
    m.impl("swiglu", &swiglu_hip);
    m.impl("fused_residual_rmsnorm", &fused_residual_rmsnorm_hip);
    m.impl("quantize_int8", &quantize_int8_hip);
    m.impl("dequantize_int8", &dequantize_int8_hip);
    m.impl("dequantize_int8_to", &dequantize_int8_to_hip);
    m.impl("quantize_dequantize", &quantize_dequantize_hip);
    m.impl("softmax_as", &softmax_as_hip);
    m.impl("softmax_scaled", &softmax_scaled_hip);
    m.impl("row_sum", &row_sum_hip);
    m.impl("lora_linear_fwd", &lora_linear_fwd_hip);
    m.impl("lora_linear_bwd", &lora_linear_bwd_hip);
    m.impl("lora_linear_bwd_input", &lora_linear_bwd_input_hip);
    m.impl("attention_scores_causal", &attention_scores_causal_hip);
    m.impl("attention_pv_causal", &attention_pv_causal_hip);
}

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "cudaforge operators on MI355X (gfx950) HIP kernels";
    m.def("cuda_kernels_available", &cudaforge_amd::cuda_kernels_available,
          "True when the extension was compiled with its HIP kernels");
    // Each returns None when the call is not an ordinary GPU one. The wrapper
    // raises what the dispatcher would (torch.OutOfMemoryError, an exception of
    // a saved-tensor hook as it is).
    m.def("try_rmsnorm", torch::wrap_pybind_function(&cudaforge_amd::try_rmsnorm));
    m.def("try_fused_residual_rmsnorm", torch::wrap_pybind_function(&cudaforge_amd::try_fused_residual_rmsnorm));
    m.def("try_softmax", torch::wrap_pybind_function(&cudaforge_amd::try_softmax));
    m.def("try_softmax_scaled", torch::wrap_pybind_function(&cudaforge_amd::try_softmax_scaled));
    m.def("try_silu", torch::wrap_pybind_function(&cudaforge_amd::try_unary<&cudaforge_amd::silu_hip>));
    m.def("try_gelu", torch::wrap_pybind_function(&cudaforge_amd::try_unary<&cudaforge_amd::gelu_hip>));
    m.def("try_swiglu", torch::wrap_pybind_function(&cudaforge_amd::try_swiglu));
    m.def("try_quantize_int8", torch::wrap_pybind_function(&cudaforge_amd::try_quantize_int8));
    m.def("try_dequantize_int8", torch::wrap_pybind_function(&cudaforge_amd::try_dequantize_int8));
    m.def("try_attention_scores", torch::wrap_pybind_function(&cudaforge_amd::try_attention_scores));
    m.def("try_attention_pv", torch::wrap_pybind_function(&cudaforge_amd::try_attention_pv));
    m.def("try_lora_linear", torch::wrap_pybind_function(&cudaforge_amd::try_lora_linear));
}
