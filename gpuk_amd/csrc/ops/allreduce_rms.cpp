// allreduce_rms for one GPU: the residual-add + RMSNorm + FP8 epilogue without the all-reduce.
// Mirrors the host op at src/ops/all_reduce_fusion.cpp:363-396 (same argument order and checks);
// the IPC workspace behind a non-zero `fptr` belongs to the multi-GPU path and is not built here.
#include <atomic>

#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPException.h>

#include "ops.h"

namespace gpuk_ops {

namespace {
// amax divisor / clamp bound of the fp8 modes.  448 = OCP e4m3fn (gfx950 hardware); 240 reproduces
// the reference's fp8e4m3fn::max_value (src/common/float8.h:216-218, gpuk/__init__.py:42-46).
// One value for the whole process: it changes the numerics of every later allreduce_rms call from any thread (the
// store itself is atomic).  Set it once at start-up, not around individual calls.
std::atomic<double> g_fp8_max{448.0};
}  // namespace

bool current_stream_is_capturing() {
    hipStreamCaptureStatus status{};
    C10_HIP_CHECK(hipStreamIsCapturing(static_cast<hipStream_t>(current_stream()), &status));
    return status != hipStreamCaptureStatusNone;
}

void set_fp8_max(double value) {
    TORCH_CHECK(value > 0.0 && value <= 448.0, "set_fp8_max: value must be in (0, 448], got ", value);
    g_fp8_max.store(value);
}

double get_fp8_max() { return g_fp8_max.load(); }

namespace {
void add_rms(const Tensor &allreduce_in, const Tensor &residual_in, const Tensor &rms_gamma, const Tensor &residual_out,
             const Tensor &norm_out, const Tensor &scale_out, double eps, int64_t quant_type) {
    TORCH_CHECK(allreduce_in.is_contiguous() && residual_in.is_contiguous() && rms_gamma.is_contiguous());
    TORCH_CHECK(residual_out.is_contiguous() && norm_out.is_contiguous() && scale_out.is_contiguous());
    TORCH_CHECK(allreduce_in.dim() >= 1, "allreduce_rms: allreduce_in needs a hidden dimension");
    const int64_t hidden = allreduce_in.size(-1);
    const int64_t size = allreduce_in.numel();
    const int64_t tokens = hidden > 0 ? size / hidden : 0;
    TORCH_CHECK(hidden > 0 && hidden % 8 == 0, "allreduce_rms: hidden must be a positive multiple of 8, got ", hidden);
    TORCH_CHECK(residual_in.numel() == size && residual_out.numel() == size && norm_out.numel() == size,
                "allreduce_rms: residual_in, residual_out and norm_out must have allreduce_in's element count");
    TORCH_CHECK(rms_gamma.numel() == hidden, "allreduce_rms: rms_gamma must have `hidden` elements");
    const auto act = allreduce_in.scalar_type();
    TORCH_CHECK(residual_in.scalar_type() == act && rms_gamma.scalar_type() == act && residual_out.scalar_type() == act,
                "allreduce_rms: residual_in, rms_gamma and residual_out must share allreduce_in's dtype");
    const int dtype = activation_dtype(allreduce_in, "allreduce_rms");
    TORCH_CHECK(quant_type != GPUK_QUANT_FP8_E4M3FNUZ,
                "allreduce_rms: quant_type 2 (e4m3fnuz) is the MI300 encoding; gfx950 encodes OCP e4m3fn (quant_type 1)");
    TORCH_CHECK(quant_type == GPUK_QUANT_NONE || quant_type == GPUK_QUANT_FP8_DYNAMIC || quant_type == GPUK_QUANT_FP8_STATIC,
                "allreduce_rms: unknown quant_type ", quant_type);
    float *scale_ptr = nullptr;
    if (quant_type == GPUK_QUANT_NONE) {
        TORCH_CHECK(norm_out.scalar_type() == act, "allreduce_rms: norm_out must have the activation dtype when quant_type is 0");
    } else {
        TORCH_CHECK(norm_out.element_size() == 1, "allreduce_rms: norm_out must be a 1-byte fp8 tensor when quant_type is ", quant_type);
        TORCH_CHECK(scale_out.scalar_type() == at::kFloat, "allreduce_rms: scale_out must be float32");
        TORCH_CHECK(scale_out.numel() >= (quant_type == GPUK_QUANT_FP8_DYNAMIC ? tokens : 1),
                    "allreduce_rms: scale_out is too small");
        scale_ptr = scale_out.data_ptr<float>();
    }
    TORCH_CHECK(allreduce_in.is_cuda(), "allreduce_rms: tensors must live on the GPU");
    const auto dev = allreduce_in.device();
    TORCH_CHECK(residual_in.device() == dev && rms_gamma.device() == dev && residual_out.device() == dev &&
                    norm_out.device() == dev && (quant_type == GPUK_QUANT_NONE || scale_out.device() == dev),
                "allreduce_rms: all tensors must be on the same device");
    DeviceGuard guard(dev);
    const int status = gpuk_add_rmsnorm_quant(allreduce_in.data_ptr(), residual_in.data_ptr(), rms_gamma.data_ptr(),
                                              residual_out.data_ptr(), norm_out.data_ptr(), scale_ptr, tokens, hidden,
                                              (float)eps, dtype, (int)quant_type, (float)g_fp8_max.load(),
                                              current_stream());
    check_status(status, "allreduce_rms");
}
}  // namespace

void allreduce_rms(int64_t fptr, Tensor &allreduce_in, Tensor &residual_in, Tensor &rms_gamma, Tensor &residual_out,
                   Tensor &norm_out, Tensor &scale_out, double eps, int64_t quant_type) {
    TORCH_CHECK(fptr == 0,
                "allreduce_rms: this build is the single-GPU share of the op; pass fptr=0 (no all-reduce workspace)");
    add_rms(allreduce_in, residual_in, rms_gamma, residual_out, norm_out, scale_out, eps, quant_type);
}

namespace {
Tensor empty_like_as(const Tensor &t, at::ScalarType dtype) {  // t is contiguous; its strides are kept, as empty_like keeps them
    return at::detail::empty_strided_cuda(t.sizes(), t.strides(), dtype, t.device());
}
void check_inputs(const Tensor &allreduce_in, const Tensor &residual_in) {
    TORCH_CHECK(allreduce_in.is_cuda() && residual_in.is_cuda(), "allreduce_rms: tensors must live on the GPU");
    TORCH_CHECK(allreduce_in.is_contiguous() && residual_in.is_contiguous());
}
// The scale is an output of this overload: the static mode would quantise by memory nobody wrote.
void check_functional_quant_type(int64_t quant_type) {
    TORCH_CHECK(quant_type == GPUK_QUANT_NONE || quant_type == GPUK_QUANT_FP8_DYNAMIC,
                "add_rms_fused: quant_type must be 0 (none) or 1 (fp8, dynamic scale), got ", quant_type,
                "; a static scale is passed to add_rms_fused.static");
}
// The scale is read by the kernel as it is: a copy or cast made here would be a hidden transfer inside the call, which a
// stream capture rejects.
void check_static_scale(const Tensor &static_scale, const Tensor &allreduce_in) {
    TORCH_CHECK_VALUE(static_scale.device() == allreduce_in.device() && static_scale.scalar_type() == at::kFloat && static_scale.numel() == 1,
                      "static_scale must be a 1-element fp32 tensor on the device of the activations");
}
}  // namespace

// Outputs allocated here, behind one pass through the dispatcher: allocated from Python, one call each, the three cost
// a decode step more than its kernel takes (9.5 us per call of one 7168-element row, 7.3 in this form, each called through
// torch.ops; the kernel 3.3).
std::tuple<Tensor, Tensor, Tensor> add_rms_fused(const Tensor &allreduce_in, const Tensor &residual_in, const Tensor &rms_gamma,
                                                 double eps, int64_t quant_type) {
    check_functional_quant_type(quant_type);
    check_inputs(allreduce_in, residual_in);
    const bool fp8 = quant_type != GPUK_QUANT_NONE;
    const Tensor &x = allreduce_in;
    Tensor residual_out = empty_like_as(residual_in, residual_in.scalar_type());
    Tensor norm_out = empty_like_as(x, fp8 ? at::kFloat8_e4m3fn : x.scalar_type());
    Tensor scale_out = fp8 ? at::detail::empty_cuda({x.size(0), 1}, at::kFloat, x.device(), std::nullopt)
                           : at::detail::empty_cuda({1}, at::kFloat, x.device(), std::nullopt);
    add_rms(x, residual_in, rms_gamma, residual_out, norm_out, scale_out, eps, quant_type);
    return {std::move(residual_out), std::move(norm_out), std::move(scale_out)};
}

std::tuple<Tensor, Tensor> add_rms_fused_static(const Tensor &allreduce_in, const Tensor &residual_in, const Tensor &rms_gamma,
                                                double eps, const Tensor &static_scale) {
    check_static_scale(static_scale, allreduce_in);
    check_inputs(allreduce_in, residual_in);
    Tensor residual_out = empty_like_as(residual_in, residual_in.scalar_type());
    Tensor norm_out = empty_like_as(allreduce_in, at::kFloat8_e4m3fn);
    add_rms(allreduce_in, residual_in, rms_gamma, residual_out, norm_out, static_scale, eps, GPUK_QUANT_FP8_STATIC);
    return {std::move(residual_out), std::move(norm_out)};
}

std::tuple<Tensor, Tensor, Tensor> add_rms_fused_meta(const Tensor &allreduce_in, const Tensor &residual_in,
                                                      const Tensor &rms_gamma, double eps, int64_t quant_type) {
    check_functional_quant_type(quant_type);
    const bool fp8 = quant_type != GPUK_QUANT_NONE;
    const auto f32 = allreduce_in.options().dtype(at::kFloat);
    return {at::empty_like(residual_in), at::empty_like(allreduce_in, fp8 ? allreduce_in.options().dtype(at::kFloat8_e4m3fn) : allreduce_in.options()),
            fp8 ? at::empty_symint({allreduce_in.sym_size(0), 1}, f32) : at::empty({1}, f32)};
}

std::tuple<Tensor, Tensor> add_rms_fused_static_meta(const Tensor &allreduce_in, const Tensor &residual_in,
                                                     const Tensor &rms_gamma, double eps, const Tensor &static_scale) {
    check_static_scale(static_scale, allreduce_in);
    return {at::empty_like(residual_in), at::empty_like(allreduce_in, allreduce_in.options().dtype(at::kFloat8_e4m3fn))};
}

}  // namespace gpuk_ops
