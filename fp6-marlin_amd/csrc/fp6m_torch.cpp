// Thin PyTorch-ROCm extension: unwraps tensors, takes the current HIP stream and calls the C ABI of
// include/fp6m.h.  Module functions keep the names and argument order of the reference's two extensions
// (fp6_marlin/fp6_marlin_cuda.cpp:47-58,125-127: `mul`; fp6_marlin/pybind.cpp:89-94: `quantization_cpu`,
// `prepacking_cpu`, `dequantization_cpu`).  Errors surface as the reference's do: RuntimeError from `mul`
// (AT_ERROR), ValueError (std::invalid_argument) from the CPU routines.
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <optional>
#include <stdexcept>
#include <string>

#include "fp6m.h"

namespace {

void check_cpu(int code)
{
    if (code != FP6M_OK) throw std::invalid_argument(fp6m_strerror(code));
}

void mul(const torch::Tensor& A, const torch::Tensor& B, torch::Tensor& C, const torch::Tensor& s,
         torch::Tensor& workspace, int quant_cols, int thread_k, int thread_n, int sms, int max_par, int group_size)
{
    TORCH_CHECK(A.is_cuda() && B.is_cuda() && C.is_cuda() && s.is_cuda() && workspace.is_cuda(),
                "all operands must be tensors on the GPU");
    TORCH_CHECK(A.is_contiguous() && B.is_contiguous() && C.is_contiguous() && s.is_contiguous() &&
                workspace.is_contiguous(), "all operands must be contiguous");
    TORCH_CHECK(A.scalar_type() == torch::kFloat16 && C.scalar_type() == torch::kFloat16 &&
                s.scalar_type() == torch::kFloat16, "A, C and s must be float16");
    TORCH_CHECK(B.element_size() == 4 && workspace.element_size() == 4, "B and workspace must hold 4-byte elements");
    TORCH_CHECK(A.dim() == 2 && C.dim() == 2 && C.size(0) == A.size(0), "A must be [m, k] and C [m, n]");
    const int dev = A.get_device();
    TORCH_CHECK(B.get_device() == dev && C.get_device() == dev && s.get_device() == dev && workspace.get_device() == dev,
                "all operands must live on the same device");
    const int prob_m = A.size(0), prob_n = C.size(1), prob_k = A.size(1);
    TORCH_CHECK(workspace.numel() >= prob_n / 128 * max_par, "workspace must be of size at least ",
                prob_n / 128 * max_par, ".");
    const int64_t qc = quant_cols <= 0 ? 0 : quant_cols, n4 = prob_n - qc;
    if (prob_k % 32 == 0 && qc <= prob_n) {
        const int64_t need_b = (int64_t)prob_k * n4 / 8 + (int64_t)prob_k * qc * 3 / 16;
        const int64_t need_s = (group_size == -1 ? n4 : (int64_t)(prob_k / 128) * n4) + qc;
        TORCH_CHECK(B.numel() >= need_b && s.numel() == need_s, "B must hold ", need_b, " words and s ", need_s,
                    " scales for this problem");
    }
    hipStream_t stream = c10::hip::getCurrentHIPStream(dev).stream();
    const int err = fp6m_mul(A.data_ptr(), B.data_ptr(), C.data_ptr(), s.data_ptr(), prob_m, prob_n, prob_k,
                             workspace.data_ptr(), dev, stream, thread_k, thread_n, sms, max_par, quant_cols, group_size);
    if (err == FP6M_ERR_PROB_SHAPE) {
        AT_ERROR("Problem (m=", prob_m, ", n=", prob_n, ", k=", prob_k, ")", " not compatible with thread_k=",
                 thread_k, ", thread_n=", thread_n, ".");
    } else if (err == FP6M_ERR_KERN_SHAPE) {
        AT_ERROR("No kernel implementation for thread_k=", thread_k, ", thread_n=", thread_n, ".");
    } else if (err != FP6M_OK) {
        AT_ERROR("fp6m_mul: ", fp6m_strerror(err), " (hip error ", fp6m_last_hip_error(), ")");
    }
}

using MaybeTensor = std::optional<torch::Tensor>;

const void* ptr(const MaybeTensor& t) { return t ? t->data_ptr() : nullptr; }

// fp6m_mul_fused (quant_rows == 0) or fp6m_mul_rows.  The checks are those of cabi._mul_extended.
void mul_extended(const torch::Tensor& A, const torch::Tensor& B, torch::Tensor& C, const torch::Tensor& s,
                  torch::Tensor& workspace, int quant_cols, int group_size, int quant_rows, const MaybeTensor& a_cols,
                  const MaybeTensor& c_cols, const MaybeTensor& bias, const MaybeTensor& residual, int sms, int max_par, bool gfx950)
{
    const auto check = [&](const char* name, const torch::Tensor& t) {
        TORCH_CHECK(t.is_cuda(), name, " must be a tensor on the GPU");
        TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
        TORCH_CHECK(t.get_device() == A.get_device(), "all operands must live on the same device");
    };
    check("A", A);
    check("B", B);
    check("C", C);
    check("s", s);
    check("workspace", workspace);
    if (a_cols) check("a_cols", *a_cols);
    if (c_cols) check("c_cols", *c_cols);
    if (bias) check("bias", *bias);
    if (residual) check("residual", *residual);
    TORCH_CHECK(A.scalar_type() == torch::kFloat16 && C.scalar_type() == torch::kFloat16 &&
                s.scalar_type() == torch::kFloat16, "A, C and s must be float16");
    TORCH_CHECK(B.element_size() == 4 && workspace.element_size() == 4,
                "B must be int32 (or another 4-byte type) and workspace a 4-byte type");
    TORCH_CHECK(A.dim() == 2 && C.dim() == 2 && C.size(0) == A.size(0), "A must be [m, lda] and C [m, n]");
    const int64_t m = A.size(0), lda = A.size(1), n = C.size(1), k = a_cols ? a_cols->numel() : lda;
    TORCH_CHECK(!a_cols || a_cols->scalar_type() == torch::kInt32, "a_cols must be int32 with ", k, " entries");
    TORCH_CHECK(!c_cols || (c_cols->scalar_type() == torch::kInt32 && c_cols->numel() == n), "c_cols must be int32 with ", n, " entries");
    TORCH_CHECK(!bias || (bias->scalar_type() == torch::kFloat16 && bias->numel() == n), "bias must be float16 with ", n, " entries");
    TORCH_CHECK(!residual || (residual->scalar_type() == torch::kFloat16 && residual->dim() == 2 && residual->size(0) == m &&
                              residual->size(1) == n), "residual must be float16 [m, n]");
    TORCH_CHECK(workspace.numel() >= n / 128 * max_par, "workspace must be of size at least ", n / 128 * max_par, ".");
    const auto sized = [&](int64_t need_b, int64_t need_s) {
        TORCH_CHECK(B.numel() >= need_b && s.numel() == need_s, "B must hold ", need_b, " words and s ", need_s, " scales for this problem");
    };
    if (quant_rows) {
        const int64_t k4 = k - quant_rows;
        TORCH_CHECK(quant_rows > 0 && k4 > 0, "quant_rows must be positive and below k");
        if (k4 % 128 == 0 && quant_rows % 64 == 0) sized(k4 * n / 8 + quant_rows * n * 3 / 16, k4 / 128 * n + n);
    } else {
        const int64_t qc = quant_cols == -1 || quant_cols == 0 ? 0 : quant_cols, n4 = n - qc;
        if (k % 32 == 0 && qc >= 0 && qc <= n) sized(k * n4 / 8 + k * qc * 3 / 16, (group_size == -1 ? n4 : k / 128 * n4) + qc);
    }
    const int dev = A.get_device(), flags = gfx950 ? FP6M_LAYOUT_GFX950 : 0;
    const c10::DeviceGuard guard(A.device());
    hipStream_t stream = c10::hip::getCurrentHIPStream(dev).stream();
    const int32_t *ac = static_cast<const int32_t*>(ptr(a_cols)), *cc = static_cast<const int32_t*>(ptr(c_cols));
    const int err = quant_rows
        ? fp6m_mul_rows(A.data_ptr(), lda, B.data_ptr(), C.data_ptr(), s.data_ptr(), m, n, k, workspace.data_ptr(), dev, stream, sms,
                        max_par, quant_rows, ac, cc, ptr(bias), ptr(residual), flags)
        : fp6m_mul_fused(A.data_ptr(), lda, B.data_ptr(), C.data_ptr(), s.data_ptr(), m, n, k, workspace.data_ptr(), dev, stream, sms,
                         max_par, quant_cols, group_size, ac, cc, ptr(bias), ptr(residual), flags);
    TORCH_CHECK(err != FP6M_ERR_PROB_SHAPE, "Problem (m=", m, ", n=", n, ", k=", k, ") not compatible with the tile shape.");
    TORCH_CHECK(err == FP6M_OK, quant_rows ? "fp6m_mul_rows: " : "fp6m_mul_fused: ", fp6m_strerror(err), " (hip error ",
                fp6m_last_hip_error(), ")");
}

// Layer.forward between its buffers and its result: what a call does to x and the residual before the GEMM and to the
// result after it, in one place, because in Python those steps and the checks took longer than the GEMM of a small batch
// (11008 x 4096 at 8 rows: 24 us on the host for 12 us on the GPU).
torch::Tensor layer_forward(const torch::Tensor& x, const MaybeTensor& residual, const torch::Tensor& B, const torch::Tensor& s,
                            torch::Tensor& workspace, int64_t n, int quant_cols, int group_size, int quant_rows,
                            const MaybeTensor& a_cols, const MaybeTensor& c_cols, const MaybeTensor& bias, bool gfx950)
{
    const bool flat = x.dim() == 2;
    const auto x2 = (flat ? x : x.reshape({-1, x.size(-1)})).to(torch::kFloat16).contiguous();
    MaybeTensor res;
    if (residual) res = residual->reshape({-1, n}).to(torch::kFloat16).contiguous();
    auto out = at::empty({x2.size(0), n}, x2.options());
    if (!quant_rows && !c_cols && !bias && !res && !gfx950)
        mul(x2, B, out, s, workspace, quant_cols, -1, -1, -1, 16, group_size);
    else
        mul_extended(x2, B, out, s, workspace, quant_cols, quant_rows ? 128 : group_size, quant_rows, a_cols, c_cols, bias, res, -1, 16, gfx950);
    if (flat) return out;
    auto shape = x.sizes().vec();
    shape.back() = n;
    return out.reshape(shape);
}

torch::Tensor quantization_cpu(torch::Tensor w)
{
    if (w.scalar_type() != torch::kFloat16) throw std::invalid_argument("Input tensor should be of type float16.");
    if (w.is_cuda() || w.dim() != 2 || w.size(0) % 256 || w.size(1) % 256)
        throw std::invalid_argument("quantize expects a 2-D CPU tensor with both dimensions multiples of 256");
    w = w.contiguous();
    const int64_t oc = w.size(0), ic = w.size(1);
    auto out = torch::empty({ic, oc / 16 * 3}, torch::kInt32);
    // the flat buffer is read as ic rows of oc values, like the reference (pybind.cpp:52-57)
    check_cpu(fp6m_fp6_quantize(reinterpret_cast<const uint16_t*>(w.data_ptr()),
                                reinterpret_cast<uint8_t*>(out.data_ptr()), (size_t)ic, (size_t)oc));
    return out;
}

torch::Tensor prepacking_cpu(torch::Tensor q)
{
    if (q.scalar_type() != torch::kInt32 || q.is_cuda() || q.dim() != 2 || q.size(1) % 3)
        throw std::invalid_argument("prepacking expects a CPU int32 tensor [OC, IC*3/16]");
    q = q.contiguous();
    const int64_t oc = q.size(0), ic = q.size(1) * 16 / 3;
    if (oc % 256 || ic % 256) throw std::invalid_argument("prepacking expects OC and IC to be multiples of 256");
    auto out = torch::empty({ic / 32 * 3, oc * 2}, torch::kInt32);
    check_cpu(fp6m_fp6_prepack(out.data_ptr<int32_t>(), q.data_ptr<int32_t>(), (size_t)oc, (size_t)ic));
    return out;
}

torch::Tensor dequantization_cpu(torch::Tensor q, torch::Tensor scale)
{
    if (q.scalar_type() != torch::kInt32 || scale.scalar_type() != torch::kFloat16 || q.is_cuda() || scale.is_cuda() ||
        q.dim() != 2 || q.size(1) % 3 || scale.numel() != q.size(0))
        throw std::invalid_argument("dequantize expects CPU int32 [OC, IC*3/16] and float16 [OC]");
    q = q.contiguous();
    scale = scale.contiguous();
    const int64_t oc = q.size(0), ic = q.size(1) / 3 * 16;
    auto out = torch::empty({oc, ic}, torch::kFloat16);
    check_cpu(fp6m_fp6_dequant(reinterpret_cast<uint16_t*>(out.data_ptr()), reinterpret_cast<const uint8_t*>(q.data_ptr()),
                               (size_t)oc, (size_t)ic, reinterpret_cast<const uint16_t*>(scale.data_ptr())));
    return out;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    namespace py = pybind11;
    m.def("mul", &mul, "mixed INT4/FP6 x FP16 GEMM (gfx950)", py::arg("A"), py::arg("B"), py::arg("C"), py::arg("s"),
          py::arg("workspace"), py::arg("quant_cols") = -1, py::arg("thread_k") = -1, py::arg("thread_n") = -1,
          py::arg("sms") = -1, py::arg("max_par") = 8, py::arg("group_size") = -1);
    // (without the interpreter's lock: a launch may block, and another Python thread may be driving another stream)
    m.def("mul_extended", &mul_extended, "the GEMM with gather, scatter, bias and residual; column or row mix (gfx950)",
          py::call_guard<py::gil_scoped_release>());
    m.def("layer_forward", &layer_forward, "one quantised linear layer (gfx950)", py::call_guard<py::gil_scoped_release>());
    m.def("quantization_cpu", &quantization_cpu, "Weight quantization (CPU)");
    m.def("prepacking_cpu", &prepacking_cpu, "Weight prepacking (CPU)");
    m.def("dequantization_cpu", &dequantization_cpu, "Weight dequantization (CPU)");
}
