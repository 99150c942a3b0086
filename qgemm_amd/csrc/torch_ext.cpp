// qgemm_python: the torch extension module the reference's packaging names (setup.py:73) and its
// HIP source begins (void fp8_mm(torch::Tensor a, b, as, bs, c), hip_mix_gemm_kernel.cpp:508-516;
// bf16_mm / int8_mm are the commented intent of src/gemm/sm80_gemm_kernel.cu:4-22).  Host code only:
// every function checks its tensors and forwards their data pointers, with torch's current stream, to the
// C ABI of libqgemm.so.
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <optional>
#include <stdexcept>
#include <string>
#include <tuple>

#include "../../include/qgemm.h"

namespace {

void *current_stream() { return (void *)c10::hip::getCurrentHIPStream().stream(); }

void check(int status, const char *what) {
    if (status != QGEMM_OK) throw std::runtime_error(std::string(what) + ": " + qgemm_status_string(status));
}

int dtype_of(const torch::Tensor &t) {
    switch (t.scalar_type()) {
        case torch::kFloat32: return QGEMM_DT_F32;
        case torch::kBFloat16: return QGEMM_DT_BF16;
        case torch::kFloat16: return QGEMM_DT_F16;
        case torch::kInt8: return QGEMM_DT_I8;
        case torch::kInt32: return QGEMM_DT_I32;
        case torch::kFloat8_e4m3fn: return QGEMM_DT_F8E4M3;
        case torch::kUInt8: return QGEMM_DT_F8E4M3;      // raw e4m3 codes
        default: throw std::runtime_error("qgemm_python: unsupported tensor dtype");
    }
}

void need_device(const torch::Tensor &t, const char *name) {
    if (!t.is_cuda()) throw std::runtime_error(std::string("qgemm_python: ") + name + " must be a device tensor");
}

// The kernels decode OCP e4m3 (torch.float8_e4m3fn or raw codes as uint8); the gfx942 "fnuz" encoding has another
// bias and another NaN and is refused.
void need_fp8(const torch::Tensor &t, const char *name) {
    if (t.scalar_type() != torch::kFloat8_e4m3fn && t.scalar_type() != torch::kUInt8)
        throw std::runtime_error(std::string("qgemm_python: ") + name + " must be float8_e4m3fn (OCP e4m3) or uint8 codes");
}

// c is [m, n] with unit inner stride; its row stride becomes ldC
void need_out(const torch::Tensor &c, size_t m, size_t n) {
    if (c.dim() != 2 || (size_t)c.size(0) != m || (size_t)c.size(1) != n || c.stride(1) != 1 || (m > 1 && (size_t)c.stride(0) < n))
        throw std::runtime_error("qgemm_python: c must be [m, n] with unit inner stride");
}

// The reference's contract (hip_mix_gemm_kernel.cpp:425-439): a is [m, k] column-major (storage a[i + j*m]),
// b is [n, k] column-major (storage [k, n] row-major), a_scale [m, k/128] and b_scale [n/128, k/128]
// column-major, c [m, n] row-major bf16; m = a.size(0), n = b.size(0), k = a.size(1).
void fp8_mm(torch::Tensor a, torch::Tensor b, torch::Tensor as, torch::Tensor bs, torch::Tensor c) {
    need_device(a, "a"); need_device(b, "b"); need_device(as, "a_scale"); need_device(bs, "b_scale"); need_device(c, "c");
    const size_t m = a.size(0), n = b.size(0), k = a.size(1);
    need_fp8(a, "a"); need_fp8(b, "b");
    need_out(c, m, n);
    check(qgemm_scaled_gemm(QGEMM_DT_F8E4M3, dtype_of(c), QGEMM_SCALE_BLOCK128, QGEMM_LAYOUT_REFERENCE, a.data_ptr(),
                            b.data_ptr(), as.data_ptr<float>(), bs.data_ptr<float>(), c.data_ptr(), c.stride(0), m, n, k, 0,
                            current_stream()),
          "fp8_mm");
}

// K-contiguous operands (a [m, k], b [n, k] row-major), one fp32 scale each; c fp32 / bf16 / fp16 (or int32 for
// the raw int8 accumulators).
void scaled_mm(torch::Tensor a, torch::Tensor b, torch::Tensor as, torch::Tensor bs, torch::Tensor c, const char *what) {
    need_device(a, "a"); need_device(b, "b"); need_device(as, "a_scale"); need_device(bs, "b_scale"); need_device(c, "c");
    if (!a.is_contiguous() || !b.is_contiguous() || a.size(1) != b.size(1))
        throw std::runtime_error(std::string(what) + ": a [m, k] and b [n, k] must be contiguous with equal k");
    const size_t m = a.size(0), n = b.size(0), k = a.size(1);
    need_out(c, m, n);
    check(qgemm_scaled_gemm(dtype_of(a), dtype_of(c), QGEMM_SCALE_PER_MATRIX, QGEMM_LAYOUT_K_CONTIGUOUS, a.data_ptr(),
                            b.data_ptr(), as.data_ptr<float>(), bs.data_ptr<float>(), c.data_ptr(), c.stride(0), m, n, k, 0,
                            current_stream()),
          what);
}
void int8_mm(torch::Tensor a, torch::Tensor b, torch::Tensor as, torch::Tensor bs, torch::Tensor c) {
    if (a.scalar_type() != torch::kInt8 || b.scalar_type() != torch::kInt8)
        throw std::runtime_error("qgemm_python: int8_mm takes int8 operands");
    scaled_mm(a, b, as, bs, c, "int8_mm");
}
void fp8_mm_per_matrix(torch::Tensor a, torch::Tensor b, torch::Tensor as, torch::Tensor bs, torch::Tensor c) {
    need_fp8(a, "a"); need_fp8(b, "b");
    scaled_mm(a, b, as, bs, c, "fp8_mm_per_matrix");
}

// c [m, n] = a [m, k] x b [n, k]^T, 16-bit operands, fp32 accumulation
void bf16_mm(torch::Tensor a, torch::Tensor b, torch::Tensor c) {
    need_device(a, "a"); need_device(b, "b"); need_device(c, "c");
    if (a.size(1) != b.size(1) || a.stride(1) != 1 || b.stride(1) != 1 || c.stride(1) != 1)
        throw std::runtime_error("bf16_mm: a [m, k] and b [n, k] with unit inner strides");
    need_out(c, a.size(0), b.size(0));
    check(qgemm_gemm(dtype_of(a), dtype_of(c), QGEMM_B_NK, a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), c.data_ptr(),
                     c.stride(0), a.size(0), b.size(0), a.size(1), current_stream()),
          "bf16_mm");
}

// ---- what qgemm_amd/ops.py calls: its functions with the reading of the tensors, the stream lookup and the call into the
// library done here (1 x 2048 x 1024, quantise and multiply: 11.6 + 8.4 us of host time through Python and ctypes, 3 of each
// in torch.cuda.current_stream(), for two kernels of 1.9 and 3.3 us; 4.1 + 3.8 here, most of it the launches).  They answer a status of the library, or kNotPlain, having
// done nothing, for anything that is not the plain case; ops.py then takes its own way, which raises what there is to raise.
constexpr int kNotPlain = -1;

// the library's number of a tensor's type, -1 for none; raw_fp8: uint8 means e4m3 codes
int plain_dtype(const at::Tensor &t, bool raw_fp8) {
    switch (t.scalar_type()) {
        case at::kFloat: return QGEMM_DT_F32;
        case at::kBFloat16: return QGEMM_DT_BF16;
        case at::kHalf: return QGEMM_DT_F16;
        case at::kChar: return QGEMM_DT_I8;
        case at::kInt: return QGEMM_DT_I32;
        case at::kFloat8_e4m3fn: return QGEMM_DT_F8E4M3;
        case at::kByte: return raw_fp8 ? QGEMM_DT_F8E4M3 : -1;
        default: return -1;
    }
}

typedef std::optional<int64_t> opt_int;

int ops_gemm(const at::Tensor &A, const at::Tensor &B, const at::Tensor &C, bool kn, opt_int M, opt_int N, opt_int K,
             opt_int ldA, opt_int ldB, opt_int ldC) {
    if (!A.is_cuda() || !B.is_cuda() || !C.is_cuda() || A.dim() != 2 || B.dim() != 2 || C.dim() < 1) return kNotPlain;
    const int in = plain_dtype(A, true), out = plain_dtype(C, false);
    if (in < 0 || out < 0) return kNotPlain;
    py::gil_scoped_release no_gil;
    return qgemm_gemm(in, out, kn ? QGEMM_B_KN : QGEMM_B_NK, A.data_ptr(), ldA ? *ldA : A.stride(0), B.data_ptr(),
                      ldB ? *ldB : B.stride(0), C.data_ptr(), ldC ? *ldC : C.stride(0), M ? *M : A.size(0),
                      N ? *N : B.size(kn ? 1 : 0), K ? *K : A.size(1), current_stream());
}

int ops_scaled_gemm(const at::Tensor &A, const at::Tensor &B, const std::optional<at::Tensor> &a_scale,
                    const std::optional<at::Tensor> &b_scale, const at::Tensor &C, int64_t M, int64_t N, int64_t K,
                    int scale_mode, int layout, int split_k, std::optional<int> in_dtype, opt_int ldC) {
    if (!A.is_cuda() || !B.is_cuda() || !C.is_cuda() || C.dim() < 1 || (a_scale && !a_scale->is_cuda()) ||
        (b_scale && !b_scale->is_cuda()))
        return kNotPlain;
    const int in = in_dtype ? *in_dtype : plain_dtype(A, true), out = plain_dtype(C, false);
    if (in < 0 || out < 0) return kNotPlain;
    py::gil_scoped_release no_gil;
    return qgemm_scaled_gemm(in, out, scale_mode, layout, A.data_ptr(), B.data_ptr(),
                             a_scale ? (const float *)a_scale->data_ptr() : nullptr,
                             b_scale ? (const float *)b_scale->data_ptr() : nullptr, C.data_ptr(), ldC ? *ldC : C.stride(0), M,
                             N, K, split_k, current_stream());
}

int ops_transpose(const at::Tensor &in, const at::Tensor &out, opt_int M, opt_int N) {
    if (!in.is_cuda() || !out.is_cuda() || (in.dim() < 2 && (!M || !N))) return kNotPlain;
    py::gil_scoped_release no_gil;
    return qgemm_transpose((int)in.element_size(), in.data_ptr(), out.data_ptr(), M ? *M : in.size(0), N ? *N : in.size(1),
                           current_stream());
}

// (status, q, scales)
std::tuple<int, at::Tensor, at::Tensor> ops_quantize(const at::Tensor &x, at::ScalarType out, int mode, bool rows_contiguous_scales) {
    const std::tuple<int, at::Tensor, at::Tensor> not_plain{kNotPlain, at::Tensor(), at::Tensor()};
    if (!x.is_cuda() || x.dim() != 2 || x.stride(1) != 1 || (out != at::kChar && out != at::kFloat8_e4m3fn)) return not_plain;
    const int in = plain_dtype(x, false);
    if (in < 0) return not_plain;
    const int64_t rows = x.size(0), cols = x.size(1);
    at::Tensor q = at::empty({rows, cols}, x.options().dtype(out)), scales;
    const auto f32 = x.options().dtype(at::kFloat);
    int64_t rs = 0, cs = 0;
    if (mode == QGEMM_QUANT_PER_MATRIX) {
        scales = at::empty({1}, f32);
    } else {
        const int64_t nbr = mode == QGEMM_QUANT_BLOCK_1x128 ? rows : (rows + 127) / 128, nbc = (cols + 127) / 128;
        scales = rows_contiguous_scales ? at::empty({nbc, nbr}, f32) : at::empty({nbr, nbc}, f32);
        rs = rows_contiguous_scales ? 1 : nbc;
        cs = rows_contiguous_scales ? nbr : 1;
    }
    py::gil_scoped_release no_gil;
    const int st = qgemm_quantize(in, out == at::kChar ? QGEMM_DT_I8 : QGEMM_DT_F8E4M3, mode, x.data_ptr(),
                                  rows > 1 ? x.stride(0) : std::max<int64_t>(cols, 1), rows, cols, q.data_ptr(), cols,
                                  (float *)scales.data_ptr(), rs, cs, current_stream());
    return {st, q, scales};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "MI355X scaled mixed-precision GEMM (torch-facing entry points over libqgemm.so)";
    m.def("fp8_mm", &fp8_mm, "block-scaled fp8 GEMM, reference layout: fp8_mm(a, b, a_scale, b_scale, c)");
    m.def("fp8_mm_per_matrix", &fp8_mm_per_matrix, "per-matrix scaled fp8 GEMM, K-contiguous operands");
    m.def("int8_mm", &int8_mm, "per-matrix scaled int8 GEMM, K-contiguous operands");
    m.def("bf16_mm", &bf16_mm, "bf16 / fp16 GEMM, b stored [n, k]");
    m.def("ops_gemm", &ops_gemm);
    m.def("ops_scaled_gemm", &ops_scaled_gemm);
    m.def("ops_transpose", &ops_transpose);
    m.def("ops_quantize", &ops_quantize);
}
