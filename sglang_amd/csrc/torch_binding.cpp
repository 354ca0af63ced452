// PyTorch-ROCm binding of the C ABI: the operators torch.ops.sgl_kernel.* (CUDA dispatch key, which is the HIP device) and
// the calls of the Python layer, as one extension module, sglang_amd._native.
//
// At decode sizes a linear layer is 5-15 us of kernels, and the host has to enqueue it faster than that.  Done in Python
// through ctypes - some twenty checks, two allocations, one foreign call - it took 13-17 us a call and left the GPU waiting;
// here the checks read the tensors directly, outputs and workspaces come from the same caching allocator (a workspace
// without a tensor around it), and a call of the Python-level wrapper takes about 4 us.
//
// Two layers:
//   * the operators: argument checks with the conditions and wording of the reference's host functions (cited at each),
//     allocation, one C-ABI call.  They throw; the GIL is not held while they run.
//   * the linear methods' fast paths (try_*): whole forward passes of fp8_utils / w8a8_int8 for the operands those meet in
//     use.  They return None for anything else, and where a mode, a tracer or a functional transform listens at the dispatcher;
//     the Python function then goes its long way, which calls the operators and raises the errors.
#include <Python.h>

#include <ATen/Context.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/ops/empty.h>
#include <ATen/record_function.h>
#include <c10/core/Allocator.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/library.h>

#include <strings.h>

#include <atomic>
#include <cmath>
#include <cstdlib>
#include <optional>

#include "mi355_qlinear.h"

namespace {

using at::Tensor;
using c10::ScalarType;
using OptTensor = std::optional<Tensor>;

constexpr auto FP8 = ScalarType::Float8_e4m3fn;

PyObject* g_error_class = nullptr;  // sglang_amd._lib.Mi355Error, set by the Python layer

// ---- pieces every call shares

void check(int status) {
  if (status == MI355_OK) return;
  const std::string msg = mi355_last_error();
  if (status == MI355_ERR_UNSUPPORTED) C10_THROW_ERROR(NotImplementedError, msg);
  PyGILState_STATE gil = PyGILState_Ensure();
  PyErr_SetString(g_error_class != nullptr ? g_error_class : PyExc_RuntimeError, msg.c_str());
  python_error err;
  err.persist();
  PyGILState_Release(gil);
  throw err;
}

int dtype_code(ScalarType t) {
  switch (t) {
    case ScalarType::Float: return MI355_F32;
    case ScalarType::Half: return MI355_F16;
    case ScalarType::BFloat16: return MI355_BF16;
    case ScalarType::Float8_e4m3fn: return MI355_FP8_E4M3FN;
    case ScalarType::Char: return MI355_I8;
    case ScalarType::Int: return MI355_I32;
    default: return -1;
  }
}
bool is_16bit(ScalarType t) { return t == ScalarType::Half || t == ScalarType::BFloat16; }
bool is_float(ScalarType t) { return is_16bit(t) || t == ScalarType::Float; }

constexpr int MAX_DEVICES = 64;
std::atomic<bool> g_device_ready[MAX_DEVICES];

// The current HIP stream; on a device's first use, the library's per-device set-up, which must not fall inside a graph
// capture (inside one it is left alone: the two entry points that need it say so in their error).
void* current_stream() {
  const c10::hip::HIPStream s = c10::hip::getCurrentHIPStream();
  const int dev = s.device_index();
  if (dev >= 0 && dev < MAX_DEVICES && !g_device_ready[dev].load(std::memory_order_acquire)) {
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s.stream(), &capturing) == hipSuccess && capturing == hipStreamCaptureStatusNone) {
      check(mi355_qlinear_init());
      g_device_ready[dev].store(true, std::memory_order_release);
    }
  }
  return s.stream();
}

Tensor new_tensor(at::IntArrayRef sizes, ScalarType dtype, const Tensor& like) {
  return at::empty(sizes, like.options().dtype(dtype).layout(at::kStrided).requires_grad(false).memory_format(std::nullopt));
}

// The same for a fast path, which nobody listens to: the device's own allocation that at::empty's kernel makes, without the dispatcher in front of it, half
// of the 0.7 us that a tensor takes (one launch is about 3).  That kernel then fills the memory where deterministic algorithms are asked for (what no
// kernel writes, the pitch of aligned scales, would differ from run to run), and a profiler that records operators gets to see at::empty: both go there.
Tensor new_plain_tensor(at::IntArrayRef sizes, ScalarType dtype, const Tensor& like) {
  const at::Context& context = at::globalContext();
  if (at::getStepCallbacksUnlessEmpty(at::RecordScope::FUNCTION).has_value() || (context.deterministicAlgorithms() && context.deterministicFillUninitializedMemory()))
    return new_tensor(sizes, dtype, like);
  return Tensor(at::detail::empty_cuda(sizes, dtype, like.device(), std::nullopt));
}

// New memory of `sizes`, contiguous, seen with other sizes and strides: the tensor that nobody else holds yet is given them itself.  (A view made
// by the dispatcher, as_strided, takes 0.3 us longer, of the 6 of a small quantizer's call.)
Tensor new_tensor_as(at::IntArrayRef sizes, ScalarType dtype, const Tensor& like, at::IntArrayRef seen, at::IntArrayRef strides) {
  Tensor t = new_plain_tensor(sizes, dtype, like);
  t.unsafeGetTensorImpl()->set_sizes_and_strides(seen, strides);
  return t;
}

// Device memory for the length of one call, stream-ordered like a tensor's but without the tensor.
struct Workspace {
  c10::DataPtr mem;
  size_t bytes;
  explicit Workspace(size_t n) : bytes(n) {
    if (n > 0) mem = c10::GetAllocator(c10::DeviceType::CUDA)->allocate(n);
  }
  void* ptr() const { return mem.get(); }
};

const void* data_or_null(const OptTensor& t) { return t.has_value() && t->defined() ? t->const_data_ptr() : nullptr; }
bool given(const OptTensor& t) { return t.has_value() && t->defined(); }

void check_input(const Tensor& t, const char* name) {  // CHECK_INPUT of sgl-kernel/include/utils.h:193-212
  TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

// The operand checks the GEMM operators of the reference share; returns nothing, throws with their wording.
void check_mm_operands(const Tensor& a, const Tensor& b) {
  TORCH_CHECK(a.is_cuda(), "mat_a must be a CUDA tensor");
  TORCH_CHECK(b.is_cuda(), "mat_b must be a CUDA tensor");
  TORCH_CHECK(a.dim() == 2, "mat_a must be a 2D tensor");
  TORCH_CHECK(b.dim() == 2, "mat_b must be a 2D tensor");
  TORCH_CHECK(a.stride(1) == 1, "mat_a must be a row major tensor");
  TORCH_CHECK(b.stride(0) == 1, "mat_b must be a column major tensor");
  TORCH_CHECK(a.size(1) == b.size(0), "mat_a and mat_b shapes cannot be multiplied");
}
void check_channel_scales(const Tensor& sa, const Tensor& sb, const OptTensor& bias, int64_t M, int64_t N, ScalarType out_dtype) {
  TORCH_CHECK(sa.numel() == M, "size of scales_a is not matched");
  TORCH_CHECK(sb.numel() == N, "size of scales_b is not matched");
  TORCH_CHECK(sa.is_contiguous(), "scales_a must be contiguous");
  TORCH_CHECK(sb.is_contiguous(), "scales_b msut be contiguous");
  TORCH_CHECK(sa.scalar_type() == ScalarType::Float, "scales_a must be Float32");
  TORCH_CHECK(sb.scalar_type() == ScalarType::Float, "scales_b must be Float32");
  if (given(bias)) {
    TORCH_CHECK(bias->numel() == N, "size of bias is not matched");
    TORCH_CHECK(bias->is_contiguous(), "bias must be contiguous");
    TORCH_CHECK(bias->scalar_type() == out_dtype, "bias dtype must match output dtype");
  }
}

// ---------------------------------------------------------------- quantizers

void launch_group_quant(const Tensor& x, const Tensor& q, const Tensor& s, int64_t M, int64_t K, int64_t group, double eps, double qmin,
                        double qmax, int mode, int kind, double pow2_floor, int64_t s_row, int64_t s_col) {
  check(mi355_group_quant_8bit(x.const_data_ptr(), dtype_code(x.scalar_type()), q.data_ptr(), dtype_code(q.scalar_type()), s.data_ptr(),
                               M, K, (int)group, (float)eps, (float)qmin, (float)qmax, mode, kind, (float)pow2_floor, s_row, s_col,
                               current_stream()));
}

void group_quant(const Tensor& input, const Tensor& output_q, const Tensor& output_s, int64_t group, double eps, double qmin, double qmax,
                 bool scale_ue8m0, int mode, double pow2_floor, const char* op) {
  check_input(input, "input");
  check_input(output_q, "output_q");
  TORCH_CHECK(group > 0 && input.numel() % group == 0, "CHECK_EQ(input.numel() % group_size, 0) failed in ", op);
  TORCH_CHECK(output_s.dim() == 2, "CHECK_EQ(output_s.dim(), 2) failed in ", op);
  TORCH_CHECK(is_float(input.scalar_type()), op, ": unsupported input dtype ", input.scalar_type());
  TORCH_CHECK(output_q.scalar_type() == FP8 || output_q.scalar_type() == ScalarType::Char, op, ": unsupported output dtype ",
              output_q.scalar_type());
  TORCH_CHECK(output_q.numel() == input.numel(), op, ": output_q must have as many elements as input");
  if (input.numel() == 0) return;
  const int64_t K = input.size(-1), M = input.numel() / K;
  TORCH_CHECK(K % group == 0, op, ": the last dimension must be divisible by group_size");
  if (group == K && mode == MI355_QUANT_DIV && !scale_ue8m0 && output_q.scalar_type() == FP8 &&
      (group * (int64_t)input.element_size() > 2048 || (group & (group - 1))) && output_s.scalar_type() == ScalarType::Float &&
      qmin == -448.0 && qmax == 448.0) {
    // the whole row is one group (a weight quantized per output channel at load time): rows longer than the group kernel's
    // 2048 bytes, or not a power of two
    TORCH_CHECK(output_s.numel() == M && output_s.is_contiguous(), op, ": output_s must hold one contiguous scale per row");
    check(mi355_row_group_quant_fp8(input.const_data_ptr(), dtype_code(input.scalar_type()), output_q.data_ptr(),
                                    static_cast<float*>(output_s.data_ptr()), M, K, (float)eps, MI355_QUANT_DIV, current_stream()));
    return;
  }
  // same test as per_token_group_quant_8bit.cu:153 / per_token_group_quant_8bit_v2.cu:426
  const bool column_major = output_s.stride(0) < output_s.stride(1);
  int kind = MI355_SCALE_F32;
  int64_t s_row = 1, s_col = output_s.stride(1);
  if (scale_ue8m0) {
    TORCH_CHECK(column_major, op, ": scale_ue8m0 needs column-major scales");
    TORCH_CHECK(output_s.scalar_type() == ScalarType::Int, op, ": packed UE8M0 scales are stored in an int32 tensor");
    kind = MI355_SCALE_UE8M0_PACKED;
  } else {
    TORCH_CHECK(output_s.scalar_type() == ScalarType::Float, op, ": output_s must be float32");
    // row-major scales are addressed by the flat group index, as in the reference kernels
    if (!column_major) s_row = K / group, s_col = 1;
  }
  launch_group_quant(input, output_q, output_s, M, K, group, eps, qmin, qmax, mode, kind, pow2_floor, s_row, s_col);
}

// sgl-kernel/csrc/gemm/per_token_group_quant_8bit.cu:116-217: q = x / (amax / max)
void per_token_group_quant_8bit(const Tensor& input, const Tensor& output_q, const Tensor& output_s, int64_t group, double eps, double qmin,
                                double qmax, bool scale_ue8m0) {
  group_quant(input, output_q, output_s, group, eps, qmin, qmax, scale_ue8m0, MI355_QUANT_DIV, 1e-10, "sgl_per_token_group_quant_8bit");
}

// The fuse_silu_and_mul branch of per_token_group_quant_8bit_v2.cu:394-514: input [T, 2H] or, with masked_m, [E, T, 2H]; the
// reference instantiates it for column-major packed UE8M0 scales only (:455-470).
void silu_mul_group_quant(const Tensor& input, const Tensor& output_q, const Tensor& output_s, int64_t group, double eps, double qmin,
                          double qmax, bool scale_ue8m0, const OptTensor& masked_m, const char* op) {
  if (!(scale_ue8m0 && output_s.scalar_type() == ScalarType::Int && output_s.dim() >= 2 && output_s.stride(-2) == 1 && group == 128 &&
        output_q.scalar_type() == FP8))
    C10_THROW_ERROR(NotImplementedError, std::string(op) + ": fuse_silu_and_mul is built for group 128, e4m3fn codes and column-major "
                    "packed UE8M0 scales, the one combination the reference instantiates");
  check_input(input, "input");
  check_input(output_q, "output_q");
  TORCH_CHECK(input.numel() > 0, op, ": input.numel() > 0");
  TORCH_CHECK(std::fabs(1e-10 - eps) < 1e-13, op, ": eps must be 1e-10");
  const bool masked = given(masked_m);
  const int64_t rank = masked ? 3 : 2;
  TORCH_CHECK(output_s.dim() == rank, op, ": output_s.dim() == ", rank);
  TORCH_CHECK(input.dim() == output_s.dim() && output_q.dim() >= 2, op, ": input and output_s ranks differ");
  TORCH_CHECK(is_16bit(input.scalar_type()), op, ": input must be float16 or bfloat16");
  TORCH_CHECK(qmin == -448.0 && qmax == 448.0, op, ": CHECK_EQ(dst_dtype_info::MIN/MAX, min_8bit/max_8bit) failed");
  const int64_t H = output_q.size(-1), T = output_q.size(-2), E = masked ? input.size(0) : 1;
  TORCH_CHECK(input.size(-1) == 2 * H && input.size(-2) == T, op, ": input must be [..., tokens, 2 * hidden]");
  TORCH_CHECK(H % 128 == 0, op, ": hidden size must be a multiple of 128");
  TORCH_CHECK(output_s.size(-2) == T && output_s.size(-1) * 4 >= H / 128, op, ": output_s shape mismatch");
  if (masked)
    TORCH_CHECK(masked_m->is_cuda() && masked_m->scalar_type() == ScalarType::Int && masked_m->numel() == E && masked_m->is_contiguous(),
                op, ": masked_m must be a contiguous int32 CUDA tensor with one entry per expert");
  check(mi355_silu_mul_group_quant_fp8(input.const_data_ptr(), dtype_code(input.scalar_type()), output_q.data_ptr(), output_s.data_ptr(), E,
                                       T, H, static_cast<const int32_t*>(data_or_null(masked_m)), masked ? output_s.stride(0) : 0,
                                       output_s.stride(-1), current_stream()));
}

// sgl-kernel/csrc/gemm/per_token_group_quant_8bit_v2.cu:394-514: q = x * (max / amax)
void per_token_group_quant_8bit_v2(const Tensor& input, const Tensor& output_q, const Tensor& output_s, int64_t group, double eps,
                                   double qmin, double qmax, bool scale_ue8m0, bool fuse_silu_and_mul, const OptTensor& masked_m) {
  const char* op = "sgl_per_token_group_quant_8bit_v2";
  if (fuse_silu_and_mul) return silu_mul_group_quant(input, output_q, output_s, group, eps, qmin, qmax, scale_ue8m0, masked_m, op);
  if (given(masked_m))
    C10_THROW_ERROR(NotImplementedError, std::string(op) + ": masked_m without fuse_silu_and_mul has no kernel in the reference either");
  TORCH_CHECK(input.numel() > 0, op, ": input.numel() > 0");
  TORCH_CHECK(std::fabs(1e-10 - eps) < 1e-13, op, ": eps must be 1e-10");
  TORCH_CHECK(group == 16 || group == 32 || group == 64 || group == 128, "Unsupported group_size");
  TORCH_CHECK(is_16bit(input.scalar_type()), op, ": input must be float16 or bfloat16");
  const bool fp8 = output_q.scalar_type() == FP8;
  TORCH_CHECK(qmin == (fp8 ? -448.0 : -128.0) && qmax == (fp8 ? 448.0 : 127.0), op,
              ": CHECK_EQ(dst_dtype_info::MIN/MAX, min_8bit/max_8bit) failed");
  group_quant(input, output_q, output_s, group, eps, qmin, qmax, scale_ue8m0, MI355_QUANT_MUL, 0.0, op);
}

// sgl-kernel/csrc/gemm/per_token_quant_fp8.cu:162-227
void per_token_quant_fp8(const Tensor& input, const Tensor& output_q, const Tensor& output_s) {
  check_input(input, "input");
  check_input(output_q, "output_q");
  check_input(output_s, "output_s");
  TORCH_CHECK(input.dim() == 2, "sgl_per_token_quant_fp8: input must be 2-D");
  const int64_t M = input.size(0), K = input.size(1);
  TORCH_CHECK(K % 8 == 0, "Hidden dimension must be divisible by 8, but got ", K);
  TORCH_CHECK(is_float(input.scalar_type()), "sgl_per_token_quant_fp8: unsupported input dtype");
  TORCH_CHECK(output_q.scalar_type() == FP8 && output_q.numel() == input.numel(), "sgl_per_token_quant_fp8: output_q mismatch");
  TORCH_CHECK(output_s.scalar_type() == ScalarType::Float && output_s.numel() == M, "sgl_per_token_quant_fp8: output_s mismatch");
  if (M > 0)
    check(mi355_per_token_quant_fp8(input.const_data_ptr(), dtype_code(input.scalar_type()), output_q.data_ptr(),
                                    static_cast<float*>(output_s.data_ptr()), M, K, current_stream()));
}

// sgl-kernel/csrc/gemm/per_tensor_quant_fp8.cu:102-130.  Dynamic mode merges block maxima into `output_s` with an atomic max,
// so the caller passes zeros (the reference's scaled_fp8_quant does).
void per_tensor_quant_fp8(const Tensor& input, const Tensor& output_q, const Tensor& output_s, bool is_static) {
  check_input(input, "input");
  check_input(output_q, "output_q");
  check_input(output_s, "output_s");
  TORCH_CHECK(is_float(input.scalar_type()), "sgl_per_tensor_quant_fp8: unsupported input dtype");
  TORCH_CHECK(output_q.scalar_type() == FP8 && output_q.numel() >= input.numel(), "sgl_per_tensor_quant_fp8: output_q mismatch");
  TORCH_CHECK(output_s.scalar_type() == ScalarType::Float && output_s.numel() >= 1, "sgl_per_tensor_quant_fp8: output_s mismatch");
  check(mi355_per_tensor_quant_fp8(input.const_data_ptr(), dtype_code(input.scalar_type()), output_q.data_ptr(),
                                   static_cast<float*>(output_s.data_ptr()), input.numel(), is_static ? 1 : 0, nullptr, 0,
                                   current_stream()));
}

// Static per-tensor quantization that also writes the scale once per row (static_quant_fp8 with repeat_scale,
// python/sglang/srt/layers/quantization/fp8_kernel.py:635-665).
void static_quant_fp8_repeat(const Tensor& input, const Tensor& output_q, const Tensor& scale, const Tensor& scale_rows) {
  check_input(input, "input");
  check_input(output_q, "output_q");
  TORCH_CHECK(scale.numel() == 1 && scale.scalar_type() == ScalarType::Float && scale.is_cuda(), "only supports per-tensor scale");
  TORCH_CHECK(scale_rows.scalar_type() == ScalarType::Float && scale_rows.is_contiguous(), "scale_rows must be contiguous float32");
  check(mi355_per_tensor_quant_fp8(input.const_data_ptr(), dtype_code(input.scalar_type()), output_q.data_ptr(),
                                   static_cast<float*>(scale.data_ptr()), input.numel(), 1, static_cast<float*>(scale_rows.data_ptr()),
                                   scale_rows.numel(), current_stream()));
}

// Codes and scales of the rows of `x2d`; with `x_sum` ([M], the input's type) also the row sums.
void per_token_quant_int8(const Tensor& x2d, const Tensor& q, const Tensor& s, const OptTensor& x_sum) {
  TORCH_CHECK(x2d.dim() == 2, "per_token_quant_int8: x must be 2-D");
  const int64_t M = x2d.size(0), K = x2d.size(1);
  if (M == 0) return;
  if (!given(x_sum)) {
    check(mi355_per_token_quant_int8(x2d.const_data_ptr(), dtype_code(x2d.scalar_type()), q.data_ptr(), static_cast<float*>(s.data_ptr()), M,
                                     K, current_stream()));
  } else {
    TORCH_CHECK(x_sum->scalar_type() == x2d.scalar_type() && x_sum->numel() == M && x_sum->is_contiguous(),
                "x_sum must be [M] in the input's type");
    check(mi355_per_token_quant_int8_sum(x2d.const_data_ptr(), dtype_code(x2d.scalar_type()), q.data_ptr(),
                                         static_cast<float*>(s.data_ptr()), x_sum->data_ptr(), M, K, current_stream()));
  }
}

// ---------------------------------------------------------------- GEMMs

void launch_fp8_mm(const Tensor& a, const void* b, int64_t ldb, const Tensor& sa, const void* sb, int64_t sb_sn, int64_t sb_sk,
                   const Tensor& out, int64_t M, int64_t N, int64_t K) {
  const Workspace ws(mi355_fp8_blockwise_mm_workspace_bytes(M, N, K));
  check(mi355_fp8_blockwise_mm(a.const_data_ptr(), b, static_cast<const float*>(sa.const_data_ptr()), static_cast<const float*>(sb),
                               out.data_ptr(), dtype_code(out.scalar_type()), M, N, K, a.stride(0), ldb, sa.stride(0), sa.stride(1), sb_sn,
                               sb_sk, out.stride(0), ws.ptr(), ws.bytes, current_stream()));
}

bool is_contiguous_vector(const Tensor& t) {
  return t.is_contiguous() && (t.dim() == 1 || (t.dim() == 2 && (t.size(0) == 1 || t.size(1) == 1)));
}

// sgl-kernel/csrc/gemm/fp8_blockwise_gemm_kernel.cu:368-465
Tensor fp8_blockwise_scaled_mm(const Tensor& mat_a, const Tensor& mat_b, const Tensor& scales_a, const Tensor& scales_b,
                               ScalarType out_dtype) {
  check_mm_operands(mat_a, mat_b);
  TORCH_CHECK(mat_a.size(1) * (int64_t)mat_a.element_size() % 16 == 0, "mat_a must be multiple of 16 bytes for memory alignment");
  TORCH_CHECK(mat_b.size(0) * (int64_t)mat_b.element_size() % 16 == 0, "mat_b must be multiple of 16 bytes for memory alignment");
  TORCH_CHECK(mat_a.scalar_type() == FP8, "mat_a must be Float8_e4m3fn");
  TORCH_CHECK(mat_b.scalar_type() == FP8, "mat_b must be Float8_e4m3fn");
  TORCH_CHECK(is_16bit(out_dtype), "out_dtype must be Half or BFloat16");
  const int64_t M = mat_a.size(0), K = mat_a.size(1), N = mat_b.size(1);
  TORCH_CHECK(scales_a.dim() == 2 && scales_b.dim() == 2, "scales must be 2D tensors");
  TORCH_CHECK(M == scales_a.size(0), "size of scales_a is not matched");
  TORCH_CHECK(K / 128 == scales_a.size(1), "size of scales_a is not matched");
  TORCH_CHECK(scales_a.stride(0) == 1 || is_contiguous_vector(scales_a), "scales_a must be M major");
  TORCH_CHECK(K / 128 == scales_b.size(0), "size of scales_b is not matched");
  TORCH_CHECK(N / 128 == scales_b.size(1), "size of scales_b is not matched");
  TORCH_CHECK(scales_b.stride(0) == 1 || is_contiguous_vector(scales_b), "scales_b must be K major");
  TORCH_CHECK(scales_a.scalar_type() == ScalarType::Float, "scales_a must be Float32");
  TORCH_CHECK(scales_b.scalar_type() == ScalarType::Float, "scales_b must be Float32");
  TORCH_CHECK(N * 2 % 16 == 0, "out must be multiple of 16 bytes for memory alignment");
  // the integer divisions above accept ragged K or N but leave the tail without scales
  TORCH_CHECK(K % 128 == 0 && N % 128 == 0, "fp8_blockwise_scaled_mm needs K and N to be multiples of 128");
  Tensor out = new_tensor({M, N}, out_dtype, mat_a);
  if (M > 0)
    launch_fp8_mm(mat_a, mat_b.const_data_ptr(), mat_b.stride(1), scales_a, scales_b.const_data_ptr(), scales_b.stride(1),
                  scales_b.stride(0), out, M, N, K);
  return out;
}

// The w8a8_block_fp8_matmul contract on flattened operands: b [N, K] row-major weight, sb [ceil(N/128), ceil(K/128)],
// sa [M, ceil(K/128)] any strides, ragged N and K allowed.
void block_fp8_matmul(const Tensor& a, const Tensor& b, const Tensor& sa, const Tensor& sb, const Tensor& out) {
  if (a.size(0) > 0)
    launch_fp8_mm(a, b.const_data_ptr(), b.stride(0), sa, sb.const_data_ptr(), sb.stride(0), sb.stride(1), out, a.size(0), b.size(0),
                  a.size(1));
}

// Blockwise FP8 GEMM with packed power-of-two scales on both sides (what deep_gemm's gemm_nt_f8f8bf16 computes for the
// reference, python/sglang/srt/layers/quantization/fp8_kernel.py:1047-1065).
Tensor fp8_blockwise_mm_ue8m0(const Tensor& a, const Tensor& b, const Tensor& a_words, const Tensor& b_words, ScalarType out_dtype,
                              const OptTensor& bias) {
  TORCH_CHECK(a.is_cuda() && b.is_cuda(), "fp8_blockwise_mm_ue8m0: operands must be CUDA tensors");
  TORCH_CHECK(a.dim() == 2 && b.dim() == 2 && a.stride(1) == 1 && b.stride(1) == 1, "fp8_blockwise_mm_ue8m0: row-major operands expected");
  TORCH_CHECK(a.scalar_type() == FP8 && b.scalar_type() == FP8, "fp8_blockwise_mm_ue8m0: operands must be Float8_e4m3fn");
  const int64_t M = a.size(0), K = a.size(1), N = b.size(0);
  TORCH_CHECK(b.size(1) == K, "fp8_blockwise_mm_ue8m0: shapes cannot be multiplied");
  const int64_t kw = ((K + 127) / 128 + 3) / 4;
  TORCH_CHECK(a_words.scalar_type() == ScalarType::Int && a_words.dim() == 2 && a_words.size(0) == M && a_words.size(1) >= kw,
              "fp8_blockwise_mm_ue8m0: a_words must be int32 [", M, ", >= ", kw, "]");
  TORCH_CHECK(b_words.scalar_type() == ScalarType::Int && b_words.dim() == 2 && b_words.size(0) == N && b_words.size(1) >= kw,
              "fp8_blockwise_mm_ue8m0: b_words must be int32 [", N, ", >= ", kw, "]");
  TORCH_CHECK(M <= 1 || a_words.stride(0) == 1, "fp8_blockwise_mm_ue8m0: a_words must be packed along tokens (stride(0) == 1)");
  TORCH_CHECK(is_16bit(out_dtype), "fp8_blockwise_mm_ue8m0: out_dtype must be Half or BFloat16");
  if (given(bias))
    TORCH_CHECK(bias->numel() == N && bias->is_contiguous() && bias->scalar_type() == out_dtype,
                "fp8_blockwise_mm_ue8m0: bias must be a contiguous [N] tensor of the output dtype");
  Tensor out = new_tensor({M, N}, out_dtype, a);
  if (M == 0 || N == 0) return out;
  const Workspace ws(mi355_fp8_blockwise_mm_ue8m0_workspace_bytes(M, N, K));
  check(mi355_fp8_blockwise_mm_ue8m0(a.const_data_ptr(), b.const_data_ptr(), a_words.const_data_ptr(), b_words.const_data_ptr(),
                                     data_or_null(bias), out.data_ptr(), dtype_code(out_dtype), M, N, K, a.stride(0), b.stride(0),
                                     a_words.stride(1), b_words.stride(0), b_words.stride(1), out.stride(0), ws.ptr(), ws.bytes,
                                     current_stream()));
  return out;
}

// sgl-kernel/csrc/gemm/fp8_gemm_kernel.cu:1450-1532
Tensor fp8_scaled_mm(const Tensor& mat_a, const Tensor& mat_b, const Tensor& scales_a, const Tensor& scales_b, ScalarType out_dtype,
                     const OptTensor& bias) {
  check_mm_operands(mat_a, mat_b);
  TORCH_CHECK(mat_a.size(1) * (int64_t)mat_a.element_size() % 16 == 0, "mat_a must be multiple of 16 bytes for memory alignment");
  TORCH_CHECK(mat_b.size(0) * (int64_t)mat_b.element_size() % 16 == 0, "mat_b must be multiple of 16 bytes for memory alignment");
  TORCH_CHECK(mat_a.scalar_type() == FP8, "mat_a must be Float8_e4m3fn");
  TORCH_CHECK(mat_b.scalar_type() == FP8, "mat_b must be Float8_e4m3fn");
  TORCH_CHECK(is_16bit(out_dtype), "out_dtype must be Half or BFloat16");
  const int64_t M = mat_a.size(0), K = mat_a.size(1), N = mat_b.size(1);
  check_channel_scales(scales_a, scales_b, bias, M, N, out_dtype);
  TORCH_CHECK(N * 2 % 16 == 0, "out must be multiple of 16 bytes for memory alignment");
  Tensor out = new_tensor({M, N}, out_dtype, mat_a);
  if (M == 0) return out;
  const Workspace ws(mi355_fp8_scaled_mm_workspace_bytes(M, N, K));
  check(mi355_fp8_scaled_mm(mat_a.const_data_ptr(), mat_b.const_data_ptr(), static_cast<const float*>(scales_a.const_data_ptr()),
                            static_cast<const float*>(scales_b.const_data_ptr()), data_or_null(bias), out.data_ptr(), dtype_code(out_dtype),
                            M, N, K, mat_a.stride(0), mat_b.stride(1), out.stride(0), ws.ptr(), ws.bytes, current_stream()));
  return out;
}

void launch_int8_mm(const Tensor& a, const Tensor& b, const void* sa, const void* sb, const void* bias, const Tensor& out) {
  const int64_t M = a.size(0), K = a.size(1), N = b.size(1);
  const Workspace ws(mi355_int8_scaled_mm_workspace_bytes(M, N, K));
  check(mi355_int8_scaled_mm(a.const_data_ptr(), b.const_data_ptr(), static_cast<const float*>(sa), static_cast<const float*>(sb), bias,
                             out.data_ptr(), dtype_code(out.scalar_type()), M, N, K, a.stride(0), b.stride(1), out.stride(0), ws.ptr(),
                             ws.bytes, current_stream()));
}

// sgl-kernel/csrc/gemm/int8_gemm_kernel.cu:663-747
Tensor int8_scaled_mm(const Tensor& mat_a, const Tensor& mat_b, const Tensor& scales_a, const Tensor& scales_b, ScalarType out_dtype,
                      const OptTensor& bias) {
  check_mm_operands(mat_a, mat_b);
  TORCH_CHECK(mat_a.size(1) % 16 == 0, "mat_a.size(1) must be multiple of 16 for memory alignment");
  TORCH_CHECK(mat_b.size(0) % 16 == 0, "mat_b.size(0) must be multiple of 16 for memory alignment");
  TORCH_CHECK(mat_b.size(1) % 8 == 0, "mat_b.size(1) must be multiple of 8 for memory alignment");
  TORCH_CHECK(mat_a.scalar_type() == ScalarType::Char, "mat_a must be Int8");
  TORCH_CHECK(mat_b.scalar_type() == ScalarType::Char, "mat_b must be Int8");
  TORCH_CHECK(is_16bit(out_dtype), "out_dtype must be Half or BFloat16");
  const int64_t M = mat_a.size(0), N = mat_b.size(1);
  check_channel_scales(scales_a, scales_b, bias, M, N, out_dtype);
  Tensor out = new_tensor({M, N}, out_dtype, mat_a);
  if (M > 0) launch_int8_mm(mat_a, mat_b, scales_a.const_data_ptr(), scales_b.const_data_ptr(), data_or_null(bias), out);
  return out;
}

// int32 accumulators of int8_scaled_mm before its epilogue (same kernel, epilogue skipped)
Tensor int8_mm_raw_accumulators(const Tensor& mat_a, const Tensor& mat_b) {
  Tensor out = new_tensor({mat_a.size(0), mat_b.size(1)}, ScalarType::Int, mat_a);
  if (mat_a.size(0) > 0) launch_int8_mm(mat_a, mat_b, nullptr, nullptr, nullptr, out);
  return out;
}

// ---------------------------------------------------------------- grouped FP8 GEMM (mixture-of-experts)

// Checks common to both grouped entry points (fp8_blockwise_moe_kernel.cu:668-677, es_fp8_blockwise.cu:46-55), the layout
// checks the kernels need, and the call.
void grouped_mm(const char* op, const Tensor& output, const Tensor& a, const Tensor& b, const Tensor& scales_a, const Tensor& scales_b,
                const Tensor& problem_sizes, const Tensor& expert_offsets, const Tensor& workspace) {
  TORCH_CHECK(problem_sizes.dim() == 2, "problem_sizes must be 2D tensor");
  TORCH_CHECK(problem_sizes.size(1) == 3, "problem_sizes must have shape (num_experts, 3)");
  TORCH_CHECK(problem_sizes.size(0) == expert_offsets.size(0), "Number of experts in problem_sizes must match expert_offsets");
  TORCH_CHECK(problem_sizes.scalar_type() == ScalarType::Int, "problem_sizes must be int32");
  TORCH_CHECK(a.scalar_type() == FP8, "a must be kFloat8_e4m3fn");
  TORCH_CHECK(b.scalar_type() == FP8, "b must be kFloat8_e4m3fn");
  TORCH_CHECK(is_16bit(output.scalar_type()), "output must be bfloat16 or half");
  TORCH_CHECK(scales_a.scalar_type() == ScalarType::Float, "scales_a must be float32");
  TORCH_CHECK(scales_b.scalar_type() == ScalarType::Float, "scales_b must be float32");
  TORCH_CHECK(expert_offsets.scalar_type() == ScalarType::Int && expert_offsets.dim() == 1, "expert_offsets must be a 1D int32 tensor");
  TORCH_CHECK(output.dim() == 2, "output must be 2D tensor");
  TORCH_CHECK(a.dim() == 2, "a must be 2D tensor");
  TORCH_CHECK(b.dim() == 3, "b must be 3D tensor");
  TORCH_CHECK(scales_a.dim() == 2, "scales_a must be 2D tensor");
  TORCH_CHECK(scales_b.dim() == 3, "scales_b must be 3D tensor");
  TORCH_CHECK(workspace.dim() == 1, "workspace must be 1D tensor");
  TORCH_CHECK(a.is_cuda() && b.is_cuda() && output.is_cuda() && problem_sizes.is_cuda() && expert_offsets.is_cuda(), op,
              ": tensors must be CUDA tensors");
  const int64_t total_m = a.size(0), K = a.size(1), E = b.size(0), N = b.size(2);
  TORCH_CHECK(b.size(1) == K && output.size(0) == total_m && output.size(1) == N && problem_sizes.size(0) == E, op,
              ": shapes do not fit together");
  TORCH_CHECK(a.stride(1) == 1 && output.stride(1) == 1, op, ": a and output must be row-major");
  TORCH_CHECK(b.stride(1) == 1 || K == 1, op, ": b must be column-major per expert ([E, K, N] view of [E, N, K] storage)");
  const int64_t kb = (K + 127) / 128, nb = (N + 127) / 128;
  TORCH_CHECK(scales_a.size(0) == total_m && scales_a.size(1) == kb, op, ": scales_a must be [", total_m, ", ", kb, "]");
  TORCH_CHECK(scales_b.size(0) == E && scales_b.size(1) == kb && scales_b.size(2) == nb, op, ": scales_b must be [", E, ", ", kb, ", ", nb,
              "]");
  TORCH_CHECK(expert_offsets.is_contiguous() && problem_sizes.is_contiguous(), op, ": problem_sizes and expert_offsets must be contiguous");
  if (total_m == 0 || N == 0 || E == 0) return;
  const size_t need = mi355_fp8_blockwise_scaled_grouped_mm_workspace_bytes(E, total_m, N, K);
  void* ws_ptr = workspace.data_ptr();
  size_t ws_bytes = (size_t)workspace.numel() * workspace.element_size();
  const bool usable = workspace.is_cuda() && workspace.is_contiguous() && ws_bytes >= need && reinterpret_cast<uintptr_t>(ws_ptr) % 256 == 0;
  const Workspace own(usable ? 0 : need);
  if (!usable) ws_ptr = own.ptr(), ws_bytes = need;
  check(mi355_fp8_blockwise_scaled_grouped_mm(
      a.const_data_ptr(), b.const_data_ptr(), static_cast<const float*>(scales_a.const_data_ptr()),
      static_cast<const float*>(scales_b.const_data_ptr()), output.data_ptr(), dtype_code(output.scalar_type()),
      static_cast<const int32_t*>(problem_sizes.const_data_ptr()), static_cast<const int32_t*>(expert_offsets.const_data_ptr()), E, total_m, N,
      K, a.stride(0), b.stride(2), b.stride(0), scales_a.stride(0), scales_a.stride(1), scales_b.stride(0), scales_b.stride(2),
      scales_b.stride(1), output.stride(0), ws_ptr, ws_bytes, current_stream()));
}

// sgl-kernel/csrc/moe/fp8_blockwise_moe_kernel.cu:650-810 (checks :668-706).  The pointer, stride and scale-layout tensors are
// scratch of the reference's kernels: they are type-checked like there and not used.
void fp8_blockwise_scaled_grouped_mm(const Tensor& output, const Tensor& a_ptrs, const Tensor& b_ptrs, const Tensor& out_ptrs,
                                     const Tensor& a_scales_ptrs, const Tensor& b_scales_ptrs, const Tensor& a, const Tensor& b,
                                     const Tensor& scales_a, const Tensor& scales_b, const Tensor& stride_a, const Tensor& stride_b,
                                     const Tensor& stride_c, const Tensor& layout_sfa, const Tensor& layout_sfb, const Tensor& problem_sizes,
                                     const Tensor& expert_offsets, const Tensor& workspace) {
  const auto is_stride = [](const Tensor& t, const char* name) {
    TORCH_CHECK(t.scalar_type() == ScalarType::Long && t.dim() == 1, name, " must be a 1D int64 tensor");
  };
  is_stride(stride_a, "stride_a"), is_stride(stride_b, "stride_b"), is_stride(stride_c, "stride_c");
  const auto is_layout = [](const Tensor& t, const char* name) {
    TORCH_CHECK(t.scalar_type() == ScalarType::Int && t.dim() == 2, name, " must be a 2D int32 tensor");
  };
  is_layout(layout_sfa, "layout_sfa"), is_layout(layout_sfb, "layout_sfb");
  const auto is_vector = [](const Tensor& t, const char* name) { TORCH_CHECK(t.dim() == 1, name, " must be 1D tensor"); };
  is_vector(a_ptrs, "a_ptrs"), is_vector(b_ptrs, "b_ptrs"), is_vector(out_ptrs, "out_ptrs");
  is_vector(a_scales_ptrs, "a_scales_ptrs"), is_vector(b_scales_ptrs, "b_scales_ptrs");
  grouped_mm("fp8_blockwise_scaled_grouped_mm", output, a, b, scales_a, scales_b, problem_sizes, expert_offsets, workspace);
}

// sgl-kernel/csrc/expert_specialization/es_fp8_blockwise.cu:33-170: the same computation without the scratch tensors
void es_fp8_blockwise_scaled_grouped_mm(const Tensor& output, const Tensor& a, const Tensor& b, const Tensor& scales_a,
                                        const Tensor& scales_b, const Tensor& /*stride_a*/, const Tensor& /*stride_b*/,
                                        const Tensor& /*stride_d*/, const Tensor& problem_sizes, const Tensor& expert_offsets,
                                        const Tensor& workspace) {
  grouped_mm("es_fp8_blockwise_scaled_grouped_mm", output, a, b, scales_a, scales_b, problem_sizes, expert_offsets, workspace);
}

// ---------------------------------------------------------------- one-call linears

void check_bias(const OptTensor& bias, int64_t N, ScalarType out_dtype, const char* op) {
  if (given(bias))
    TORCH_CHECK(bias->numel() == N && bias->is_contiguous() && bias->scalar_type() == out_dtype, op,
                ": bias must be a contiguous [N] tensor of the output dtype");
}

// The launches without checks: `x` holds M rows of K values, `out` M rows of N.
void launch_block_linear(const Tensor& x, const Tensor& w, const Tensor& ws, const void* bias, const Tensor& out, int64_t M, int64_t N,
                         int64_t K, bool by_reciprocal, int bias_flag = 0) {
  const Workspace mem(mi355_fp8_block_linear_workspace_bytes(M, N, K));
  check(mi355_fp8_block_linear_mode(x.const_data_ptr(), dtype_code(x.scalar_type()), by_reciprocal ? MI355_QUANT_RCP : MI355_QUANT_DIV,
                                    w.const_data_ptr(), static_cast<const float*>(ws.const_data_ptr()), ws.stride(0), ws.stride(1), bias,
                                    out.data_ptr(), dtype_code(out.scalar_type()) | bias_flag, M, N, K, w.stride(0), N, mem.ptr(), mem.bytes,
                                    current_stream()));
}
void launch_block_linear_ue8m0(const Tensor& x, const Tensor& w, const Tensor& words, const void* bias, const Tensor& out, int64_t M,
                               int64_t N, int64_t K, int bias_flag = 0) {
  const Workspace mem(mi355_fp8_block_linear_ue8m0_workspace_bytes(M, N, K));
  check(mi355_fp8_block_linear_ue8m0(x.const_data_ptr(), dtype_code(x.scalar_type()), w.const_data_ptr(), words.const_data_ptr(),
                                     words.stride(0), words.stride(1), bias, out.data_ptr(), dtype_code(out.scalar_type()) | bias_flag, M, N, K,
                                     w.stride(0), N, mem.ptr(), mem.bytes, current_stream()));
}
void launch_per_token_linear(const Tensor& x, const Tensor& w_kn, const Tensor& ws, const void* bias, const Tensor& out, int64_t M,
                             int64_t N, int64_t K) {
  const Workspace mem(mi355_fp8_per_token_linear_workspace_bytes(M, N, K));
  check(mi355_fp8_per_token_linear(x.const_data_ptr(), dtype_code(x.scalar_type()), w_kn.const_data_ptr(),
                                   static_cast<const float*>(ws.const_data_ptr()), bias, out.data_ptr(), dtype_code(out.scalar_type()), M, N,
                                   K, w_kn.stride(1), N, mem.ptr(), mem.bytes, current_stream()));
}
void launch_int8_linear(const Tensor& x, const Tensor& w_kn, const Tensor& ws, const void* bias, const Tensor& out, int64_t M, int64_t N,
                        int64_t K) {
  const Workspace mem(mi355_int8_linear_workspace_bytes(M, N, K));
  check(mi355_int8_linear(x.const_data_ptr(), dtype_code(x.scalar_type()), w_kn.const_data_ptr(), static_cast<const float*>(ws.const_data_ptr()),
                          bias, out.data_ptr(), dtype_code(out.scalar_type()), M, N, K, w_kn.stride(1), N, mem.ptr(), mem.bytes,
                          current_stream()));
}

Tensor block_fp8_linear(const Tensor& x2d, const Tensor& weight, const Tensor& weight_scale, const OptTensor& bias, ScalarType out_dtype,
                        bool by_reciprocal) {
  const char* op = "block_fp8_linear";
  TORCH_CHECK(x2d.is_cuda() && weight.is_cuda(), op, ": operands must be CUDA tensors");
  TORCH_CHECK(x2d.dim() == 2 && x2d.is_contiguous(), op, ": x must be a contiguous 2-D tensor");
  TORCH_CHECK(weight.dim() == 2 && weight.stride(1) == 1 && weight.scalar_type() == FP8, op,
              ": weight must be a row-major Float8_e4m3fn matrix");
  const int64_t M = x2d.size(0), K = x2d.size(1), N = weight.size(0);
  TORCH_CHECK(weight.size(1) == K && K % 128 == 0, op, ": K must match and be a multiple of 128");
  TORCH_CHECK(weight_scale.dim() == 2 && weight_scale.size(0) == (N + 127) / 128 && weight_scale.size(1) == K / 128 &&
                  weight_scale.scalar_type() == ScalarType::Float, op, ": weight_scale must be float32 [ceil(N/128), K/128]");
  TORCH_CHECK(is_16bit(out_dtype), op, ": out_dtype must be Half or BFloat16");
  check_bias(bias, N, out_dtype, op);
  Tensor out = new_tensor({M, N}, out_dtype, x2d);
  if (M > 0) launch_block_linear(x2d, weight, weight_scale, data_or_null(bias), out, M, N, K, by_reciprocal);
  return out;
}

Tensor block_fp8_linear_ue8m0(const Tensor& x2d, const Tensor& weight, const Tensor& weight_words, const OptTensor& bias,
                              ScalarType out_dtype) {
  const char* op = "block_fp8_linear_ue8m0";
  TORCH_CHECK(x2d.is_cuda() && weight.is_cuda(), op, ": operands must be CUDA tensors");
  TORCH_CHECK(x2d.dim() == 2 && x2d.is_contiguous() && is_16bit(x2d.scalar_type()), op, ": x must be a contiguous 2-D bf16/fp16 tensor");
  TORCH_CHECK(weight.dim() == 2 && weight.stride(1) == 1 && weight.scalar_type() == FP8, op,
              ": weight must be a row-major Float8_e4m3fn matrix");
  const int64_t M = x2d.size(0), K = x2d.size(1), N = weight.size(0);
  TORCH_CHECK(weight.size(1) == K && K % 128 == 0, op, ": K must match and be a multiple of 128");
  const int64_t kw = (K / 128 + 3) / 4;
  TORCH_CHECK(weight_words.scalar_type() == ScalarType::Int && weight_words.dim() == 2 && weight_words.size(0) == N &&
                  weight_words.size(1) >= kw, op, ": weight_words must be int32 [", N, ", >= ", kw, "]");
  TORCH_CHECK(is_16bit(out_dtype), op, ": out_dtype must be Half or BFloat16");
  check_bias(bias, N, out_dtype, op);
  Tensor out = new_tensor({M, N}, out_dtype, x2d);
  if (M > 0 && N > 0) launch_block_linear_ue8m0(x2d, weight, weight_words, data_or_null(bias), out, M, N, K);
  return out;
}

Tensor fp8_per_token_linear(const Tensor& x2d, const Tensor& weight_kn, const Tensor& weight_scale, const OptTensor& bias,
                            ScalarType out_dtype) {
  const char* op = "fp8_per_token_linear";
  TORCH_CHECK(x2d.is_cuda() && weight_kn.is_cuda(), op, ": operands must be CUDA tensors");
  TORCH_CHECK(x2d.dim() == 2 && x2d.is_contiguous(), op, ": x must be a contiguous 2-D tensor");
  TORCH_CHECK(is_float(x2d.scalar_type()), op, ": unsupported input dtype");
  TORCH_CHECK(weight_kn.dim() == 2 && weight_kn.stride(0) == 1 && weight_kn.scalar_type() == FP8, op,
              ": weight must be a column-major Float8_e4m3fn matrix [K, N]");
  const int64_t M = x2d.size(0), K = x2d.size(1), N = weight_kn.size(1);
  TORCH_CHECK(weight_kn.size(0) == K, op, ": x and weight shapes cannot be multiplied");
  TORCH_CHECK(K % 16 == 0, op, ": K must be multiple of 16 bytes for memory alignment");
  TORCH_CHECK(weight_scale.numel() == N && weight_scale.is_contiguous() && weight_scale.scalar_type() == ScalarType::Float, op,
              ": weight_scale must be a contiguous Float32 tensor of N elements");
  TORCH_CHECK(is_16bit(out_dtype), op, ": out_dtype must be Half or BFloat16");
  TORCH_CHECK(N % 8 == 0, op, ": out must be multiple of 16 bytes for memory alignment");
  check_bias(bias, N, out_dtype, op);
  Tensor out = new_tensor({M, N}, out_dtype, x2d);
  if (M > 0) launch_per_token_linear(x2d, weight_kn, weight_scale, data_or_null(bias), out, M, N, K);
  return out;
}

Tensor int8_linear(const Tensor& x2d, const Tensor& weight_kn, const Tensor& weight_scale, const OptTensor& bias, ScalarType out_dtype) {
  const char* op = "int8_linear";
  TORCH_CHECK(x2d.is_cuda() && weight_kn.is_cuda(), op, ": operands must be CUDA tensors");
  TORCH_CHECK(x2d.dim() == 2 && x2d.is_contiguous(), op, ": x must be a contiguous 2-D tensor");
  TORCH_CHECK(is_float(x2d.scalar_type()), op, ": unsupported input dtype");
  TORCH_CHECK(weight_kn.dim() == 2 && weight_kn.stride(0) == 1 && weight_kn.scalar_type() == ScalarType::Char, op,
              ": weight must be a column-major Int8 matrix [K, N]");
  const int64_t M = x2d.size(0), K = x2d.size(1), N = weight_kn.size(1);
  TORCH_CHECK(weight_kn.size(0) == K, op, ": x and weight shapes cannot be multiplied");
  TORCH_CHECK(K % 16 == 0, op, ": K must be multiple of 16 for memory alignment");
  TORCH_CHECK(N % 8 == 0, op, ": N must be multiple of 8 for memory alignment");
  TORCH_CHECK(weight_scale.numel() == N && weight_scale.is_contiguous() && weight_scale.scalar_type() == ScalarType::Float, op,
              ": weight_scale must be a contiguous Float32 tensor of N elements");
  TORCH_CHECK(is_16bit(out_dtype), op, ": out_dtype must be Half or BFloat16");
  check_bias(bias, N, out_dtype, op);
  Tensor out = new_tensor({M, N}, out_dtype, x2d);
  if (M > 0) launch_int8_linear(x2d, weight_kn, weight_scale, data_or_null(bias), out, M, N, K);
  return out;
}

// ---------------------------------------------------------------- fast paths of the linear methods and the quantizer functions
// A std::nullopt means "not the operands this is for".

// [..., K] -> [..., N]
Tensor new_output(const Tensor& x, int64_t N) {
  c10::SmallVector<int64_t, 6> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = N;
  return new_plain_tensor(sizes, x.scalar_type(), x);
}
bool plain_activation(const Tensor& x) { return x.is_cuda() && x.dim() >= 1 && x.is_contiguous() && x.numel() > 0 && is_16bit(x.scalar_type()); }
bool plain_block_weight(const Tensor& w, int64_t K) {
  return w.dim() == 2 && w.is_cuda() && w.is_contiguous() && w.scalar_type() == FP8 && w.size(1) == K && w.size(0) > 0;
}
bool plain_epilogue_bias(const OptTensor& bias, ScalarType dtype, int64_t N) {
  return !given(bias) || (bias->is_cuda() && bias->scalar_type() == dtype && bias->is_contiguous() && bias->numel() == N);
}

// `output += bias` in the GEMM's epilogue (same bits, no pass over the output) where nothing about it is unusual
bool fused_bias(const OptTensor& bias, const Tensor& out, int64_t N) {
  return given(bias) && bias->dim() == 1 && bias->numel() == N && bias->is_contiguous() && bias->scalar_type() == out.scalar_type() &&
         bias->device() == out.device() && !(bias->requires_grad() && c10::GradMode::is_enabled());
}

// fp8_utils.triton_w8a8_block_fp8_linear / cutlass_w8a8_block_fp8_linear_with_fallback: the latter's `x / s` quantizer for
// N a multiple of 128, else the former's `x * (1 / s)`; the bias is added to the rounded output.
std::optional<Tensor> try_block_linear(const Tensor& x, const Tensor& w, const Tensor& ws, const OptTensor& bias, bool triton) {
  if (!plain_activation(x)) return std::nullopt;
  const int64_t K = x.size(-1), M = x.numel() / K;
  if (K % 128 != 0 || !plain_block_weight(w, K)) return std::nullopt;
  const int64_t N = w.size(0);
  if (ws.scalar_type() != ScalarType::Float || !ws.is_cuda() || ws.dim() != 2 || ws.size(0) != (N + 127) / 128 || ws.size(1) != K / 128)
    return std::nullopt;
  Tensor out = new_output(x, N);
  const bool fused = fused_bias(bias, out, N);
  launch_block_linear(x, w, ws, fused ? bias->const_data_ptr() : nullptr, out, M, N, K, triton || N % 128 != 0, MI355_BIAS_ON_ROUNDED);
  if (given(bias) && !fused) out.add_(*bias);
  return out;
}

// fp8_utils.deepgemm_w8a8_block_fp8_linear_with_fallback for packed weight scales
std::optional<Tensor> try_block_linear_ue8m0(const Tensor& x, const Tensor& w, const Tensor& words, const OptTensor& bias) {
  if (!plain_activation(x) || x.scalar_type() != ScalarType::BFloat16) return std::nullopt;
  const int64_t K = x.size(-1), M = x.numel() / K;
  if (K % 128 != 0 || !plain_block_weight(w, K)) return std::nullopt;
  const int64_t N = w.size(0);
  if (words.scalar_type() != ScalarType::Int || !words.is_cuda() || words.dim() != 2 || words.size(0) != N || words.size(1) < (K / 128 + 3) / 4)
    return std::nullopt;
  Tensor out = new_output(x, N);
  const bool fused = fused_bias(bias, out, N);
  launch_block_linear_ue8m0(x, w, words, fused ? bias->const_data_ptr() : nullptr, out, M, N, K, MI355_BIAS_ON_ROUNDED);
  if (given(bias) && !fused) out.add_(*bias);
  return out;
}

// Operands of the two per-channel linears: w [K, N] column-major, N fp32 channel scales, a bias for the epilogue.
bool plain_channel_operands(const Tensor& x, const Tensor& w, const Tensor& ws, const OptTensor& bias, ScalarType code) {
  if (!plain_activation(x) || w.dim() != 2) return false;
  const int64_t K = x.size(-1), N = w.size(1);
  return w.is_cuda() && w.scalar_type() == code && w.stride(0) == 1 && w.size(0) == K && K % 16 == 0 && N % 8 == 0 && N > 0 &&
         ws.is_cuda() && ws.scalar_type() == ScalarType::Float && ws.is_contiguous() && ws.numel() == N &&
         plain_epilogue_bias(bias, x.scalar_type(), N);
}

// w8a8_int8.apply_w8a8_int8_linear
std::optional<Tensor> try_int8_linear(const Tensor& x, const Tensor& w, const Tensor& ws, const OptTensor& bias) {
  if (!plain_channel_operands(x, w, ws, bias, ScalarType::Char)) return std::nullopt;
  const int64_t K = x.size(-1), N = w.size(1);
  Tensor out = new_output(x, N);
  launch_int8_linear(x, w, ws, data_or_null(bias), out, x.numel() / K, N, K);
  return out;
}

// fp8_utils.apply_fp8_linear without compressed_tensor_quant: dynamic per-token scales, or a static per-tensor input scale
std::optional<Tensor> try_token_linear(const Tensor& x, const Tensor& w, const Tensor& ws, const OptTensor& input_scale,
                                       const OptTensor& bias) {
  if (!plain_channel_operands(x, w, ws, bias, FP8)) return std::nullopt;
  const int64_t K = x.size(-1), N = w.size(1), M = x.numel() / K;
  if (!given(input_scale)) {
    Tensor out = new_output(x, N);
    launch_per_token_linear(x, w, ws, data_or_null(bias), out, M, N, K);
    return out;
  }
  if (!(input_scale->numel() == 1 && input_scale->is_cuda() && input_scale->scalar_type() == ScalarType::Float)) return std::nullopt;
  Tensor out = new_output(x, N);
  const Workspace mem(mi355_fp8_per_token_linear_workspace_bytes(M, N, K));
  check(mi355_fp8_static_linear(x.const_data_ptr(), dtype_code(x.scalar_type()), static_cast<const float*>(input_scale->const_data_ptr()),
                                w.const_data_ptr(), static_cast<const float*>(ws.const_data_ptr()), data_or_null(bias), out.data_ptr(),
                                dtype_code(out.scalar_type()), M, N, K, w.stride(1), N, mem.ptr(), mem.bytes, current_stream()));
  return out;
}

// A scale tensor with the shapes and strides of create_per_token_group_quant_fp8_output_scale
// (python/sglang/srt/layers/quantization/fp8_kernel.py:433-474) for a 2-D x, or any rank where the scales are row-major.
Tensor new_group_scales(const Tensor& x, int64_t group, bool column_major, bool tma_aligned, bool ue8m0) {
  const int64_t K = x.size(-1);
  if (!column_major) {
    c10::SmallVector<int64_t, 6> sizes(x.sizes().begin(), x.sizes().end());
    sizes.back() = K / group;
    return new_plain_tensor(sizes, ScalarType::Float, x);
  }
  const int64_t M = x.size(0), aligned = (M + 3) / 4 * 4;
  // words for `pitch` rows are allocated and the first M are the tensor
  const auto strided = [&](int64_t cols, int64_t pitch, ScalarType t) {
    return new_tensor_as({cols, pitch}, t, x, {M, cols}, {1, pitch});
  };
  if (ue8m0) return strided((K / 128 + 3) / 4, aligned, ScalarType::Int);
  return strided(K / group, tma_aligned ? aligned : M, ScalarType::Float);
}

struct Quantized {
  Tensor q, s;
};

// Codes and scales of x as new tensors.  by_wrapper: the arithmetic of fp8_kernel.per_token_group_quant_fp8 (row-major scales:
// x * (1 / s), column-major: x / s); otherwise that of the sgl_kernel operator (v2: x * (max / amax), else x / s).
std::optional<Quantized> try_group_quant(const Tensor& x, int64_t group, double eps, ScalarType code, bool column_major, bool tma_aligned,
                                         bool ue8m0, bool by_wrapper, bool v2) {
  if (!x.is_cuda() || x.dim() < 1 || !x.is_contiguous() || x.numel() == 0 || !is_float(x.scalar_type()) || group <= 0) return std::nullopt;
  const int64_t K = x.size(-1), M = x.numel() / K;
  const bool wide_row = group == K && (group * (int64_t)x.element_size() > 2048 || (group & (group - 1)));
  if (K % group != 0 || wide_row || (column_major && x.dim() != 2) || (ue8m0 && (!column_major || group != 128 || !tma_aligned)) ||
      (code != FP8 && code != ScalarType::Char) || (code != FP8 && column_major))
    return std::nullopt;
  if (!by_wrapper && x.dim() != 2) return std::nullopt;  // the operator takes 2-D scales
  if (v2 && (!is_16bit(x.scalar_type()) || std::fabs(1e-10 - eps) >= 1e-13 || !(group == 16 || group == 32 || group == 64 || group == 128)))
    return std::nullopt;
  Quantized r{new_plain_tensor(x.sizes(), code, x), new_group_scales(x, group, column_major, tma_aligned, ue8m0)};
  const int mode = by_wrapper ? (column_major ? MI355_QUANT_DIV : MI355_QUANT_RCP) : v2 ? MI355_QUANT_MUL : MI355_QUANT_DIV;
  const double qmin = code == FP8 ? -448.0 : -128.0, qmax = code == FP8 ? 448.0 : 127.0;
  launch_group_quant(x, r.q, r.s, M, K, group, eps, qmin, qmax, mode, ue8m0 ? MI355_SCALE_UE8M0_PACKED : MI355_SCALE_F32,
                     by_wrapper || v2 ? 0.0 : 1e-10, column_major ? 1 : K / group, column_major ? r.s.stride(1) : 1);
  return r;
}

// fp8_kernel._per_token_group_quant_8bit_fuse_silu_and_mul: x [T, 2H], or [E, T, 2H] with masked_m; rows past masked_m are zeros
std::optional<Quantized> try_silu_quant(const Tensor& x, const OptTensor& masked_m) {
  const bool masked = given(masked_m);
  if (!x.is_cuda() || x.dim() != (masked ? 3 : 2) || !x.is_contiguous() || x.numel() == 0 || !is_16bit(x.scalar_type())) return std::nullopt;
  const int64_t E = masked ? x.size(0) : 1, T = x.size(-2), H = x.size(-1) / 2;
  if (x.size(-1) % 256 != 0) return std::nullopt;
  if (masked && !(masked_m->is_cuda() && masked_m->scalar_type() == ScalarType::Int && masked_m->numel() == E && masked_m->is_contiguous()))
    return std::nullopt;
  const int64_t words = (H / 128 + 3) / 4, pitch = (T + 3) / 4 * 4;
  Quantized r;
  if (masked) {
    r.q = new_plain_tensor({E, T, H}, FP8, x);
    r.s = new_tensor_as({E, words, pitch}, ScalarType::Int, x, {E, T, words}, {words * pitch, 1, pitch});
  } else {
    r.q = new_plain_tensor({T, H}, FP8, x);
    r.s = new_tensor_as({words, pitch}, ScalarType::Int, x, {T, words}, {1, pitch});
  }
  check(mi355_silu_mul_group_quant_fp8_zero_rest(x.const_data_ptr(), dtype_code(x.scalar_type()), r.q.data_ptr(), r.s.data_ptr(), E, T, H,
                                                 static_cast<const int32_t*>(data_or_null(masked_m)), masked ? words * pitch : 0, pitch,
                                                 current_stream()));
  return r;
}

}  // namespace

TORCH_LIBRARY_IMPL(sgl_kernel, CUDA, m) {
  m.impl("int8_scaled_mm", &int8_scaled_mm);
  m.impl("fp8_blockwise_scaled_mm", &fp8_blockwise_scaled_mm);
  m.impl("sgl_per_token_group_quant_8bit", &per_token_group_quant_8bit);
  m.impl("sgl_per_token_group_quant_8bit_v2", &per_token_group_quant_8bit_v2);
  m.impl("fp8_scaled_mm", &fp8_scaled_mm);
  m.impl("sgl_per_token_quant_fp8", &per_token_quant_fp8);
  m.impl("sgl_per_tensor_quant_fp8", &per_tensor_quant_fp8);
  m.impl("fp8_blockwise_scaled_grouped_mm", &fp8_blockwise_scaled_grouped_mm);
  m.impl("es_fp8_blockwise_scaled_grouped_mm", &es_fp8_blockwise_scaled_grouped_mm);
}

// ---------------------------------------------------------------- Python calls
namespace {

const Tensor& as_tensor(PyObject* o) {
  TORCH_CHECK_TYPE(THPVariable_Check(o), "a Tensor is expected, got ", Py_TYPE(o)->tp_name);
  return THPVariable_Unpack(o);
}
OptTensor as_opt_tensor(PyObject* o) {
  if (o == Py_None) return std::nullopt;
  return as_tensor(o);
}
ScalarType as_dtype(PyObject* o) {
  TORCH_CHECK_TYPE(THPDtype_Check(o), "a dtype is expected, got ", Py_TYPE(o)->tp_name);
  return reinterpret_cast<THPDtype*>(o)->scalar_type;
}
int64_t as_int(PyObject* o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
double as_double(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw python_error();
  return v;
}
bool as_bool(PyObject* o) {
  const int v = PyObject_IsTrue(o);
  if (v < 0) throw python_error();
  return v != 0;
}

struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// How an argument of a C++ function is read from Python and a result given back.
template <class T> struct From;
template <> struct From<const Tensor&> { static const Tensor& get(PyObject* o) { return as_tensor(o); } };
template <> struct From<const OptTensor&> { static OptTensor get(PyObject* o) { return as_opt_tensor(o); } };
template <> struct From<ScalarType> { static ScalarType get(PyObject* o) { return as_dtype(o); } };
template <> struct From<int64_t> { static int64_t get(PyObject* o) { return as_int(o); } };
template <> struct From<double> { static double get(PyObject* o) { return as_double(o); } };
template <> struct From<bool> { static bool get(PyObject* o) { return as_bool(o); } };

PyObject* give(Tensor&& t) { return THPVariable_Wrap(std::move(t)); }
PyObject* give(std::optional<Tensor>&& t) {
  if (!t.has_value()) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(*t));
}
PyObject* give(std::optional<Quantized>&& r) {
  if (!r.has_value()) Py_RETURN_NONE;
  THPObjectPtr q(THPVariable_Wrap(std::move(r->q)));
  THPObjectPtr s(THPVariable_Wrap(std::move(r->s)));
  if (!q || !s) throw python_error();
  return PyTuple_Pack(2, q.get(), s.get());
}

template <auto FN> struct Call;
template <class R, class... A, R (*FN)(A...)> struct Call<FN> {
  template <size_t... I> static PyObject* go(PyObject* const* args, std::index_sequence<I...>) {
    // read every argument while the GIL is held, then let it go: a launch may wait for room in the queue
    std::tuple<decltype(From<A>::get(nullptr))...> a{From<A>::get(args[I])...};
    if constexpr (std::is_void_v<R>) {
      {
        NoGil no_gil;
        FN(std::get<I>(a)...);
      }
      Py_RETURN_NONE;
    } else {
      R r = [&] {
        NoGil no_gil;
        return FN(std::get<I>(a)...);
      }();
      return give(std::move(r));
    }
  }
  static PyObject* py(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == (Py_ssize_t)sizeof...(A), sizeof...(A), " arguments are expected, got ", n);
    return go(args, std::index_sequence_for<A...>{});
    END_HANDLE_TH_ERRORS
  }
};

bool is_pair_of_128(PyObject* o) {
  const bool list = PyList_CheckExact(o), tuple = PyTuple_CheckExact(o);
  if (!(list || tuple) || (list ? PyList_GET_SIZE(o) : PyTuple_GET_SIZE(o)) != 2) return false;
  for (int i = 0; i < 2; ++i) {
    PyObject* v = list ? PyList_GET_ITEM(o, i) : PyTuple_GET_ITEM(o, i);
    if (!PyLong_CheckExact(v) || PyLong_AsLong(v) != 128) return false;
  }
  return true;
}

// Whether an operator called on tensors with these keys here and now would end in the CUDA kernel itself.  A fast path launches kernels without
// the dispatcher, so whoever listens there would see its allocations and not what fills them: modes, tracers and functional
// wrappers (vmap, grad) announce themselves in the thread's or a tensor's key set, function modes in a state of their own.
// Autograd and autocast keys may be set: the operators have no formula for either, and the calls record nothing with them.
bool plain_dispatch(c10::DispatchKeySet of_tensors) {
  using c10::DispatchKey;
  constexpr c10::DispatchKeySet direct({DispatchKey::Dense, DispatchKey::BackendSelect, DispatchKey::ADInplaceOrView,
                                        DispatchKey::AutogradFunctionality, DispatchKey::AutocastCUDA, DispatchKey::AutocastCPU});
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  const c10::DispatchKeySet keys = ((of_tensors | tls.included_) - tls.excluded_) - direct;
  return (keys.raw_repr() & ~c10::full_backend_mask) == 0 && !at::impl::torch_function_mode_enabled();
}

PyObject* plain_dispatch_py(PyObject*, PyObject* t) {
  HANDLE_TH_ERRORS
  return PyBool_FromLong(plain_dispatch(as_tensor(t).key_set()));
  END_HANDLE_TH_ERRORS
}

// The fast path FN, tried only for plain tensors (a subclass may mean something else by an operation), only where nobody looks
// on (plain_dispatch) and, where BLOCK is an argument's index, for 128 x 128 blocks; that argument is not handed on.
template <auto FN, int BLOCK> struct Try;
template <class R, class... A, R (*FN)(A...), int BLOCK> struct Try<FN, BLOCK> {
  static constexpr Py_ssize_t COUNT = (Py_ssize_t)sizeof...(A) + (BLOCK >= 0 ? 1 : 0);
  static PyObject* py(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK_TYPE(n == COUNT, COUNT, " arguments are expected, got ", n);
    PyObject* rest[sizeof...(A)];
    int at = 0;
    c10::DispatchKeySet keys;  // of all tensors together: the thread's state is looked up once a call
    for (int i = 0; i < COUNT; ++i) {
      if (i == BLOCK) {
        if (!is_pair_of_128(args[i])) Py_RETURN_NONE;
        continue;
      }
      if (THPVariable_Check(args[i])) {
        if (!THPVariable_CheckExact(args[i])) Py_RETURN_NONE;
        keys = keys | THPVariable_Unpack(args[i]).key_set();
      }
      rest[at++] = args[i];
    }
    if (!plain_dispatch(keys)) Py_RETURN_NONE;
    return Call<FN>::py(self, rest, (Py_ssize_t)sizeof...(A));
    END_HANDLE_TH_ERRORS
  }
};

// Truth value of an environment variable with the reference's spelling rules (sglang.srt.utils.get_bool_env_var), read at
// each call as there.  The GIL is held, as it is when Python changes the environment.
PyObject* env_flag(PyObject*, PyObject* name) {
  const char* key = PyUnicode_AsUTF8(name);
  if (key == nullptr) return nullptr;
  const char* v = std::getenv(key);
  const bool on = v != nullptr && (strcasecmp(v, "1") == 0 || strcasecmp(v, "true") == 0);
  return PyBool_FromLong(on);
}

PyObject* set_error_class(PyObject*, PyObject* cls) {
  Py_INCREF(cls);
  Py_XSETREF(g_error_class, cls);
  Py_RETURN_NONE;
}

#define CALL(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Call<&fn>::py)), METH_FASTCALL, nullptr}
#define TRY(name, fn, block) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Try<&fn, block>::py)), METH_FASTCALL, nullptr}

PyMethodDef METHODS[] = {
    CALL("int8_scaled_mm", int8_scaled_mm),
    CALL("fp8_blockwise_scaled_mm", fp8_blockwise_scaled_mm),
    CALL("sgl_per_token_group_quant_8bit", per_token_group_quant_8bit),
    CALL("sgl_per_token_group_quant_8bit_v2", per_token_group_quant_8bit_v2),
    CALL("fp8_scaled_mm", fp8_scaled_mm),
    CALL("sgl_per_token_quant_fp8", per_token_quant_fp8),
    CALL("sgl_per_tensor_quant_fp8", per_tensor_quant_fp8),
    CALL("fp8_blockwise_scaled_grouped_mm", fp8_blockwise_scaled_grouped_mm),
    CALL("es_fp8_blockwise_scaled_grouped_mm", es_fp8_blockwise_scaled_grouped_mm),
    CALL("static_quant_fp8_repeat", static_quant_fp8_repeat),
    CALL("per_token_quant_int8", per_token_quant_int8),
    CALL("block_fp8_matmul", block_fp8_matmul),
    CALL("fp8_blockwise_mm_ue8m0", fp8_blockwise_mm_ue8m0),
    CALL("int8_mm_raw_accumulators", int8_mm_raw_accumulators),
    CALL("block_fp8_linear", block_fp8_linear),
    CALL("block_fp8_linear_ue8m0", block_fp8_linear_ue8m0),
    CALL("fp8_per_token_linear", fp8_per_token_linear),
    CALL("int8_linear", int8_linear),
    TRY("try_block_linear", try_block_linear, 2),
    TRY("try_block_linear_ue8m0", try_block_linear_ue8m0, 2),
    TRY("try_int8_linear", try_int8_linear, -1),
    TRY("try_token_linear", try_token_linear, -1),
    TRY("try_group_quant", try_group_quant, -1),
    TRY("try_silu_quant", try_silu_quant, -1),
    {"plain_dispatch", &plain_dispatch_py, METH_O, nullptr},
    {"env_flag", &env_flag, METH_O, nullptr},
    {"set_error_class", &set_error_class, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef MODULE = {PyModuleDef_HEAD_INIT, "_native", "gfx950 quantized-linear operators for PyTorch-ROCm", -1, METHODS,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__native() { return PyModule_Create(&MODULE); }
