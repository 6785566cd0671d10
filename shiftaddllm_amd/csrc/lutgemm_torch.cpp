// Python module `lutgemm`: the reference extension's call signatures
// (lut_gemm/lutgemm_cuda.cpp:43-98,225-230 in the ShiftAddLLM checkout) on top
// of the gfx950 C ABI in lutgemm_gfx950.h.  Host-only translation unit: it
// validates tensors, picks the current HIP stream and forwards raw pointers.
//
// Differences from the reference bindings, all on the strict side:
//  * every operand is checked (dtype, device, contiguity, element counts) and a
//    violation raises instead of reading out of bounds;
//  * launches go to PyTorch's current stream of the output's device, not the
//    legacy default stream;
//  * `d_input` may hold M rows ([M, K] or [..., K]); the reference's row-wise
//    and uniform entry points are batch-1 only.
#include <torch/extension.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <string>
#include <type_traits>
#include <utility>
#include <vector>

#include "lutgemm_gfx950.h"

namespace {

void check_common(const torch::Tensor &output, const torch::Tensor &bWeight,
                  const torch::Tensor &d_input, int64_t mSize, int64_t kSize, int64_t nb, bool any_type = false)
{
    TORCH_CHECK(output.is_cuda(), "output must be a GPU tensor");
    TORCH_CHECK(bWeight.is_cuda() && d_input.is_cuda(), "bWeight and d_input must be GPU tensors");
    TORCH_CHECK(bWeight.get_device() == output.get_device() &&
                    d_input.get_device() == output.get_device(),
                "all operands must live on the same device");
    TORCH_CHECK(any_type || output.scalar_type() == torch::kHalf, "output must be float16");
    TORCH_CHECK(any_type || d_input.scalar_type() == torch::kHalf, "d_input must be float16");
    TORCH_CHECK(bWeight.scalar_type() == torch::kInt32, "bWeight must be int32");
    TORCH_CHECK(output.is_contiguous() && bWeight.is_contiguous() && d_input.is_contiguous(),
                "operands must be contiguous");
    TORCH_CHECK(kSize > 0 && kSize % 32 == 0, "kSize must be a positive multiple of 32, got ", kSize);
    TORCH_CHECK(mSize > 0 && mSize % 4 == 0, "mSize must be a positive multiple of 4, got ", mSize);
    TORCH_CHECK(nb >= 1 && nb <= 4, "nb must be in 1..4, got ", nb);
    TORCH_CHECK(bWeight.numel() == (kSize / 32) * nb * mSize, "bWeight must hold [kSize/32, nb, mSize] = ",
                (kSize / 32) * nb * mSize, " words, got ", bWeight.numel());
    TORCH_CHECK(d_input.numel() > 0 && d_input.numel() % kSize == 0 && d_input.size(-1) == kSize,
                "d_input must be [..., kSize]");
    const int64_t rows = d_input.numel() / kSize;
    TORCH_CHECK(output.numel() == rows * mSize, "output must hold ", rows * mSize,
                " elements ([rows, mSize]), got ", output.numel());
}

void check_alpha(const torch::Tensor &alpha, const torch::Tensor &output, c10::ScalarType dtype,
                 int64_t numel, const char *what)
{
    TORCH_CHECK(alpha.is_cuda() && alpha.get_device() == output.get_device(), what,
                " must be on the output's device");
    TORCH_CHECK(alpha.scalar_type() == dtype, what, " has the wrong dtype: expected ",
                c10::toString(dtype), ", got ", c10::toString(alpha.scalar_type()));
    TORCH_CHECK(alpha.is_contiguous(), what, " must be contiguous");
    TORCH_CHECK(alpha.numel() == numel, what, " must hold ", numel, " elements, got ", alpha.numel());
}

void raise_on_error(int rc, const char *fn)
{
    if (rc == LUTGEMM_OK) return;
    std::string msg = std::string(fn) + ": " + lutgemm_strerror(rc);
    if (rc == LUTGEMM_EHIP || rc == LUTGEMM_ENOMEM)
        msg += " [hipError " + std::to_string(lutgemm_last_hip_error()) + "]";
    TORCH_CHECK(false, msg);
}

int rows_of(const torch::Tensor &d_input, int64_t kSize) { return (int)(d_input.numel() / kSize); }

}  // namespace

// lutgemm_cuda.cpp:43-52
void lutgemm_compute_shift_scale(const torch::Tensor &output, const torch::Tensor &bWeight, const torch::Tensor &alpha,
                                 const torch::Tensor &d_input, int64_t mSize, int64_t kSize, int64_t nb,
                                 int64_t num_groups)
{
    check_common(output, bWeight, d_input, mSize, kSize, nb);
    TORCH_CHECK(num_groups > 0 && kSize % num_groups == 0 && (kSize / num_groups) % 32 == 0,
                "kSize/num_groups must be a multiple of 32");
    check_alpha(alpha, output, torch::kHalf, num_groups * nb * mSize, "alpha [num_groups, nb, mSize]");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(output.device());
    int rc = lutgemm_gemv_rowwise_f16((const uint32_t *)bWeight.data_ptr<int32_t>(), alpha.data_ptr(),
                                      d_input.data_ptr(), output.data_ptr(), (int)mSize, (int)kSize,
                                      (int)nb, (int)num_groups, rows_of(d_input, kSize),
                                      c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream());
    raise_on_error(rc, "lutgemm_compute_shift_scale");
}

// lutgemm_compute_shift_scale for alphas the caller knows to be powers of two (what the
// reference's quantiser produces, quantizers/bcq_quant/bcq_shift.py:15-24): a few rows on a large
// matrix take the block-scaled matrix-core kernel.  No counterpart in the reference's extension.
void lutgemm_compute_shift_scale_pow2(const torch::Tensor &output, const torch::Tensor &bWeight, const torch::Tensor &alpha,
                                      const torch::Tensor &d_input, int64_t mSize, int64_t kSize, int64_t nb,
                                      int64_t num_groups)
{
    check_common(output, bWeight, d_input, mSize, kSize, nb);
    TORCH_CHECK(num_groups > 0 && kSize % num_groups == 0 && (kSize / num_groups) % 32 == 0,
                "kSize/num_groups must be a multiple of 32");
    check_alpha(alpha, output, torch::kHalf, num_groups * nb * mSize, "alpha [num_groups, nb, mSize]");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(output.device());
    int rc = lutgemm_gemv_rowwise_pow2_f16((const uint32_t *)bWeight.data_ptr<int32_t>(), alpha.data_ptr(),
                                           d_input.data_ptr(), output.data_ptr(), (int)mSize, (int)kSize,
                                           (int)nb, (int)num_groups, rows_of(d_input, kSize),
                                           c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream());
    raise_on_error(rc, "lutgemm_compute_shift_scale_pow2");
}

// lutgemm_cuda.cpp:88-98
void lutgemm_compute(const torch::Tensor &output, const torch::Tensor &bWeight, const torch::Tensor &alpha,
                     const torch::Tensor &q_bias, const torch::Tensor &d_input, int64_t mSize, int64_t kSize,
                     int64_t nb, int64_t num_groups)
{
    check_common(output, bWeight, d_input, mSize, kSize, nb);
    TORCH_CHECK(num_groups > 0 && kSize % num_groups == 0 && (kSize / num_groups) % 32 == 0,
                "kSize/num_groups must be a multiple of 32");
    check_alpha(alpha, output, torch::kHalf, num_groups * mSize, "alpha [num_groups, mSize]");
    check_alpha(q_bias, output, torch::kHalf, num_groups * mSize, "q_bias [num_groups, mSize]");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(output.device());
    int rc = lutgemm_gemv_uniform_f16((const uint32_t *)bWeight.data_ptr<int32_t>(), alpha.data_ptr(),
                                      q_bias.data_ptr(), d_input.data_ptr(), output.data_ptr(),
                                      (int)mSize, (int)kSize, (int)nb, (int)num_groups,
                                      rows_of(d_input, kSize),
                                      c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream());
    raise_on_error(rc, "lutgemm_compute");
}

static void check_block(int64_t mSize, int64_t num_groups)
{
    TORCH_CHECK(num_groups > 0 && mSize % num_groups == 0 && (mSize / num_groups) % 4 == 0,
                "mSize/num_groups (rows per alpha block) must be a multiple of 4");
}

// lutgemm_cuda.cpp:54-63
void lutgemm_compute_block(const torch::Tensor &output, const torch::Tensor &bWeight, const torch::Tensor &alpha,
                           const torch::Tensor &d_input, int64_t mSize, int64_t kSize, int64_t nb,
                           int64_t num_groups)
{
    check_common(output, bWeight, d_input, mSize, kSize, nb);
    check_block(mSize, num_groups);
    check_alpha(alpha, output, torch::kHalf, (kSize / 8) * nb * num_groups,
                "alpha [kSize/8, nb, num_groups]");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(output.device());
    int rc = lutgemm_gemv_block_f16((const uint32_t *)bWeight.data_ptr<int32_t>(), alpha.data_ptr(),
                                    d_input.data_ptr(), output.data_ptr(), (int)mSize, (int)kSize,
                                    (int)nb, (int)num_groups, rows_of(d_input, kSize),
                                    c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream());
    raise_on_error(rc, "lutgemm_compute_block");
}

// lutgemm_cuda.cpp:65-74
void lutgemm_compute_block_shift(const torch::Tensor &output, const torch::Tensor &bWeight, const torch::Tensor &alpha,
                                 const torch::Tensor &d_input, int64_t mSize, int64_t kSize, int64_t nb,
                                 int64_t num_groups, int64_t num_apot)
{
    check_common(output, bWeight, d_input, mSize, kSize, nb);
    check_block(mSize, num_groups);
    TORCH_CHECK(num_apot == 3, "num_apot must be 3 (the packed uint16 always carries three shift fields)");
    check_alpha(alpha, output, torch::kShort, (kSize / 8) * nb * num_groups,
                "alpha [kSize/8, nb, num_groups] (int16 holding uint16 shift fields)");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(output.device());
    int rc = lutgemm_gemv_block_shift_u16((const uint32_t *)bWeight.data_ptr<int32_t>(),
                                          (const uint16_t *)alpha.data_ptr<int16_t>(),
                                          d_input.data_ptr(), output.data_ptr(), (int)mSize,
                                          (int)kSize, (int)nb, (int)num_groups, (int)num_apot,
                                          rows_of(d_input, kSize),
                                          c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream());
    raise_on_error(rc, "lutgemm_compute_block_shift");
}

// lutgemm_cuda.cpp:76-85
void lutgemm_compute_block_shiftInt8(const torch::Tensor &output, const torch::Tensor &bWeight,
                                     const torch::Tensor &alpha, const torch::Tensor &d_input, int64_t mSize,
                                     int64_t kSize, int64_t nb, int64_t num_groups, int64_t num_apot)
{
    check_common(output, bWeight, d_input, mSize, kSize, nb);
    check_block(mSize, num_groups);
    TORCH_CHECK(num_apot == 3, "num_apot must be 3 (alpha carries three int8 exponents per entry)");
    check_alpha(alpha, output, torch::kChar, (kSize / 8) * nb * num_groups * 3,
                "alpha [kSize/8, nb, num_groups, 3]");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(output.device());
    int rc = lutgemm_gemv_block_apot_i8((const uint32_t *)bWeight.data_ptr<int32_t>(),
                                        alpha.data_ptr<int8_t>(), d_input.data_ptr(),
                                        output.data_ptr(), (int)mSize, (int)kSize, (int)nb,
                                        (int)num_groups, (int)num_apot, rows_of(d_input, kSize),
                                        c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream());
    raise_on_error(rc, "lutgemm_compute_block_shiftInt8");
}

// ---- LutLinear.forward ------------------------------------------------------------------------
int io_type(c10::ScalarType t)
{
    return t == at::kHalf ? LUTGEMM_TYPE_F16 : t == at::kBFloat16 ? LUTGEMM_TYPE_BF16 : t == at::kFloat ? LUTGEMM_TYPE_F32 : -1;
}

// linear_forward(x, binaryWeight, alpha, bias, out, format, N, K, nb, num_groups, alpha_pow2) -> y
// The whole of lut_gemm/quant.py:41-54 in one native call: the activations as contiguous rows, the output
// [..., N] in their dtype (allocated here, or `out`, fp16 [rows, N], where the caller reuses one), ONE launch
// that adds the bias itself.  At one row the layer is bound by the host, not the device: through five
// framework calls and the checked functions above a forward took 11.9 us of host time around a 4.5 us
// kernel.  A plain CPython function, because the argument conversions of pybind11 are a tenth of what is left.
// bf16 and fp32 activations are converted by the kernel itself where it does that (the call says
// LUTGEMM_EUNSUP otherwise), and by a launch ahead of it elsewhere; the result is written in the caller's type.
// (A conversion is 4 us of host time and 3 of the device: bf16 rows of a 2208 x 2964 layer 14.5 -> 7.9 us.)
at::Tensor linear_forward(const at::Tensor &x, const at::Tensor &bW, const at::Tensor &alpha, const at::Tensor *bias,
                          const at::Tensor *out, int64_t format, int64_t N, int64_t K, int64_t nb, int64_t groups,
                          bool alpha_pow2)
{
    const auto dims = x.sizes();
    TORCH_CHECK_VALUE(!dims.empty() && dims.back() == K, "expected last dimension ", K, ", got ", dims);
    TORCH_CHECK(x.is_cuda(), "the input must be a GPU tensor");
    TORCH_CHECK(x.numel() > 0, "the input is empty");
    const int64_t rows = x.numel() / K;
    const auto device = x.device();
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(device);
    const c10::ScalarType dtype = x.scalar_type();
    c10::ScalarType out_dtype = out || io_type(dtype) < 0 ? at::kHalf : dtype;
    at::Tensor in = x.is_contiguous() ? x : x.contiguous();
    if (io_type(dtype) < 0 || (dtype != at::kHalf && (uintptr_t)in.const_data_ptr() % 16 != 0)) in = in.to(at::kHalf);

    c10::SmallVector<int64_t, 5> shape(dims.begin(), dims.end());
    shape.back() = N;
    auto allocate = [&]() { return at::Tensor(at::detail::empty_cuda(shape, out_dtype, device, c10::nullopt)); };
    at::Tensor y = out ? *out : allocate();
    check_common(y, bW, in, N, K, nb, out == nullptr);
    int64_t entries;
    c10::ScalarType type = at::kHalf;
    switch (format) {
    case LUTGEMM_FORMAT_ROWWISE_F16:
        TORCH_CHECK(groups > 0 && K % groups == 0 && (K / groups) % 32 == 0, "K/num_groups must be a multiple of 32");
        entries = groups * nb * N;
        break;
    case LUTGEMM_FORMAT_BLOCK_F16:
    case LUTGEMM_FORMAT_BLOCK_SHIFT_U16:
    case LUTGEMM_FORMAT_BLOCK_APOT_I8:
        check_block(N, groups);
        entries = (K / 8) * nb * groups * (format == LUTGEMM_FORMAT_BLOCK_APOT_I8 ? 3 : 1);
        if (format != LUTGEMM_FORMAT_BLOCK_F16) type = format == LUTGEMM_FORMAT_BLOCK_APOT_I8 ? at::kChar : at::kShort;
        break;
    default: TORCH_CHECK(false, "unknown alpha format ", format);
    }
    check_alpha(alpha, y, type, entries, "alpha");
    if (bias)
        TORCH_CHECK(bias->scalar_type() == at::kHalf && bias->device() == device && bias->is_contiguous() && bias->numel() == N,
                    "bias must be ", N, " contiguous float16 values on the input's device");
    lutgemm_linear layer{};
    layer.bW = (const uint32_t *)bW.const_data_ptr();
    layer.alpha = alpha.const_data_ptr();
    layer.bias_f16 = bias ? bias->const_data_ptr() : nullptr;
    layer.format = (int)format;
    layer.N = (int)N;
    layer.K = (int)K;
    layer.nb = (int)nb;
    layer.num_groups = (int)groups;
    layer.M = (int)rows;
    layer.alpha_pow2 = alpha_pow2;
    const auto stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
    auto launch = [&]() {
        layer.x = in.const_data_ptr();
        layer.x_type = io_type(in.scalar_type());
        layer.out = y.data_ptr();
        layer.out_type = io_type(out_dtype);
        return lutgemm_linear_f16(&layer, stream);
    };
    int rc = launch();
    if (rc == LUTGEMM_EUNSUP && layer.x_type != LUTGEMM_TYPE_F16) {
        in = in.to(at::kHalf);
        rc = launch();
    }
    if (rc == LUTGEMM_EUNSUP && layer.out_type != LUTGEMM_TYPE_F16) {
        out_dtype = at::kHalf;
        y = allocate();
        rc = launch();
    }
    raise_on_error(rc, "LutLinear.forward");
    if (out_dtype != dtype) y = y.to(dtype);
    return out ? y.view(shape) : y;
}

PyObject *linear_forward_py(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 11, "linear_forward takes 11 arguments");
    for (int i = 0; i < 5; ++i)
        TORCH_CHECK(THPVariable_Check(args[i]) || (i >= 3 && args[i] == Py_None), "argument ", i, " of linear_forward must be a tensor");
    int64_t v[6];
    for (int i = 0; i < 6; ++i) {
        v[i] = PyLong_AsLongLong(args[5 + i]);
        if (v[i] == -1 && PyErr_Occurred()) return nullptr;
    }
    const at::Tensor *bias = args[3] == Py_None ? nullptr : &THPVariable_Unpack(args[3]);
    const at::Tensor *out = args[4] == Py_None ? nullptr : &THPVariable_Unpack(args[4]);
    return THPVariable_Wrap(linear_forward(THPVariable_Unpack(args[0]), THPVariable_Unpack(args[1]), THPVariable_Unpack(args[2]),
                                           bias, out, v[0], v[1], v[2], v[3], v[4], v[5] != 0));
    END_HANDLE_TH_ERRORS
}

PyMethodDef linear_forward_def = {"linear_forward", (PyCFunction)(void (*)(void))linear_forward_py, METH_FASTCALL,
                                  "LutLinear.forward in one call"};

// Calibration copy for profiler byte counters (no reference counterpart).
void copy_bytes(torch::Tensor dst, torch::Tensor src)
{
    TORCH_CHECK(dst.is_cuda() && src.is_cuda() && dst.is_contiguous() && src.is_contiguous(),
                "copy_bytes needs contiguous GPU tensors");
    TORCH_CHECK(dst.nbytes() == src.nbytes() && dst.nbytes() % 16 == 0, "sizes must match, multiple of 16");
    const c10::hip::HIPGuardMasqueradingAsCUDA guard(dst.device());
    int rc = lutgemm_copy_bytes(dst.data_ptr(), src.data_ptr(), dst.nbytes(),
                                c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream());
    raise_on_error(rc, "copy_bytes");
}

// ---- test-data helpers of the reference module -------------------------------------
// (lut_gemm/lutgemm_cuda.cpp:104-223: makeRandom* fill a caller's tensor in place,
// element by element through index_put_; parsing moves host tensors to a device as the
// flat buffers the kernels read.)  Same signatures, the same value distributions and
// the same in-place contract, but generated by tensor operations on the tensor's own
// device, from PyTorch's generator of that device instead of the C library's rand().

// The reference's rand_fp32(): a random sign times the product of two uniforms in [0, 1].
torch::Tensor rand_fp32_like(const torch::Tensor &t, at::IntArrayRef shape)
{
    const auto opt = torch::TensorOptions().dtype(torch::kFloat32).device(t.device());
    const torch::Tensor sign = torch::randint(0, 2, shape, opt) * 2.0 - 1.0;
    return sign * torch::rand(shape, opt) * torch::rand(shape, opt);
}

void makeRandomInput(torch::Tensor inp, int64_t M, int64_t K)
{
    TORCH_CHECK(inp.dim() == 2 && inp.size(0) >= M && inp.size(1) >= K, "inp must be at least [M, K]");
    using namespace torch::indexing;
    inp.index_put_({Slice(0, M), Slice(0, K)}, rand_fp32_like(inp, {M, K}).to(inp.scalar_type()));
}

void makeRandomWeight(torch::Tensor qW, torch::Tensor bW, int64_t N, int64_t NUM_BITS, int64_t K)
{
    TORCH_CHECK(K % 32 == 0, "K must be a multiple of 32");
    TORCH_CHECK(qW.dim() == 3 && qW.size(0) >= K && qW.size(1) >= NUM_BITS && qW.size(2) >= N,
                "qW must be at least [K, NUM_BITS, N]");
    TORCH_CHECK(bW.dim() == 3 && bW.size(0) >= K / 32 && bW.size(1) >= NUM_BITS && bW.size(2) >= N,
                "bW must be at least [K/32, NUM_BITS, N]");
    TORCH_CHECK(bW.scalar_type() == torch::kInt32, "bW must be int32");
    using namespace torch::indexing;
    const auto opt = torch::TensorOptions().dtype(torch::kInt64).device(qW.device());
    const torch::Tensor bits = torch::randint(0, 2, {K, NUM_BITS, N}, opt);           // 1 <=> +1
    qW.index_put_({Slice(0, K), Slice(0, NUM_BITS), Slice(0, N)}, (bits * 2 - 1).to(qW.scalar_type()));
    // bit t of word k/32 <=> qW[k + t] = +1; the sum wraps bit 31 into the int32 sign
    const torch::Tensor weight = torch::ones({}, opt).bitwise_left_shift(torch::arange(32, opt)).view({1, 32, 1, 1});
    const torch::Tensor words = (bits.view({K / 32, 32, NUM_BITS, N}) * weight).sum(1);
    bW.index_put_({Slice(0, K / 32), Slice(0, NUM_BITS), Slice(0, N)}, words.to(torch::kInt32).to(bW.device()));
}

void makeRandomWeight_int3(torch::Tensor weight_int3, int64_t N, int64_t K_new)
{
    TORCH_CHECK(weight_int3.dim() == 2 && weight_int3.size(0) >= K_new && weight_int3.size(1) >= N,
                "weight_int3 must be at least [K_new, N]");
    using namespace torch::indexing;
    const auto opt = torch::TensorOptions().dtype(torch::kInt64).device(weight_int3.device());
    // rand(): uniform in [0, RAND_MAX]
    weight_int3.index_put_({Slice(0, K_new), Slice(0, N)},
                           torch::randint(0, (int64_t)2147483647, {K_new, N}, opt).to(weight_int3.scalar_type()));
}

void makeRandomAlpha(torch::Tensor alpha, torch::Tensor q_bias, int64_t num_groups, int64_t NUM_BITS, int64_t N)
{
    TORCH_CHECK(alpha.dim() == 3 && alpha.size(0) >= num_groups && alpha.size(1) >= NUM_BITS && alpha.size(2) >= N,
                "alpha must be at least [num_groups, NUM_BITS, N]");
    TORCH_CHECK(q_bias.dim() == 2 && q_bias.size(0) >= num_groups && q_bias.size(1) >= N,
                "q_bias must be at least [num_groups, N]");
    using namespace torch::indexing;
    q_bias.index_put_({Slice(0, num_groups), Slice(0, N)},
                      (rand_fp32_like(q_bias, {num_groups, N}) / (double)(1 << NUM_BITS)).to(q_bias.scalar_type()));
    const auto opt = torch::TensorOptions().dtype(torch::kFloat32).device(alpha.device());
    const torch::Tensor scale = torch::exp2(-torch::arange(NUM_BITS, opt)).view({1, NUM_BITS, 1});   // 1 / 2^b
    alpha.index_put_({Slice(0, num_groups), Slice(0, NUM_BITS), Slice(0, N)},
                     (rand_fp32_like(alpha, {num_groups, NUM_BITS, N}) * scale).to(alpha.scalar_type()));
}

void makeRandomScale(torch::Tensor scale, int64_t N)
{
    TORCH_CHECK(scale.dim() == 1 && scale.size(0) >= N, "scale must hold at least N elements");
    using namespace torch::indexing;
    scale.index_put_({Slice(0, N)}, rand_fp32_like(scale, {N}).to(scale.scalar_type()));
}

void makeRandomBias(torch::Tensor bias, int64_t N) { makeRandomScale(bias, N); }

// bW int32 (any shape, kSize * mSize * nb / 32 words), A and q_bias floating point with
// at least num_groups * mSize * nb and num_groups * mSize elements -> flat device
// tensors {bWeight int32, q_bias fp16, alpha fp16} on GPU `cuda`
// (lut_gemm/lutgemm_cuda.cpp:173-223).
std::vector<torch::Tensor> parsing(torch::Tensor bW, torch::Tensor A, int64_t row, int64_t col, int64_t num_bits,
                                   bool is_row_wise_quantize, int64_t num_alpha_groups, torch::Tensor q_bias,
                                   int64_t cuda)
{
    const int64_t mSize = is_row_wise_quantize ? row : col, kSize = is_row_wise_quantize ? col : row;
    const int64_t words = kSize * mSize * num_bits / 32;
    TORCH_CHECK(bW.scalar_type() == torch::kInt32 && bW.numel() >= words, "bW must hold ", words, " int32 words");
    TORCH_CHECK(A.numel() >= num_alpha_groups * mSize * num_bits, "A must hold num_groups * mSize * nb elements");
    TORCH_CHECK(q_bias.numel() >= num_alpha_groups * mSize, "q_bias must hold num_groups * mSize elements");
    const torch::Device dev(torch::kCUDA, (c10::DeviceIndex)cuda);
    const torch::Tensor p_q_bias = q_bias.reshape({-1}).narrow(0, 0, num_alpha_groups * mSize).to(dev, torch::kHalf);
    const torch::Tensor p_alpha = A.reshape({-1}).narrow(0, 0, num_alpha_groups * mSize * num_bits).to(dev, torch::kHalf);
    const torch::Tensor bWeight = bW.reshape({-1}).narrow(0, 0, words).to(dev).contiguous();
    return {bWeight, p_q_bias.contiguous(), p_alpha.contiguous()};
}

// The compute functions as plain CPython functions of positional arguments: tensors, then whole numbers.
// (pybind11's conversions of nine arguments take 1 us, the kernel of one row of 4096 x 4096 five.)
template <auto Fn>
struct Positional;

template <typename... Args, void (*Fn)(Args...)>
struct Positional<Fn> {
    template <typename T>
    static T convert(PyObject *o, const char *name)
    {
        if constexpr (std::is_same_v<T, int64_t>) {
            const int64_t v = PyLong_AsLongLong(o);
            if (v == -1 && PyErr_Occurred()) throw python_error();
            return v;
        } else {
            TORCH_CHECK_TYPE(THPVariable_Check(o), name, ": expected a tensor, got ", Py_TYPE(o)->tp_name);
            return THPVariable_Unpack(o);
        }
    }
    template <size_t... I>
    static void spread(PyObject *const *args, const char *name, std::index_sequence<I...>)
    {
        Fn(convert<Args>(args[I], name)...);
    }
    static PyObject *call(PyObject *self, PyObject *const *args, Py_ssize_t n)
    {
        HANDLE_TH_ERRORS
        const char *name = (const char *)PyCapsule_GetPointer(self, nullptr);
        TORCH_CHECK_TYPE(n == (Py_ssize_t)sizeof...(Args), name, " takes ", sizeof...(Args), " arguments, got ", n);
        spread(args, name, std::index_sequence_for<Args...>{});
        Py_RETURN_NONE;
        END_HANDLE_TH_ERRORS
    }
    static void define(py::module_ &m, const char *name, const char *doc)
    {
        static PyMethodDef def;
        def = {name, (PyCFunction)(void (*)(void))call, METH_FASTCALL, doc};
        m.add_object(name, py::reinterpret_steal<py::object>(PyCFunction_New(&def, py::capsule((const void *)name).ptr())));
    }
};

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m)
{
    m.doc() = "MI355X (gfx950) LUT-GEMM engine behind the ShiftAddLLM `lutgemm` call signatures";
    // (name, arguments and "--" in front of a description are where help() and inspect find the signature)
    Positional<&lutgemm_compute>::define(m, "lutgemm_compute",
        "lutgemm_compute(output, bWeight, alpha, q_bias, d_input, mSize, kSize, nb, num_groups, /)\n--\n\nUniform-quant LUT-GEMV (alpha, q_bias).");
    Positional<&lutgemm_compute_shift_scale>::define(m, "lutgemm_compute_shift_scale",
        "lutgemm_compute_shift_scale(output, bWeight, alpha, d_input, mSize, kSize, nb, num_groups, /)\n--\n\nRow-wise alpha LUT-GEMV.");
    Positional<&lutgemm_compute_shift_scale_pow2>::define(m, "lutgemm_compute_shift_scale_pow2",
        "lutgemm_compute_shift_scale_pow2(output, bWeight, alpha, d_input, mSize, kSize, nb, num_groups, /)\n--\n\nRow-wise alpha LUT-GEMV, alphas promised to be powers of two.");
    Positional<&lutgemm_compute_block>::define(m, "lutgemm_compute_block",
        "lutgemm_compute_block(output, bWeight, alpha, d_input, mSize, kSize, nb, num_groups, /)\n--\n\nBlock alpha LUT-GEMV (fp16 alpha).");
    Positional<&lutgemm_compute_block_shift>::define(m, "lutgemm_compute_block_shift",
        "lutgemm_compute_block_shift(output, bWeight, alpha, d_input, mSize, kSize, nb, num_groups, num_apot, /)\n--\n\nBlock alpha LUT-GEMV (uint16 shift fields).");
    Positional<&lutgemm_compute_block_shiftInt8>::define(m, "lutgemm_compute_block_shiftInt8",
        "lutgemm_compute_block_shiftInt8(output, bWeight, alpha, d_input, mSize, kSize, nb, num_groups, num_apot, /)\n--\n\nBlock alpha LUT-GEMV (int8 exponents).");
    m.def("makeRandomInput", &makeRandomInput, "fill inp[:M, :K] with the reference's random activations");
    m.def("makeRandomAlpha", &makeRandomAlpha, "fill alpha [num_groups, NUM_BITS, N] and q_bias [num_groups, N]");
    m.def("makeRandomBias", &makeRandomBias, "fill bias[:N]");
    m.def("makeRandomScale", &makeRandomScale, "fill scale[:N]");
    m.def("makeRandomWeight_int3", &makeRandomWeight_int3, "fill weight_int3[:K_new, :N] with random words");
    m.def("makeRandomWeight", &makeRandomWeight, "fill qW [K, NUM_BITS, N] with +-1 and bW [K/32, NUM_BITS, N] with their packing");
    m.def("parsing", &parsing, "host tensors -> flat device buffers {bWeight, q_bias, alpha}");
    m.add_object("linear_forward", py::reinterpret_steal<py::object>(PyCFunction_New(&linear_forward_def, nullptr)));
    m.def("copy_bytes", &copy_bytes, "calibration copy kernel");
}
