"""The matrix-core and GEMM kernels form weights as fp16 pieces on a power-of-two unit: scales of neighbouring
outputs, or of successive alpha groups of one output, that are far apart cost no output its precision.  Every
output by itself against the dense fp64 product, results in fp32."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from shiftaddllm_amd.lut_gemm.quant import encode_apot_int8
from test_gpu_tile import BLOCK_F16, BLOCK_I8, ROW, UNIFORM, _dense

pytestmark = pytest.mark.gpu

MFMA, TILE = 1, 3
CASES = [  # kernel, format, K, N, planes, groups or row groups
    (MFMA, ROW, 4096, 128, 1, 32), (MFMA, ROW, 4096, 128, 3, 8), (MFMA, ROW, 4096, 192, 4, 32), (MFMA, ROW, 4064, 100, 2, 127),
    (MFMA, ROW, 4064, 128, 4, 127), (MFMA, UNIFORM, 4096, 128, 3, 8), (MFMA, UNIFORM, 4064, 64, 4, 127),
    (MFMA, ROW, 1024, 128, 3, 8), (MFMA, ROW, 992, 100, 4, 31), (MFMA, UNIFORM, 992, 64, 2, 31), (MFMA, BLOCK_F16, 1024, 256, 4, 8),  # one step a wave
    (MFMA, BLOCK_F16, 4096, 256, 2, 8), (MFMA, BLOCK_I8, 4064, 128, 4, 4), (MFMA, BLOCK_I8, 4096, 256, 3, 1),
    (TILE, ROW, 1024, 320, 1, 8), (TILE, ROW, 1024, 512, 3, 8), (TILE, ROW, 992, 260, 4, 31), (TILE, UNIFORM, 1024, 256, 4, 8),
    (TILE, UNIFORM, 992, 256, 2, 31), (TILE, BLOCK_F16, 1024, 512, 3, 32), (TILE, BLOCK_I8, 992, 512, 4, 4), (TILE, BLOCK_I8, 1024, 512, 2, 16),
]


def _exponents(pattern, outer, inner, first, dev):
    """[outer, inner] binades, twenty-four apart: between the outputs (row groups), or along K (half way, between two K-steps)."""
    if pattern == "outputs":
        return (-12 + 12 * (torch.arange(inner, device=dev) % 3)).view(1, inner).expand(outer, inner)
    e = torch.where(first == (pattern != "rising"), 12, -12)
    return e.view(outer, 1).expand(outer, inner)


@pytest.mark.parametrize("scales", ["pow2", "any"])
@pytest.mark.parametrize("pattern", ["outputs", "rising", "falling", "zeros first"])
@pytest.mark.parametrize("kernel,fmt,K,N,nb,groups", CASES)
def test_every_output_keeps_its_precision(gpu_device, kernel, fmt, K, N, nb, groups, pattern, scales):
    dev, lib = gpu_device, native.cabi()
    M = 8 if kernel == MFMA else 40
    g = torch.Generator(device=dev).manual_seed(K + N + nb)
    per_column = fmt in (ROW, UNIFORM)
    outer, inner = (groups, N) if per_column else (K // 8, groups)
    planes = 1 if fmt == UNIFORM else nb
    edge = 2048 if K > 4000 else 512
    first = torch.arange(outer, device=dev) * (K // outer) < edge
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32)
    a = torch.exp2(_exponents(pattern, outer, inner, first, dev).float().view(outer, 1, inner) - torch.arange(planes, device=dev).view(1, planes, 1))
    if scales == "any":
        a = a * (1 + torch.rand(a.shape, generator=g, device=dev))
    if pattern == "zeros first":
        a = torch.where(first.view(outer, 1, 1), torch.zeros_like(a), a)
    q_bias = None
    if fmt == UNIFORM:
        alpha = a[:, 0].half()
        q_bias = (a[:, 0] * (0.25 if scales == "pow2" else 0.3)).half()
    else:
        alpha = encode_apot_int8(a) if fmt == BLOCK_I8 else a.half()
    x = torch.randn((M, K), generator=g, device=dev)
    if pattern in ("rising", "falling"):        # the inputs of the large scales are small: both halves of K count alike
        x = x * torch.where((torch.arange(K, device=dev) < edge) == (pattern == "falling"), 2.0 ** -12, 2.0 ** 12)
    x = x.half()
    out = torch.empty((M, N), device=dev)
    plan = native.Plan()
    options = {"TILE_MIN_M": 33, "MFMA_BLOCKS": 1}      # (one K-slice: sums of several meet in units of 2^-31)
    try:
        for name, value in options.items():
            assert lib.lutgemm_set_option(native.OPTIONS[name], value) == 0
        assert lib.lutgemm_describe_tile_plan(fmt, N, K, nb, groups, M, ctypes.byref(plan)) == 0
        assert plan.kernel == kernel and (kernel == TILE or plan.k_slices == 1)
        ptr = lambda t: t.data_ptr() if t is not None else None
        call = native.Linear(ptr(bW), ptr(alpha), ptr(q_bias), ptr(x), None, ptr(out), fmt, N, K, nb, groups, M, 0, 0, 2)
        rc = lib.lutgemm_linear_f16(ctypes.byref(call), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    finally:
        for name in options:
            lib.lutgemm_set_option(native.OPTIONS[name], -1)
    assert rc == 0, lib.lutgemm_strerror(rc).decode()
    torch.cuda.synchronize()
    want = x.double() @ _dense(fmt, bW, alpha, q_bias)
    rel = (out.double() - want).norm(dim=0) / want.norm(dim=0)
    # sums of K products in fp32: an error of at most K * 2^-24 of the sum of magnitudes, about its root in practice
    assert rel.max().item() <= K ** 0.5 * 2.0 ** -21, (rel.max().item(), int(rel.argmax()))
