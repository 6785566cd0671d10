"""LutLinear on bf16 and fp32 activations: the kernels that convert them themselves (one and two rows on the
look-up kernel, few rows on the matrix-core kernels) and those that only write the caller's type, against the
dense fp64 product of the activations as fp16."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from shiftaddllm_amd.lut_gemm.quant import LutLinear, encode_apot_int8
from test_gpu_tile import BLOCK_F16, BLOCK_I8, ROW, _dense, _scales

pytestmark = pytest.mark.gpu

NAMES = {ROW: "rowwise_fp16", BLOCK_F16: "block_fp16", BLOCK_I8: "apot_int8"}
CASES = [  # format, K, N, planes, rows, groups or row groups, scales
    (ROW, 32, 4, 3, 1, 1, "any"), (ROW, 4096, 4096, 4, 1, 32, "pow2"), (ROW, 8192, 28672, 3, 1, 64, "pow2"), (ROW, 8192, 28672, 3, 2, 64, "any"),
    (ROW, 1056, 260, 1, 2, 33, "any"), (ROW, 2208, 2964, 3, 7, 23, "any"), (ROW, 8192, 8192, 4, 5, 64, "pow2"), (ROW, 1024, 512, 2, 300, 8, "any"),
    (BLOCK_I8, 768, 768, 3, 1, 2, "pow2"), (BLOCK_F16, 2048, 2048, 4, 2, 8, "any"), (BLOCK_I8, 1120, 1000, 2, 20, 5, "any"),
    (BLOCK_F16, 800, 800, 3, 3, 200, "any"),                       # row groups of four outputs: converted by launches of its own
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("fmt,K,N,nb,M,groups,kind", CASES)
def test_activation_types_against_a_dense_product(gpu_device, fmt, K, N, nb, M, groups, kind, dtype):
    dev = gpu_device
    g = torch.Generator(device=dev).manual_seed(K + N + nb + M)
    lin = LutLinear(K, N, group_size=K // groups, wbit=nb, alpha_format=NAMES[fmt]).to(dev)
    lin.binaryWeight = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32)
    alpha = _scales(g, dev, groups if fmt == ROW else K // 8, nb, N if fmt == ROW else groups, kind)
    lin.alpha = encode_apot_int8(alpha) if fmt == BLOCK_I8 else alpha.half()
    lin.bias = torch.randn(N, generator=g, device=dev).half()
    x = torch.randn((M, K), generator=g, device=dev).to(dtype)
    with torch.no_grad():
        got = [lin(x) for _ in range(2)]
    assert got[0].dtype == dtype and got[0].shape == (M, N) and torch.equal(got[0], got[1])
    want = x.half().double() @ _dense(fmt, lin.binaryWeight, lin.alpha, None) + lin.bias.double()
    err = got[0].double() - want
    assert (err.norm() / want.norm()).item() <= (3e-3 if dtype == torch.bfloat16 else 3e-4)
    # a view that starts off the 16-byte grid gives the same
    off = torch.empty(M * K + 1, dtype=dtype, device=dev)[1:].view(M, K).copy_(x)
    with torch.no_grad():
        assert (lin(off).double() - want).norm().item() <= (3e-3 if dtype == torch.bfloat16 else 6e-4) * want.norm().item()


@pytest.mark.parametrize("K,N,nb,M,one_launch", [(13184, 2944, 3, 100, True), (8192, 2432, 1, 300, True), (4096, 11008, 3, 48, True),
                                                 (13824, 5120, 3, 128, False), (8192, 8192, 4, 96, False)])
def test_bf16_calls_near_the_line_between_two_kernels(gpu_device, K, N, nb, M, one_launch):
    """A conversion ahead of the GEMM kernel is part of its price: where the matrix-core kernel, which converts on the way, is
    within that, a bf16 call is one launch.  LUTGEMM_EUNSUP asks the caller to convert."""
    dev, lib, EUNSUP = gpu_device, native.cabi(), -3
    g = torch.Generator(device=dev).manual_seed(K + N + M)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32)
    alpha = _scales(g, dev, K // 128, nb, N, "pow2").half()
    x = torch.randn((M, K), generator=g, device=dev).bfloat16()
    out = torch.full((M, N), float("nan"), dtype=torch.float32, device=dev)
    def call(rows, x_type):
        layer = native.Linear(bW.data_ptr(), alpha.data_ptr(), None, rows.data_ptr(), None, out.data_ptr(), ROW, N, K, nb, K // 128, M, 0, x_type, 2)
        rc = lib.lutgemm_linear_f16(ctypes.byref(layer), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        return rc
    assert call(x, 1) == (0 if one_launch else EUNSUP)
    if not one_launch:
        assert call(x.half(), 0) == 0
    want = x.half().double() @ _dense(ROW, bW, alpha, None)
    # fp32 sums of K products: sqrt(K) roundings of 2^-24
    assert float((out.double() - want).norm() / want.norm()) <= 2.0 ** -24 * K ** 0.5
