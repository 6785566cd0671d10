"""The matrix-core kernel on the problems it takes beside whole 128-input row-wise groups: every alpha format,
alpha groups of any length, any K and N, against the dense fp64 product (helpers of the GEMM kernel's test)."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from shiftaddllm_amd.lut_gemm.quant import encode_apot_int8
from test_gpu_tile import BLOCK_F16, BLOCK_I8, BLOCK_U16, ROW, UNIFORM, _dense, _scales

pytestmark = pytest.mark.gpu

CASES = [  # format, K, N, planes, rows, groups (row-wise, uniform) or row groups (block), scales
    (ROW, 32, 4, 3, 5, 1, "pow2"), (ROW, 96, 100, 1, 3, 3, "any"), (ROW, 2208, 2964, 3, 7, 23, "any"), (ROW, 1056, 512, 4, 17, 33, "wide"),
    (ROW, 4096, 4096, 3, 2, 128, "pow2"), (ROW, 1024, 260, 2, 40, 16, "any"), (ROW, 2048, 256, 4, 8, 16, "wide"),
    (UNIFORM, 288, 100, 1, 3, 9, ""), (UNIFORM, 512, 512, 2, 16, 4, ""), (UNIFORM, 768, 768, 3, 2, 6, ""), (UNIFORM, 1024, 256, 4, 33, 8, ""),
    (BLOCK_F16, 32, 24, 4, 5, 1, "any"), (BLOCK_F16, 1120, 1000, 2, 17, 25, "pow2"), (BLOCK_F16, 2048, 512, 4, 20, 8, "wide"),
    (BLOCK_U16, 512, 768, 3, 4, 8, ""), (BLOCK_U16, 96, 24, 1, 3, 1, ""),
    (BLOCK_I8, 768, 768, 3, 1, 8, "any"), (BLOCK_I8, 96, 5504, 3, 5, 4, "pow2"), (BLOCK_I8, 2048, 512, 3, 4, 8, "wide"),
    (BLOCK_I8, 1024, 1024, 2, 48, 16, "any"),
]


@pytest.mark.parametrize("fmt,K,N,nb,M,groups,kind", CASES)
def test_few_rows_against_a_dense_product(gpu_device, fmt, K, N, nb, M, groups, kind):
    dev, lib = gpu_device, native.cabi()
    g = torch.Generator(device=dev).manual_seed(K + N + nb + M)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32)
    x = torch.randn((M, K), generator=g, device=dev) * (2.0 ** -10 if kind == "wide" else 2.0 ** -8 if fmt == BLOCK_U16 else 1.0)
    q_bias = None
    if fmt == UNIFORM:
        alpha = (0.02 * (0.5 + torch.rand((groups, N), generator=g, device=dev))).half()
        q_bias = (0.005 * torch.randn((groups, N), generator=g, device=dev)).half()
    elif fmt == BLOCK_U16:
        alpha = torch.randint(0, 512, (K // 8, nb, groups), generator=g, device=dev).to(torch.int16)
    elif fmt == ROW:
        alpha = _scales(g, dev, groups, nb, N, kind).half()
    else:
        alpha = _scales(g, dev, K // 8, nb, groups, kind)
        alpha = alpha.half() if fmt == BLOCK_F16 else encode_apot_int8(alpha)
    x = x.half()
    bias = torch.randn(N, generator=g, device=dev).half()
    plan = native.Plan()
    assert lib.lutgemm_describe_tile_plan(fmt, N, K, nb, groups, M, ctypes.byref(plan)) == 0 and plan.kernel == 1
    out = torch.full((M, N), 7.0, dtype=torch.float16, device=dev)       # overwritten
    ptr = lambda t: t.data_ptr() if t is not None else None
    call = native.Linear(ptr(bW), ptr(alpha), ptr(q_bias), ptr(x), ptr(bias), ptr(out), fmt, N, K, nb, groups, M, 0)
    for _ in range(2):                                                    # twice: the accumulator words are left at zero
        rc = lib.lutgemm_linear_f16(ctypes.byref(call), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, lib.lutgemm_strerror(rc).decode()
    torch.cuda.synchronize()
    want = x.double() @ _dense(fmt, bW, alpha, q_bias) + bias.double()
    ok = want.abs() < 60000
    err = (out.double() - want)[ok]
    assert (err.norm() / want[ok].norm()).item() <= 3e-4 and (err.abs().max() / want[ok].abs().max()).item() <= 1e-3
