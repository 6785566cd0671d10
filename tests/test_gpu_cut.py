"""Tile heights and K-slices of the matrix-core kernel above 16 rows where they lie at the ends of their range: 16-row tiles
of many rows with a last tile of one row, 32-row tiles in many slices for few rows, or uncut; against the dense
fp64 product."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from test_gpu_tile import BLOCK_F16, BLOCK_I8, ROW, UNIFORM, _dense, _scales

pytestmark = pytest.mark.gpu

CASES = [  # format, K, N, planes, rows, groups or row groups, rows of a tile, K-slices
    (ROW, 2048, 1988, 3, 113, 16, 16, 1),        # the last tile: one row
    (ROW, 1024, 1024, 2, 256, 32, 16, 1),
    (ROW, 8192, 1024, 4, 33, 64, 16, 4),
    (BLOCK_I8, 4096, 4080, 4, 17, 5, 32, 4),     # the second 16 rows: one row
    (UNIFORM, 4096, 4096, 4, 31, 32, 32, 4),
    (BLOCK_F16, 1056, 16320, 1, 24, 8, 32, 1),   # a workgroup per CU; the last step is one word
]


@pytest.mark.parametrize("fmt,K,N,nb,M,groups,rows,slices", CASES)
def test_against_a_dense_product(gpu_device, fmt, K, N, nb, M, groups, rows, slices):
    dev, lib = gpu_device, native.cabi()
    plan = native.Plan()
    assert lib.lutgemm_describe_plan(fmt, N, K, nb, groups, M, ctypes.byref(plan)) == 0
    assert (plan.kernel, plan.rows_per_pass, plan.k_slices) == (1, rows, slices)
    g = torch.Generator(device=dev).manual_seed(K + N + nb + M)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32)
    x = torch.randn((M, K), generator=g, device=dev).half()
    q_bias = None
    if fmt == UNIFORM:
        alpha = (0.02 * (0.5 + torch.rand((groups, N), generator=g, device=dev))).half()
        q_bias = (0.005 * torch.randn((groups, N), generator=g, device=dev)).half()
    elif fmt == BLOCK_I8:
        alpha = torch.randint(-9, -3, (K // 8, nb, groups, 3), generator=g, device=dev).to(torch.int8)
    else:
        alpha = _scales(g, dev, groups if fmt == ROW else K // 8, nb, N if fmt == ROW else groups, "any").half()
    out = torch.full((M, N), float("nan"), dtype=torch.float32, device=dev)
    layer = native.Linear(bW.data_ptr(), alpha.data_ptr(), q_bias.data_ptr() if q_bias is not None else None, x.data_ptr(), None, out.data_ptr(),
                          fmt, N, K, nb, groups, M, 0, 0, 2)
    sp = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    want = x.double() @ _dense(fmt, bW, alpha, q_bias)
    for _ in range(2):      # (the accumulator words are zero again)
        assert lib.lutgemm_linear_f16(ctypes.byref(layer), sp) == 0
        torch.cuda.synchronize()
        # fp32 sums of K products (sqrt(K) roundings of 2^-24) and, between K-slices, sums in units of 2^-31
        rel = float((out.double() - want).norm() / want.norm())
        assert rel <= 2.0 ** -24 * K ** 0.5 + 2.0 ** -31 * slices * (M * N) ** 0.5 / float(want.norm()), rel
        out.fill_(float("nan"))
