"""Matrix-core kernel with 32-row tiles, whose waves load whole rows of activations and turn them round in LDS: rows
that fill no tile, K that fills no step, groups shorter than a step, every format; against the dense fp64 product."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from test_gpu_tile import BLOCK_F16, BLOCK_I8, BLOCK_U16, ROW, _dense, _scales

pytestmark = pytest.mark.gpu

CASES = [  # format, K, N, planes, rows, groups or row groups, scales, type of x (LUTGEMM_TYPE_*)
    (ROW, 128, 16128, 3, 17, 1, "pow2", 0),        # one step: seven waves of a workgroup have none
    (ROW, 1056, 33024, 4, 31, 33, "any", 1),       # the last step is a word; bf16 activations
    (ROW, 2176, 8144, 2, 33, 17, "pow2", 0),      # a tile of one row; an odd number of steps
    (BLOCK_I8, 352, 33024, 3, 20, 8, "pow2", 0),   # the last step is three words
    (BLOCK_F16, 4096, 8192, 4, 32, 8, "wide", 0),
    (BLOCK_U16, 1152, 16128, 1, 24, 8, "", 1),
]


@pytest.mark.parametrize("fmt,K,N,nb,M,groups,kind,x_type", CASES)
def test_rows_of_32_row_tiles(gpu_device, fmt, K, N, nb, M, groups, kind, x_type):
    dev, lib = gpu_device, native.cabi()
    g = torch.Generator(device=dev).manual_seed(K + N + nb + M)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32)
    scale = 2.0 ** -10 if kind == "wide" else 2.0 ** -8 if fmt == BLOCK_U16 else 1.0
    x = (torch.randn((M, K), generator=g, device=dev) * scale).to((torch.float16, torch.bfloat16)[x_type])
    if fmt == BLOCK_I8:
        alpha = torch.randint(-9, -3, (K // 8, nb, groups, 3), generator=g, device=dev).to(torch.int8)
    elif fmt == BLOCK_U16:
        alpha = torch.randint(0, 512, (K // 8, nb, groups), generator=g, device=dev).to(torch.int16)
    else:
        alpha = _scales(g, dev, groups if fmt == ROW else K // 8, nb, N if fmt == ROW else groups, kind).half()
    out = torch.full((M, N), float("nan"), dtype=torch.float32, device=dev)
    layer = native.Linear(bW.data_ptr(), alpha.data_ptr(), None, x.data_ptr(), None, out.data_ptr(), fmt, N, K, nb, groups, M, 0, x_type, 2)
    assert lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 65) == 0
    try:
        plan = native.Plan()
        assert lib.lutgemm_describe_plan(fmt, N, K, nb, groups, M, ctypes.byref(plan)) == 0
        assert (plan.kernel, plan.rows_per_pass) == (1, 32)
        assert lib.lutgemm_linear_f16(ctypes.byref(layer), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    finally:
        lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)
    want = x.half().double() @ _dense(fmt, bW, alpha, None)
    # fp32 sums of K products (sqrt(K) roundings of 2^-24) and, between K-slices, sums in units of 2^-31
    rel = float((out.double() - want).norm() / want.norm())
    slack = 2.0 ** -31 / float(want.pow(2).mean().sqrt()) if plan.k_slices > 1 else 0.0
    assert rel <= 2.0 ** -24 * K ** 0.5 + slack, rel
