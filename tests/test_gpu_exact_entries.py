"""Weights of four planes are one fp16 piece where every sum of the scales is an fp16 number, two where one may not be.  Scales
at that line, in 32-bit results: a piece left out where it was due shows as an error of 2^-12 of a weight, which every case of
such scales is checked to see.  The kernels decide for a wave's outputs together, so a matrix has the same scales throughout."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from test_exact_entries_rule import PLANES, UNIFORM_SCALES, entries, exact
from test_gpu_tile import BLOCK_F16, ROW, UNIFORM, _dense

pytestmark = pytest.mark.gpu

MATRIX_CORE, GEMM = 1, 3
SHAPES = [  # kernel, rows of a tile, M, K, N, groups (block format: row groups)
    (MATRIX_CORE, 16, 8, 512, 260, 4), (MATRIX_CORE, 32, 17, 512, 16128, 4), (GEMM, 64, 40, 512, 260, 4),
]
BLOCK_SHAPES = [
    (MATRIX_CORE, 16, 8, 512, 512, 8), (MATRIX_CORE, 32, 17, 512, 16128, 8),
    (GEMM, 64, 40, 512, 512, 8), (GEMM, 64, 40, 512, 1000, 25),      # row groups of 64 outputs, and of 40, which a wave's straddle
]


def _check(dev, fmt, scales, kernel, tile_rows, M, K, N, groups):
    lib = native.cabi()
    g = torch.Generator(device=dev).manual_seed(K + N + M)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, 4, N), generator=g, device=dev, dtype=torch.int32)
    full = lambda v, *shape: torch.full(shape, v, device=dev, dtype=torch.float32)
    if fmt == UNIFORM:
        alpha, q_bias = full(scales[0], groups, N).half(), full(scales[1], groups, N).half()
    else:
        outer, inner = (K // 8, groups) if fmt == BLOCK_F16 else (groups, N)
        alpha, q_bias = torch.stack([full(v, outer, inner) for v in scales], 1).half().contiguous(), None
    x = torch.randn((M, K), generator=g, device=dev).half()
    out = torch.empty((M, N), dtype=torch.float32, device=dev)
    ptr = lambda t: t.data_ptr() if t is not None else None
    call = native.Linear(ptr(bW), ptr(alpha), ptr(q_bias), ptr(x), None, ptr(out), fmt, N, K, 4, groups, M, 0, 0, 2)
    assert lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 33 if kernel == GEMM else 1 << 20) == 0
    try:
        plan = native.Plan()
        assert lib.lutgemm_describe_plan(fmt, N, K, 4, groups, M, ctypes.byref(plan)) == 0
        assert (plan.kernel, plan.rows_per_pass) == (kernel, tile_rows)
        rc = lib.lutgemm_linear_f16(ctypes.byref(call), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    finally:
        lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)
    assert rc == 0, lib.lutgemm_strerror(rc).decode()
    W = _dense(fmt, bW, alpha, q_bias)
    want = x.double() @ W
    # every output by itself: fp32 sums of K products (2^-24 each, K / 16 chained), weights to 2^-23 of themselves
    bound = 2e-6 * (x.double() ** 2).sum(1, keepdim=True).sqrt() * (W ** 2).sum(0, keepdim=True).sqrt() + 1e-30
    assert ((out.double() - want).abs() <= bound).all()
    if not exact(entries(scales, fmt == UNIFORM)):      # what one piece would give
        assert ((x.double() @ W.half().double() - want).abs() > 2 * bound).any()


@pytest.mark.parametrize("kernel,tile_rows,M,K,N,groups", SHAPES)
@pytest.mark.parametrize("scales", PLANES)
def test_row_scales_at_the_line(gpu_device, scales, kernel, tile_rows, M, K, N, groups):
    _check(gpu_device, ROW, scales, kernel, tile_rows, M, K, N, groups)


@pytest.mark.parametrize("kernel,tile_rows,M,K,N,row_groups", BLOCK_SHAPES)
@pytest.mark.parametrize("scales", PLANES)
def test_block_scales_at_the_line(gpu_device, scales, kernel, tile_rows, M, K, N, row_groups):
    _check(gpu_device, BLOCK_F16, scales, kernel, tile_rows, M, K, N, row_groups)


@pytest.mark.parametrize("kernel,tile_rows,M,K,N,groups", SHAPES)
@pytest.mark.parametrize("scales", UNIFORM_SCALES)
def test_uniform_scales_at_the_line(gpu_device, scales, kernel, tile_rows, M, K, N, groups):
    _check(gpu_device, UNIFORM, scales, kernel, tile_rows, M, K, N, groups)
