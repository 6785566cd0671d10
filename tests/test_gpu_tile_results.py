"""Results of the GEMM kernel for many rows at whole and partial tiles, by lone teams, two teams and K-slices, written over and
added to what the caller has there, against the dense fp64 product."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from test_gpu_tile import ROW, _dense

pytestmark = pytest.mark.gpu


SIZES = [  # K, N, M, rows of a tile, teams of a workgroup, K-slices
    (128, 300, 97, 128, 1, 1), (256, 8196, 330, 128, 1, 1), (128, 260, 64, 64, 1, 1), (1024, 2172, 700, 128, 2, 1), (2048, 516, 131, 128, 1, 16),
    (8192, 512, 60, 64, 2, 16),
]


@pytest.fixture(autouse=True)
def _gemm_kernel():
    assert native.cabi().lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 33) == 0
    yield
    native.cabi().lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)


def _layer(dev, K, N, M, tile_rows, teams, slices):
    """Weights and inputs of a call whose plan is as stated, its result in 64 bits and the size that fp32 sums round on."""
    plan = native.Plan()
    assert native.cabi().lutgemm_describe_plan(ROW, N, K, 3, K // 128, M, ctypes.byref(plan)) == 0
    assert (plan.kernel, plan.rows_per_pass, plan.ranges, plan.k_slices) == (3, tile_rows, teams, slices)
    g = torch.Generator(device=dev).manual_seed(K + N + M)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, 3, N), generator=g, device=dev, dtype=torch.int32)
    alpha = torch.exp2(torch.randint(-8, -5, (K // 128, 3, N), generator=g, device=dev).float()).half()
    x = torch.randn((M, K), generator=g, device=dev).half()
    size = (x.double() ** 2).sum(1, keepdim=True).sqrt() * alpha.double().abs().sum(1).max() * K ** 0.5
    return g, bW, alpha, x, x.double() @ _dense(ROW, bW, alpha, None), 2.0 ** -20 * size


@pytest.mark.parametrize("K,N,M,tile_rows,teams,slices", SIZES)
@pytest.mark.parametrize("out_type", [0, 1, 2])
@pytest.mark.parametrize("with_bias", [False, True])
def test_results_of_partial_tiles(gpu_device, K, N, M, tile_rows, teams, slices, out_type, with_bias):
    """Whole tiles and remainders of rows and outputs, by lone teams, two teams and slices, in every type of results."""
    dev, lib = gpu_device, native.cabi()
    g, bW, alpha, x, want, sums = _layer(dev, K, N, M, tile_rows, teams, slices)
    bias = torch.randn(N, generator=g, device=dev).half() if with_bias else None
    room = torch.full((M + 2, N), 7.0, dtype=(torch.float16, torch.bfloat16, torch.float32)[out_type], device=dev)
    out = room[1:-1]
    call = native.Linear(bW.data_ptr(), alpha.data_ptr(), None, x.data_ptr(), bias.data_ptr() if with_bias else None, out.data_ptr(), ROW, N, K, 3,
                         K // 128, M, 0, 0, out_type)
    rc = lib.lutgemm_linear_f16(ctypes.byref(call), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, lib.lutgemm_strerror(rc).decode()
    want = want + (bias.double() if with_bias else 0.0)
    assert (room[0] == 7.0).all() and (room[-1] == 7.0).all()      # the rows around the result
    ulp = (2.0 ** -11, 2.0 ** -8, 2.0 ** -24)[out_type]            # the rounding of the result, and fp32 sums
    assert ((out.double() - want).abs() <= ulp * want.abs() + sums).all()


@pytest.mark.parametrize("K,N,M,tile_rows,teams,slices", SIZES)
def test_results_added_to_the_callers_outputs(gpu_device, K, N, M, tile_rows, teams, slices):
    """The accumulating entry points read each output before they write it: another value everywhere, twice over, and through the one
    that takes slices in turn."""
    dev, lib = gpu_device, native.cabi()
    g, bW, alpha, x, product, sums = _layer(dev, K, N, M, tile_rows, teams, slices)
    room = torch.randn((M + 2, N), generator=g, device=dev).half()
    before, out = room.clone(), room[1:-1]
    calls = [lib.lutgemm_gemv_rowwise_f16] * 2 + [lib.lutgemm_gemv_rowwise_f16_noalloc] * (M * N <= native.NOALLOC_MAX_WORDS)
    for call in calls:
        want = out.double() + product
        rc = call(bW.data_ptr(), alpha.data_ptr(), x.data_ptr(), out.data_ptr(), N, K, 3, K // 128, M,
                  ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, lib.lutgemm_strerror(rc).decode()
        assert ((out.double() - want).abs() <= 2.0 ** -11 * want.abs() + sums).all()
    assert torch.equal(room[0], before[0]) and torch.equal(room[-1], before[-1])
