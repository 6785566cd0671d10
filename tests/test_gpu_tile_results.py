"""Results of the GEMM kernel for many rows at whole and partial tiles, against the dense fp64 product."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from test_gpu_tile import ROW, _dense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,N,M", [(128, 300, 97), (256, 8196, 330), (1024, 2172, 700), (2048, 516, 131)])
@pytest.mark.parametrize("out_type", [0, 1, 2])
@pytest.mark.parametrize("with_bias", [False, True])
def test_results_of_partial_tiles(gpu_device, K, N, M, out_type, with_bias):
    """Whole tiles and remainders of rows and outputs, by lone teams, two teams and slices, in every type of results."""
    dev, lib = gpu_device, native.cabi()
    g = torch.Generator(device=dev).manual_seed(K + N + M)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, 3, N), generator=g, device=dev, dtype=torch.int32)
    alpha = torch.exp2(torch.randint(-8, -5, (K // 128, 3, N), generator=g, device=dev).float()).half()
    x = torch.randn((M, K), generator=g, device=dev).half()
    bias = torch.randn(N, generator=g, device=dev).half() if with_bias else None
    room = torch.full((M + 2, N), 7.0, dtype=(torch.float16, torch.bfloat16, torch.float32)[out_type], device=dev)
    out = room[1:-1]
    call = native.Linear(bW.data_ptr(), alpha.data_ptr(), None, x.data_ptr(), bias.data_ptr() if with_bias else None, out.data_ptr(), ROW, N, K, 3,
                         K // 128, M, 0, 0, out_type)
    assert lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 33) == 0
    try:
        rc = lib.lutgemm_linear_f16(ctypes.byref(call), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    finally:
        lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)
    assert rc == 0, lib.lutgemm_strerror(rc).decode()
    want = x.double() @ _dense(ROW, bW, alpha, None) + (bias.double() if with_bias else 0.0)
    assert (room[0] == 7.0).all() and (room[-1] == 7.0).all()      # the rows around the result
    ulp = (2.0 ** -11, 2.0 ** -8, 2.0 ** -24)[out_type]            # the rounding of the result, and fp32 sums
    size = (x.double() ** 2).sum(1, keepdim=True).sqrt() * alpha.double().abs().sum(1).max() * K ** 0.5
    assert ((out.double() - want).abs() <= ulp * want.abs() + 2.0 ** -20 * size).all()
