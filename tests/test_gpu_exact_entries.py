"""Weights of four planes are one fp16 piece where every sum of the scales is an fp16 number, two where one may not be.  Scales
at that line, in 32-bit results: a piece left out where it was due would show as an error of 2^-12 of a weight."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from test_gpu_tile import BLOCK_F16, ROW, UNIFORM, _dense

pytestmark = pytest.mark.gpu

PLANES = [  # scales of the four planes
    (1024, 512, 256, 255), (1025, 513, 257, 253), (1025, 513, 257, 255), (1024, 512, 256, 257), (2046, 1, 1, 1), (2047, 1, 1, 2),
    (1, 2, 4, 2040), (0, 0, 3, 0), (0, 0, 0, 0), (5, 0, 1023, 0), (1.5, 0.75, 0.375, 1.125), (1 + 2 ** -10, 1, 2, 4), (4, 2, 1, 2 ** -9), (4, 2, 1, 2 ** -8),
    (2.0 ** -24, 2.0 ** -23, 3 * 2.0 ** -24, 0), (-1024, 511, -256, 255),
]


@pytest.mark.parametrize("M", [17, 40])      # 32-row tiles of the matrix-core kernel, the GEMM kernel
@pytest.mark.parametrize("fmt,K,N,groups", [(ROW, 512, 260, 4), (ROW, 96, 64, 3), (BLOCK_F16, 512, 512, 8), (UNIFORM, 512, 260, 4)])
def test_scales_at_the_line(gpu_device, fmt, K, N, groups, M):
    dev, lib = gpu_device, native.cabi()
    g = torch.Generator(device=dev).manual_seed(K + N + M)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, 4, N), generator=g, device=dev, dtype=torch.int32)
    outer, inner = (K // 8, groups) if fmt == BLOCK_F16 else (groups, N)
    pick = torch.randint(0, len(PLANES), (outer, inner), generator=g, device=dev)
    a = torch.tensor(PLANES, device=dev, dtype=torch.float32)[pick].permute(0, 2, 1).contiguous()
    q_bias = a[:, 1].half().contiguous() if fmt == UNIFORM else None
    alpha = (a[:, 0] if fmt == UNIFORM else a).half().contiguous()
    x = torch.randn((M, K), generator=g, device=dev).half()
    out = torch.empty((M, N), dtype=torch.float32, device=dev)
    ptr = lambda t: t.data_ptr() if t is not None else None
    call = native.Linear(bW.data_ptr(), alpha.data_ptr(), ptr(q_bias), x.data_ptr(), None, out.data_ptr(), fmt, N, K, 4, groups, M, 0, 0, 2)
    assert lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 33) == 0
    try:
        rc = lib.lutgemm_linear_f16(ctypes.byref(call), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    finally:
        lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)
    assert rc == 0, lib.lutgemm_strerror(rc).decode()
    W = _dense(fmt, bW, alpha, q_bias)
    want = x.double() @ W
    # every output by itself: fp32 sums of K products (2^-24 each, K / 16 chained), weights to 2^-23 of themselves
    size = (x.double() ** 2).sum(1, keepdim=True).sqrt() * (W ** 2).sum(0, keepdim=True).sqrt()
    assert ((out.double() - want).abs() <= 2e-6 * size + 1e-30).all()
