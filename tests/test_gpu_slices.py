"""The K-slices of the GEMM kernel depend on the sizes alone: a call gives the same bits eagerly, under capture on a
stream that holds no memory for the slices' sums, and through the entry point that allocates nothing."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from test_gpu_tile import BLOCK_F16, BLOCK_I8, ROW, UNIFORM, _scales

pytestmark = pytest.mark.gpu

CASES = [  # format, N, K, planes, groups or row groups, rows, type of the result (LUTGEMM_TYPE_*)
    (ROW, 2048, 4096, 3, 32, 100, 0), (ROW, 1540, 4128, 4, 43, 64, 2), (ROW, 512, 8192, 1, 64, 256, 1), (UNIFORM, 1024, 4096, 2, 32, 40, 0),
    (BLOCK_F16, 2000, 4096, 3, 5, 72, 2), (BLOCK_I8, 2048, 3072, 4, 8, 128, 0),
]


@pytest.mark.parametrize("fmt,N,K,nb,groups,M,out_type", CASES)
def test_same_bits_eager_captured_and_without_allocation(gpu_device, fmt, N, K, nb, groups, M, out_type):
    dev, lib = gpu_device, native.cabi()
    g = torch.Generator(device=dev).manual_seed(N + K + M)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32)
    q_bias = None
    if fmt == UNIFORM:
        alpha = (0.02 * (0.5 + torch.rand((groups, N), generator=g, device=dev))).half()
        q_bias = (0.005 * torch.randn((groups, N), generator=g, device=dev)).half()
    elif fmt == BLOCK_I8:
        alpha = torch.randint(-9, -3, (K // 8, nb, groups, 3), generator=g, device=dev).to(torch.int8)
    else:
        alpha = _scales(g, dev, groups if fmt == ROW else K // 8, nb, N if fmt == ROW else groups, "any").half()
    x = torch.randn((M, K), generator=g, device=dev).half()
    bias = torch.randn(N, generator=g, device=dev).half()
    dtype = (torch.float16, torch.bfloat16, torch.float32)[out_type]
    out = torch.empty((M, N), dtype=dtype, device=dev)
    ptr = lambda t: t.data_ptr() if t is not None else None
    layer = native.Linear(ptr(bW), ptr(alpha), ptr(q_bias), ptr(x), ptr(bias), ptr(out), fmt, N, K, nb, groups, M, 0, 0, out_type)
    sp = lambda s: ctypes.c_void_p(s.cuda_stream)
    bits = lambda t: t.clone().view(torch.int32 if out_type == 2 else torch.int16)
    torch.cuda.synchronize()
    lib.lutgemm_release_workspaces()
    assert lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 33) == 0
    try:
        plan = native.Plan()
        assert lib.lutgemm_describe_plan(fmt, N, K, nb, groups, M, ctypes.byref(plan)) == 0
        assert plan.kernel == 3 and plan.k_slices > 1
        captured_on, eager_on = torch.cuda.Stream(), torch.cuda.Stream()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=captured_on):     # (holds no memory of the library: the slices run in turn)
            assert lib.lutgemm_linear_f16(ctypes.byref(layer), sp(captured_on)) == 0
        assert lib.lutgemm_linear_f16(ctypes.byref(layer), sp(eager_on)) == 0
        torch.cuda.synchronize()
        want = bits(out)
        for _ in range(3):
            out.fill_(7.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(bits(out), want)
        if fmt == ROW and out_type == 0 and M * N <= native.NOALLOC_MAX_WORDS:
            fixed = bias.expand(M, N).contiguous()
            torch.cuda.synchronize()
            assert lib.lutgemm_gemv_rowwise_f16_noalloc(ptr(bW), ptr(alpha), ptr(x), ptr(fixed), N, K, nb, groups, M, sp(eager_on)) == 0
            torch.cuda.synchronize()
            assert torch.equal(bits(fixed), want)
    finally:
        lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)
