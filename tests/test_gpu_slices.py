"""The K-slices of the GEMM kernel depend on the sizes alone: a call gives the same bits eagerly, under capture on a
stream that holds no memory for the slices' sums, and through the entry point that allocates nothing."""
import ctypes
import threading

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


@pytest.mark.parametrize("N,K,M", [(2048, 4096, 100), (5120, 13824, 512)])
def test_a_reserved_stream_allocates_nothing_for_slices(gpu_device, N, K, M):
    """lutgemm_reserve_workspace(stream, M * N): an eager call of many rows then takes no device memory."""
    dev, lib = gpu_device, native.cabi()
    bW = torch.zeros((K // 32, 2, N), dtype=torch.int32, device=dev)
    alpha = torch.full((K // 128, 2, N), 2.0 ** -6, device=dev).half()
    x = torch.ones((M, K), device=dev).half()
    out = torch.zeros((M, N), device=dev).half()
    stream = torch.cuda.Stream()
    sp = ctypes.c_void_p(stream.cuda_stream)
    torch.cuda.synchronize()
    lib.lutgemm_release_workspaces()
    assert lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 33) == 0
    try:
        plan = native.Plan()
        assert lib.lutgemm_describe_plan(ROW, N, K, 2, K // 128, M, ctypes.byref(plan)) == 0 and plan.kernel == 3 and plan.k_slices > 1
        # (the kernel's code object is loaded by a call on another stream)
        assert lib.lutgemm_gemv_rowwise_f16(bW.data_ptr(), alpha.data_ptr(), x.data_ptr(), out.data_ptr(), N, K, 2, K // 128, M, None) == 0
        torch.cuda.synchronize()
        assert lib.lutgemm_reserve_workspace(sp, lib.lutgemm_workspace_words(N, M)) == 0
        free = torch.cuda.mem_get_info()[0]
        assert lib.lutgemm_gemv_rowwise_f16(bW.data_ptr(), alpha.data_ptr(), x.data_ptr(), out.data_ptr(), N, K, 2, K // 128, M, sp) == 0
        torch.cuda.synchronize()
        assert torch.cuda.mem_get_info()[0] >= free
    finally:
        lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)
    assert torch.equal(out, torch.full_like(out, -2.0 * K * 2 * 2.0 ** -6))     # all signs -1, two planes, two calls


def test_calls_of_rising_size_keep_a_bounded_amount_of_memory(gpu_device):
    """Thirty prompts, each longer than the one before: the buffers that a stream outgrows together stay below the
    largest one, whose size is a power of two."""
    dev, lib = gpu_device, native.cabi()
    N, K, most = 2048, 4096, 512
    bW = torch.zeros((K // 32, 2, N), dtype=torch.int32, device=dev)
    alpha = torch.full((K // 128, 2, N), 2.0 ** -6, device=dev).half()
    x = torch.ones((most, K), device=dev).half()
    out = torch.zeros((most, N), device=dev).half()
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    lib.lutgemm_release_workspaces()
    assert lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 33) == 0
    call = lambda M, sp: lib.lutgemm_gemv_rowwise_f16(bW.data_ptr(), alpha.data_ptr(), x.data_ptr(), out.data_ptr(), N, K, 2, K // 128, M, sp)
    try:
        plan = native.Plan()
        assert lib.lutgemm_describe_plan(ROW, N, K, 2, K // 128, most, ctypes.byref(plan)) == 0 and plan.kernel == 3
        largest = plan.k_slices * most * N * 4
        assert call(64, None) == 0 and call(128, None) == 0             # (code objects are loaded)
        torch.cuda.synchronize()
        lib.lutgemm_release_workspaces()
        free = torch.cuda.mem_get_info()[0]
        for M in range(48, most + 1, 16):
            assert call(M, ctypes.c_void_p(stream.cuda_stream)) == 0
        torch.cuda.synchronize()
        taken = free - torch.cuda.mem_get_info()[0]
    finally:
        lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)
    power = 1 << (largest - 1).bit_length()
    assert largest <= taken <= 2 * power + (2 << 20), (largest, taken)


def test_two_host_threads_on_one_stream(gpu_device):
    """A call whose slices are added up by a second launch keeps the two together: calls of another host thread on
    the same stream share the buffer between them."""
    dev, lib = gpu_device, native.cabi()
    N, K, M = 1024, 4096, 64
    stream = torch.cuda.Stream()
    sp = ctypes.c_void_p(stream.cuda_stream)
    alpha = torch.full((K // 128, 2, N), 2.0 ** -6, device=dev).half()
    x = torch.ones((M, K), device=dev).half()
    # all signs -1 in one thread, +1 in the other
    weights = [torch.full((K // 32, 2, N), v, dtype=torch.int32, device=dev) for v in (0, -1)]
    outs = [[torch.zeros((M, N), device=dev).half() for _ in range(60)] for _ in weights]
    codes = [[], []]
    torch.cuda.synchronize()
    assert lib.lutgemm_reserve_workspace(sp, lib.lutgemm_workspace_words(N, M)) == 0
    assert lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 33) == 0
    try:
        plan = native.Plan()
        assert lib.lutgemm_describe_plan(ROW, N, K, 2, K // 128, M, ctypes.byref(plan)) == 0 and plan.kernel == 3 and plan.k_slices > 1

        def work(i):
            for out in outs[i]:        # (ctypes lets the other thread run during the call)
                codes[i].append(lib.lutgemm_gemv_rowwise_f16(weights[i].data_ptr(), alpha.data_ptr(), x.data_ptr(), out.data_ptr(), N, K, 2,
                                                             K // 128, M, sp))
        threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
    finally:
        lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)
    assert codes == [[0] * 60] * 2
    want = 2 * K * 2.0 ** -6
    assert all(bool((o == -want).all()) for o in outs[0]) and all(bool((o == want).all()) for o in outs[1])
