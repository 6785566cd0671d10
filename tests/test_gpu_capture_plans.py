"""lutgemm_describe_plan's needs_workspace against the launch itself: on a stream under capture with nothing
reserved, a call is taken exactly where its plan needs no accumulator words, and with the words of the plan
reserved every call is taken and replays to the eager result."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from test_gpu_tile import BLOCK_F16, BLOCK_I8, ROW, UNIFORM

pytestmark = pytest.mark.gpu

CASES = [  # format, N, K, planes, groups or row groups, rows
    (ROW, 7716, 2304, 1, 4, 32), (UNIFORM, 7948, 2432, 1, 2, 32), (ROW, 4096, 4096, 3, 32, 1), (ROW, 768, 256, 3, 2, 1),
    (ROW, 2964, 2208, 3, 23, 7), (ROW, 28672, 1024, 2, 8, 20), (BLOCK_I8, 768, 3072, 3, 8, 40), (BLOCK_F16, 1024, 1024, 2, 64, 3),
    (UNIFORM, 512, 512, 4, 4, 1), (ROW, 16384, 512, 2, 4, 512), (BLOCK_I8, 5120, 13824, 2, 8, 512),
]


@pytest.mark.parametrize("fmt,N,K,nb,groups,M", CASES)
def test_needs_workspace_is_what_the_launch_needs(gpu_device, fmt, N, K, nb, groups, M):
    dev, lib = gpu_device, native.cabi()
    g = torch.Generator(device=dev).manual_seed(N + K + M)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32)
    if fmt == BLOCK_I8:
        alpha = torch.randint(-9, -3, (K // 8, nb, groups, 3), generator=g, device=dev).to(torch.int8)
    else:
        shape = {ROW: (groups, nb, N), UNIFORM: (groups, N), BLOCK_F16: (K // 8, nb, groups)}[fmt]
        alpha = (0.02 * (0.5 + torch.rand(shape, generator=g, device=dev))).half()
    q_bias = (alpha * 0.25) if fmt == UNIFORM else None
    x = torch.randn((M, K), generator=g, device=dev).half()
    out = torch.zeros((M, N), dtype=torch.float16, device=dev)
    ptr = lambda t: t.data_ptr() if t is not None else None
    layer = native.Linear(ptr(bW), ptr(alpha), ptr(q_bias), ptr(x), None, ptr(out), fmt, N, K, nb, groups, M, 0)
    call = lambda s: lib.lutgemm_linear_f16(ctypes.byref(layer), ctypes.c_void_p(s.cuda_stream))
    plan = native.Plan()
    assert lib.lutgemm_describe_plan(fmt, N, K, nb, groups, M, ctypes.byref(plan)) == 0
    torch.cuda.synchronize()
    lib.lutgemm_release_workspaces()          # (torch hands streams out again: what earlier calls left on them)

    s1 = torch.cuda.Stream()
    g1 = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g1, stream=s1):
        rc = call(s1)
        x.add_(0)                             # something capturable, so that the graph is not empty
    assert rc == (-6 if plan.needs_workspace else 0)

    s2 = torch.cuda.Stream()
    assert lib.lutgemm_reserve_workspace(ctypes.c_void_p(s2.cuda_stream), lib.lutgemm_workspace_words(N, M)) == 0
    g2 = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g2, stream=s2):
        assert call(s2) == 0
    s3 = torch.cuda.Stream()
    s3.wait_stream(torch.cuda.current_stream())
    assert call(s3) == 0
    torch.cuda.synchronize()
    want = out.clone()
    for _ in range(3):
        out.fill_(7.0)
        g2.replay()
        torch.cuda.synchronize()
        assert (out.double() - want.double()).norm() <= 3e-4 * want.double().norm()
