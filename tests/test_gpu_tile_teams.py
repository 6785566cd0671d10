"""GEMM kernel with two teams of waves per workgroup, each on half of a slice's steps: halves of unequal length, a slice of
two steps, which leaves the second team none, K that fills no step, tiles of 64 and 128 rows; against the dense fp64
product and, where there are several slices, bit for bit against the kernel that takes halves and slices in turn (a capture
on a stream that holds no memory; calls of one slice are captured as they are)."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from test_gpu_tile import BLOCK_F16, BLOCK_I8, ROW, UNIFORM, _dense, _scales

pytestmark = pytest.mark.gpu

# format, K, N, planes, rows, groups or row groups, scales, K-slices (steps of 64 inputs, rounded up to an even number)
CASES = [   # sizes that are cut for teams
    (ROW, 896, 20480, 3, 129, 7, "pow2", 1),        # 14 steps: halves of 8 and 6; rows one beyond a tile
    (ROW, 1568, 20480, 2, 150, 49, "any", 1),       # 49 words: the last step is half empty
    (BLOCK_F16, 1152, 20480, 4, 200, 5, "wide", 1), # another unit on the way, in either team; tiles straddling row groups
    (UNIFORM, 896, 20476, 3, 129, 7, "", 1),        # N off the tile
    (BLOCK_I8, 8192, 2560, 2, 256, 8, "pow2", 11),  # 12 steps a slice, the last one shorter
    (ROW, 8224, 8192, 4, 64, 257, "any", 7),        # 64-row tiles
    (ROW, 9312, 256, 3, 207, 97, "any", 13),        # 12 steps a slice, the last one two
    (UNIFORM, 9312, 256, 3, 207, 97, "", 13),
    (BLOCK_F16, 10080, 1160, 4, 197, 5, "wide", 14),  # as above; row groups of 232 outputs, in two of which some waves' 64 lie
    (UNIFORM, 4096, 4100, 2, 500, 32, "", 3),       # N off the tile
    (BLOCK_F16, 4096, 4000, 3, 500, 5, "any", 4),
    (BLOCK_I8, 7712, 940, 2, 39, 5, "pow2", 16),    # 64-row tiles
]


@pytest.fixture(autouse=True)
def _gemm_kernel():
    assert native.cabi().lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 33) == 0
    yield
    native.cabi().lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)


@pytest.mark.parametrize("fmt,K,N,nb,M,groups,kind,slices", CASES)
def test_teams_against_a_dense_product_and_in_turn(gpu_device, fmt, K, N, nb, M, groups, kind, slices):
    dev, lib = gpu_device, native.cabi()
    g = torch.Generator(device=dev).manual_seed(K + N + nb + M)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32)
    x = (torch.randn((M, K), generator=g, device=dev) * (2.0 ** -10 if kind == "wide" else 1.0)).half()
    q_bias = None
    if fmt == UNIFORM:
        alpha = (0.02 * (0.5 + torch.rand((groups, N), generator=g, device=dev))).half()
        q_bias = (0.005 * torch.randn((groups, N), generator=g, device=dev)).half()
    elif fmt == BLOCK_I8:
        alpha = torch.randint(-9, -3, (K // 8, nb, groups, 3), generator=g, device=dev).to(torch.int8)
    else:
        alpha = _scales(g, dev, groups if fmt == ROW else K // 8, nb, N if fmt == ROW else groups, kind).half()
    plan = native.Plan()
    assert lib.lutgemm_describe_plan(fmt, N, K, nb, groups, M, ctypes.byref(plan)) == 0
    assert (plan.kernel, plan.k_slices, plan.ranges) == (3, slices, 2), (plan.kernel, plan.k_slices, plan.ranges, plan.units_per_slice, plan.k_units)
    out = torch.empty((M, N), dtype=torch.float32, device=dev)
    ptr = lambda t: t.data_ptr() if t is not None else None
    layer = native.Linear(ptr(bW), ptr(alpha), ptr(q_bias), ptr(x), None, ptr(out), fmt, N, K, nb, groups, M, 0, 0, 2)
    want = x.double() @ _dense(fmt, bW, alpha, q_bias)
    torch.cuda.synchronize()
    lib.lutgemm_release_workspaces()
    eager, captured_on = torch.cuda.Stream(), torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=captured_on):
        assert lib.lutgemm_linear_f16(ctypes.byref(layer), ctypes.c_void_p(captured_on.cuda_stream)) == 0
    assert lib.lutgemm_linear_f16(ctypes.byref(layer), ctypes.c_void_p(eager.cuda_stream)) == 0
    torch.cuda.synchronize()
    got = out.clone()
    # fp32 sums of K products of exact weights: a rounding of 2^-24 of the running sum each, which grows like the square
    # root of its length, so sqrt(K) / 2 of them on the scale of the result at most
    rel = float((got.double() - want).norm() / want.norm())
    assert rel <= 2.0 ** -24 * K ** 0.5, rel
    for _ in range(2):
        out.fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int32), got.view(torch.int32))
