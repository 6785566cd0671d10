"""Infinities, NaN and sums beyond the 65536 of an accumulator word in the matrix-core and GEMM kernels."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from test_gpu_tile import BLOCK_F16, ROW, UNIFORM, _scales

pytestmark = pytest.mark.gpu

MFMA, TILE = 1, 3
F16, BF16, F32 = range(3)


def _call(kernel, fmt, bW, alpha, q_bias, x, groups, out_type=F16, blocks=-1):
    """(result, plan) of one linear call on the kernel named."""
    lib = native.cabi()
    KW, nb, N = bW.shape
    M, K = x.shape
    out = torch.empty((M, N), dtype=(torch.float16, torch.bfloat16, torch.float32)[out_type], device=x.device)
    options = {"TILE_MIN_M": 33, "MFMA_BLOCKS": blocks}
    plan = native.Plan()
    ptr = lambda t: t.data_ptr() if t is not None else None
    call = native.Linear(ptr(bW), ptr(alpha), ptr(q_bias), ptr(x), None, ptr(out), fmt, N, K, nb, groups, M, 0, 0, out_type)
    try:
        for name, value in options.items():
            assert lib.lutgemm_set_option(native.OPTIONS[name], value) == 0
        assert lib.lutgemm_describe_plan(fmt, N, K, nb, groups, M, ctypes.byref(plan)) == 0 and plan.kernel == kernel
        rc = lib.lutgemm_linear_f16(ctypes.byref(call), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    finally:
        for name in options:
            lib.lutgemm_set_option(native.OPTIONS[name], -1)
    assert rc == 0, lib.lutgemm_strerror(rc).decode()
    torch.cuda.synchronize()
    return out, plan


def _problem(fmt, K, N, nb, groups, M, kind, dev):
    g = torch.Generator(device=dev).manual_seed(K + N + nb)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32)
    q_bias = None
    if fmt == UNIFORM:
        alpha = (0.02 * (0.5 + torch.rand((groups, N), generator=g, device=dev))).half()
        q_bias = (0.005 * torch.randn((groups, N), generator=g, device=dev)).half()
    else:
        alpha = _scales(g, dev, groups if fmt == ROW else K // 8, nb, N if fmt == ROW else groups, kind).half()
    return bW, alpha, q_bias, torch.randn((M, K), generator=g, device=dev).half()


@pytest.mark.parametrize("out_type", [F16, F32])
@pytest.mark.parametrize("fmt,K,N,nb,groups,kind", [(ROW, 1024, 256, 3, 8, "pow2"), (ROW, 992, 260, 4, 31, "any"), (ROW, 1024, 64, 1, 8, "pow2"),
                                                    (UNIFORM, 1024, 256, 2, 8, ""), (BLOCK_F16, 1120, 512, 3, 8, "any")])
@pytest.mark.parametrize("kernel,M", [(MFMA, 7), (TILE, 45)])
def test_special_activations_stay_in_their_rows(gpu_device, kernel, M, fmt, K, N, nb, groups, kind, out_type):
    bW, alpha, q_bias, x = _problem(fmt, K, N, nb, groups, M, kind, gpu_device)
    clean, _ = _call(kernel, fmt, bW, alpha, q_bias, x, groups, out_type)
    special = {1: (float("nan"), 5), 3: (float("inf"), K - 1), 4: (-float("inf"), K // 2), M - 1: (float("nan"), K - 1)}
    for row, (value, k) in special.items():
        x[row, k] = value
    got, _ = _call(kernel, fmt, bW, alpha, q_bias, x, groups, out_type)
    for row in range(M):
        if row not in special:
            assert torch.equal(got[row], clean[row]), row
        elif special[row][0] != special[row][0]:
            assert torch.isnan(got[row]).all(), row
        else:       # an infinity where its weights are exact, NaN where they are zero or have a second piece
            assert not torch.isfinite(got[row]).any(), row


@pytest.mark.parametrize("kernel,M,fmt,K,N,nb,groups,kind", [
    # 32-row tiles, whose activations pass through LDS; K that fills no step; K-slices
    (MFMA, 31, ROW, 1056, 33024, 4, 33, "any"), (MFMA, 32, BLOCK_F16, 4096, 8192, 4, 8, "any"), (MFMA, 20, ROW, 8192, 6144, 2, 64, "pow2"),
    # two teams of waves per workgroup, of which one holds the value; several slices
    (TILE, 129, ROW, 896, 20480, 3, 7, "pow2"), (TILE, 207, ROW, 9312, 256, 3, 97, "any"), (TILE, 39, BLOCK_F16, 7712, 940, 2, 5, "any"),
    (TILE, 207, UNIFORM, 9312, 256, 2, 97, ""),
])
def test_special_activations_in_tall_tiles_and_teams(gpu_device, kernel, M, fmt, K, N, nb, groups, kind):
    bW, alpha, q_bias, x = _problem(fmt, K, N, nb, groups, M, kind, gpu_device)
    clean, plan = _call(kernel, fmt, bW, alpha, q_bias, x, groups, F32)
    assert (plan.rows_per_pass == 32) if kernel == MFMA else plan.ranges == 2
    special = {1: (float("nan"), 5), 3: (float("inf"), K - 1), 4: (-float("inf"), K // 2), 17: (float("inf"), K - 9), M - 1: (float("nan"), K - 1)}
    for row, (value, k) in special.items():
        x[row, k] = value
    got, _ = _call(kernel, fmt, bW, alpha, q_bias, x, groups, F32)
    for row in range(M):
        if row not in special:
            assert torch.equal(got[row], clean[row]), row
        elif special[row][0] != special[row][0]:
            assert torch.isnan(got[row]).all(), row
        else:
            assert not torch.isfinite(got[row]).any(), row


@pytest.mark.parametrize("special", [float("inf"), float("nan")])
@pytest.mark.parametrize("fmt,groups", [(ROW, 8), (UNIFORM, 8), (BLOCK_F16, 8)])
@pytest.mark.parametrize("kernel,M", [(MFMA, 7), (TILE, 45)])
def test_special_scales_stay_in_their_outputs(gpu_device, kernel, M, fmt, groups, special):
    K, N, nb = 1024, 512, 3
    bW, alpha, q_bias, x = _problem(fmt, K, N, nb, groups, M, "any", gpu_device)
    clean, _ = _call(kernel, fmt, bW, alpha, q_bias, x, groups)
    flat = alpha.view(alpha.shape[0], -1, alpha.shape[-1])
    flat[3, 0, 5] = special                                 # output 5, or the sixth row group
    got, _ = _call(kernel, fmt, bW, alpha, q_bias, x, groups)
    hit = torch.zeros(N, dtype=torch.bool, device=gpu_device)
    if fmt == BLOCK_F16:
        hit[5 * (N // groups):6 * (N // groups)] = True
    else:
        hit[5] = True
    assert not torch.isfinite(got[:, hit]).any()
    assert torch.equal(got[:, ~hit], clean[:, ~hit])


def test_sums_beyond_the_accumulator_word(gpu_device):
    """fp32 results: a partial sum beyond 65536 counts as infinite where K-slices meet in accumulator words, and is
    carried in fp32 in a single slice and in the GEMM kernel.  fp16 results are infinite either way."""
    dev = gpu_device
    N, K, nb, groups = 256, 4096, 2, 32
    bW = torch.full((K // 32, nb, N), -1, dtype=torch.int32, device=dev)
    bW[:, :, ::2] = 0                                       # every other output negative
    alpha = torch.full((groups, nb, N), 16.0, device=dev).half()
    sign = torch.where(torch.arange(N, device=dev) % 2 == 0, -1.0, 1.0)
    for kernel, M, blocks, finite in ((MFMA, 7, 1 << 20, False), (MFMA, 7, 1, True), (TILE, 45, -1, True)):
        x = torch.full((M, K), 32.0, device=dev).half()
        got, plan = _call(kernel, ROW, bW, alpha, None, x, groups, F32, blocks)
        assert kernel == TILE or (plan.k_slices == 1) == finite
        want = sign * (2 * 16.0 * 32.0 * K if finite else float("inf"))
        assert torch.equal(got, want.expand(M, N))
        got, _ = _call(kernel, ROW, bW, alpha, None, x, groups, F16, blocks)
        assert torch.equal(got.float(), (sign * float("inf")).expand(M, N))
