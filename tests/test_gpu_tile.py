"""The GEMM kernel for many activation rows (every alpha format) against the dense fp64 product of the
dequantised matrix, formed on the GPU by framework operations."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from shiftaddllm_amd.lut_gemm.quant import decode_apot_int8, encode_apot_int8

pytestmark = pytest.mark.gpu
ROW, BLOCK_F16, BLOCK_U16, BLOCK_I8, UNIFORM = range(5)


def _dense(fmt, bW, alpha, q_bias):
    """W_q [K, N] fp64."""
    KW, nb, N = bW.shape
    K = 32 * KW
    signs = ((bW.unsqueeze(1) >> torch.arange(32, device=bW.device).view(1, 32, 1, 1)) & 1).double() * 2 - 1
    signs = signs.reshape(K, nb, N)
    if fmt == UNIFORM:
        c = torch.exp2(-1.0 - torch.arange(nb, device=bW.device)).double().view(1, nb, 1)
        rep = K // alpha.shape[0]
        return (signs * c).sum(1) * alpha.double().repeat_interleave(rep, 0) + q_bias.double().repeat_interleave(rep, 0)
    if fmt == ROW:
        return (signs * alpha.double().repeat_interleave(K // alpha.shape[0], 0)).sum(1)
    if fmt == BLOCK_U16:
        u = alpha.int() & 0xffff
        alpha = (1 << (u & 7)) + (1 << ((u >> 3) & 7)) + (1 << ((u >> 6) & 7))
    elif fmt == BLOCK_I8:
        alpha = decode_apot_int8(alpha)
    return (signs * alpha.double().repeat_interleave(8, 0).repeat_interleave(N // alpha.shape[2], 2)).sum(1)


def _scales(g, dev, outer, nb, inner, kind):
    a = torch.exp2(torch.randint(-8, -5, (outer, 1, inner), generator=g, device=dev).float()
                   - torch.arange(nb, device=dev).view(1, nb, 1))
    if kind == "any":
        a = a * (1 + torch.rand((outer, nb, inner), generator=g, device=dev))
    if kind == "wide":      # over twenty binades: the kernel changes its unit on the way along K
        a = a * torch.exp2(torch.randint(-6, 14, (outer, nb, inner), generator=g, device=dev).float())
    return a


CASES = [  # format, K, N, planes, rows, groups (row-wise, uniform) or row groups (block), scales, bias
    (ROW, 256, 256, 1, 33, 2, "pow2", False), (ROW, 512, 256, 2, 64, 4, "any", True), (ROW, 2048, 512, 3, 65, 16, "pow2", True),
    (ROW, 512, 260, 4, 129, 8, "any", False), (ROW, 32, 4, 3, 300, 1, "pow2", False), (ROW, 96, 64, 4, 40, 3, "any", True),
    (ROW, 2208, 2964, 3, 77, 23, "any", True), (ROW, 4096, 512, 4, 128, 32, "wide", False),
    (UNIFORM, 512, 512, 1, 70, 4, "", False), (UNIFORM, 512, 500, 2, 33, 16, "", True), (UNIFORM, 544, 512, 3, 130, 1, "", False),
    (UNIFORM, 1024, 256, 4, 128, 8, "", False),
    (BLOCK_F16, 512, 1000, 2, 100, 1, "any", True), (BLOCK_F16, 512, 1000, 3, 40, 250, "pow2", False),
    (BLOCK_F16, 2048, 512, 4, 128, 8, "wide", False), (BLOCK_U16, 512, 768, 3, 40, 8, "", False),
    (BLOCK_U16, 96, 24, 1, 200, 2, "", False), (BLOCK_I8, 1024, 1024, 3, 65, 8, "any", True),
    (BLOCK_I8, 32, 4, 4, 33, 1, "any", False), (BLOCK_I8, 3072, 768, 3, 128, 8, "pow2", True), (BLOCK_I8, 736, 1380, 2, 150, 5, "pow2", False),
]


@pytest.mark.parametrize("fmt,K,N,nb,M,groups,kind,with_bias", CASES)
def test_many_rows_against_a_dense_product(gpu_device, fmt, K, N, nb, M, groups, kind, with_bias):
    dev, lib = gpu_device, native.cabi()
    g = torch.Generator(device=dev).manual_seed(K + N + nb + M)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32)
    x = torch.randn((M, K), generator=g, device=dev) * (2.0 ** -10 if kind == "wide" else 2.0 ** -8 if fmt == BLOCK_U16 else 1.0)
    q_bias = None
    if fmt == UNIFORM:
        alpha = (0.02 * (0.5 + torch.rand((groups, N), generator=g, device=dev))).half()
        q_bias = (0.005 * torch.randn((groups, N), generator=g, device=dev)).half()
    elif fmt == BLOCK_U16:
        alpha = torch.randint(0, 512, (K // 8, nb, groups), generator=g, device=dev).to(torch.int16)
    elif fmt == ROW:
        alpha = _scales(g, dev, groups, nb, N, kind).half()
    else:
        alpha = _scales(g, dev, K // 8, nb, groups, kind)
        alpha = alpha.half() if fmt == BLOCK_F16 else encode_apot_int8(alpha)
    x = x.half()
    bias = torch.randn(N, generator=g, device=dev).half() if with_bias else None
    plan = native.Plan()
    assert lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 33) == 0
    assert lib.lutgemm_describe_tile_plan(fmt, N, K, nb, groups, M, ctypes.byref(plan)) == 0 and plan.kernel == 3
    assert (plan.k_slices - 1) * plan.units_per_slice < plan.k_units <= plan.k_slices * plan.units_per_slice
    out = torch.full((M, N), 7.0, dtype=torch.float16, device=dev)       # overwritten
    ptr = lambda t: t.data_ptr() if t is not None else None
    call = native.Linear(ptr(bW), ptr(alpha), ptr(q_bias), ptr(x), ptr(bias), ptr(out), fmt, N, K, nb, groups, M, 0)
    try:
        rc = lib.lutgemm_linear_f16(ctypes.byref(call), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    finally:
        lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)
    assert rc == 0, lib.lutgemm_strerror(rc).decode()
    torch.cuda.synchronize()
    want = x.double() @ _dense(fmt, bW, alpha, q_bias)
    if with_bias:
        want = want + bias.double()
    ok = want.abs() < 60000
    err = (out.double() - want)[ok]
    assert (err.norm() / want[ok].norm()).item() <= 3e-4 and (err.abs().max() / want[ok].abs().max()).item() <= 1e-3


@pytest.mark.parametrize("K,N,M,out_type", [(512, 260, 130, 0), (8192, 512, 64, 0), (8192, 516, 40, 1), (256, 260, 64, 2)])
def test_bias_that_begins_on_any_value(gpu_device, K, N, M, out_type):
    """A bias is aligned to its values only, in the kernel itself and where the slices' sums are added up."""
    dev, lib = gpu_device, native.cabi()
    g = torch.Generator(device=dev).manual_seed(K + N)
    bW = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, 2, N), generator=g, device=dev, dtype=torch.int32)
    alpha = _scales(g, dev, K // 128, 2, N, "any").half()
    x = torch.randn((M, K), generator=g, device=dev).half()
    room = torch.randn(N + 4, generator=g, device=dev).half()
    got = []
    assert lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 33) == 0
    try:
        for first in range(4):
            bias = room[first:first + N]
            out = torch.empty((M, N), dtype=(torch.float16, torch.bfloat16, torch.float32)[out_type], device=dev)
            call = native.Linear(bW.data_ptr(), alpha.data_ptr(), None, x.data_ptr(), bias.data_ptr(), out.data_ptr(), ROW, N, K, 2,
                                 K // 128, M, 0, 0, out_type)
            rc = lib.lutgemm_linear_f16(ctypes.byref(call), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
            assert rc == 0, lib.lutgemm_strerror(rc).decode()
            got.append(out.double() - bias.double())
    finally:
        lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)
    want = x.double() @ _dense(ROW, bW, alpha, None)
    for y in got:       # (the rounding of the result: 2^-11, bf16 2^-8, of the sum with the bias)
        assert ((y - want).norm() / want.norm()).item() <= (6e-4, 5e-3, 1e-6)[out_type]
