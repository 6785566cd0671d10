"""Gate and up projection with their product formed by the launch that computes both: the same bits as the two
launches it stands for, call after call (its words are zero again) and replay after replay."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native

pytestmark = pytest.mark.gpu

CASES = [  # M, N, K, planes of gate and up, alpha groups of each, split RMSNorm
    (3, 64, 128, 3, 3, 1, False), (8, 100, 1024, 2, 4, 8, True), (16, 1540, 2048, 4, 1, 16, True), (17, 200, 4096, 3, 2, 32, False),
    (8, 11008, 4096, 3, 2, 32, True), (32, 20480, 1024, 1, 3, 8, True), (40, 72, 2048, 4, 4, 16, False), (2, 512, 1024, 3, 3, 8, True),
]


@pytest.mark.parametrize("M,N,K,gate_bits,up_bits,groups,split", CASES)
def test_same_bits_as_two_launches(gpu_device, M, N, K, gate_bits, up_bits, groups, split):
    dev, lib = gpu_device, native.cabi()
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn((M, K), generator=g, device=dev).half()
    sums = (x.float() ** 2).view(M, K // 32, 32).sum(-1).contiguous() if split else None
    outs = [torch.empty((M, N), dtype=torch.float16, device=dev) for _ in range(2)]
    weights = [(torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32),
                (0.02 * torch.randn((groups, nb, N), generator=g, device=dev)).half()) for nb in (gate_bits, up_bits)]
    pair = (native.FusedProblem * 2)()
    for i, ((bW, alpha), nb) in enumerate(zip(weights, (gate_bits, up_bits))):
        pair[i] = native.FusedProblem(bW.data_ptr(), alpha.data_ptr(), x.data_ptr(), outs[i].data_ptr(), N, K, nb, groups, M, 1, None, None,
                                      1e-5, None, None, None, sums.data_ptr() if split else None, K // 32 if split else 0)
    want, act = torch.empty_like(outs[0]), torch.empty_like(outs[0])
    stream = torch.cuda.Stream()
    sp = ctypes.c_void_p(stream.cuda_stream)
    torch.cuda.synchronize()
    assert lib.lutgemm_gemv_rowwise_f16_fused(2, pair, sp) == 0
    assert lib.lutgemm_decode_silu_mul_f16(outs[0].data_ptr(), outs[1].data_ptr(), want.data_ptr(), M * N, sp) == 0
    torch.cuda.synchronize()
    assert torch.isfinite(want.float()).all() and want.float().abs().max() > 0
    for _ in range(3):
        act.fill_(7.0)
        torch.cuda.synchronize()
        assert lib.lutgemm_gemv_rowwise_f16_gated(pair, act.data_ptr(), sp) == 0
        torch.cuda.synchronize()
        assert torch.equal(act, want)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        assert lib.lutgemm_gemv_rowwise_f16_gated(pair, act.data_ptr(), sp) == 0
    for _ in range(3):
        act.fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(act, want)
        assert lib.lutgemm_gemv_rowwise_f16_gated(pair, want.data_ptr(), sp) == 0      # (the words are shared with eager calls)
        torch.cuda.synchronize()


@pytest.mark.parametrize("M,N,K", [(8, 1024, 1024), (16, 8192, 8192), (24, 1024, 4096)])   # one K-slice, several, 32-row tiles
def test_special_activations_and_sums(gpu_device, M, N, K):
    """Infinite and NaN sums (the exchanged word of an output is never taken for an empty one), sums beyond fp16, zeros of
    either sign: the bits of two launches, NaN as NaN."""
    dev, lib, nb = gpu_device, native.cabi(), 2
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn((M, K), generator=g, device=dev).half()
    x[0, 3], x[1, K - 1], x[2, K // 2] = float("nan"), float("inf"), -float("inf")
    x[3] = 0.0
    x[4] = 30000.0
    outs = [torch.empty((M, N), dtype=torch.float16, device=dev) for _ in range(2)]
    weights = [(torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32),
                (0.02 * torch.randn((8, nb, N), generator=g, device=dev)).half()) for _ in range(2)]
    pair = (native.FusedProblem * 2)()
    for i, (bW, alpha) in enumerate(weights):
        pair[i] = native.FusedProblem(bW.data_ptr(), alpha.data_ptr(), x.data_ptr(), outs[i].data_ptr(), N, K, nb, 8, M, 1, None, None,
                                      1e-5, None, None, None, None, 0)
    want, act = torch.empty_like(outs[0]), torch.empty_like(outs[0])
    sp = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.lutgemm_gemv_rowwise_f16_fused(2, pair, sp) == 0
    assert lib.lutgemm_decode_silu_mul_f16(outs[0].data_ptr(), outs[1].data_ptr(), want.data_ptr(), M * N, sp) == 0
    torch.cuda.synchronize()
    assert torch.isnan(want[0]).all() and not torch.isfinite(want[4]).all() and (want[3] == 0).all()
    for _ in range(2):
        act.fill_(7.0)
        assert lib.lutgemm_gemv_rowwise_f16_gated(pair, act.data_ptr(), sp) == 0
        torch.cuda.synchronize()
        nan = torch.isnan(want)
        assert torch.equal(torch.isnan(act), nan)
        assert torch.equal(act[~nan].view(torch.int16), want[~nan].view(torch.int16))


def test_what_is_refused(gpu_device):
    lib = native.cabi()
    t = torch.zeros(1 << 16, dtype=torch.float16, device=gpu_device)
    at = lambda i: t.data_ptr() + 8192 * i
    def call(**change):
        field = dict(bW=at(0), alpha_f16=at(1), x_f16=at(2), N=64, K=128, nb=1, num_groups=1, M=8, overwrite=1)
        field.update({k: v for k, v in change.items() if k != "act"})
        pair = (native.FusedProblem * 2)(native.FusedProblem(out_f16=at(3), **{**field, "N": 64, "overwrite": 1}),
                                         native.FusedProblem(out_f16=at(4), **field))
        return lib.lutgemm_gemv_rowwise_f16_gated(pair, change.get("act", at(5)), None)
    assert call() == 0
    torch.cuda.synchronize()
    for change in (dict(N=128), dict(overwrite=0), dict(act=at(4)), dict(act=at(2)), dict(act=None), dict(act=at(5) + 8), dict(sumsq_out_f32=at(6))):
        assert call(**change) != 0, change
