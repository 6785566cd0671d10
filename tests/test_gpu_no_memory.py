"""Calls whose buffers have no memory: a failed growth takes nothing from the stream and leaves no error behind for the next
launch's check, and the gated call goes on without the words that its product would take."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native

pytestmark = pytest.mark.gpu

ENOMEM, ECAPTURE = -5, -6


def _problems(dev, M, N, K, nb=3, groups=8):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn((M, K), generator=g, device=dev).half()
    outs = [torch.empty((M, N), dtype=torch.float16, device=dev) for _ in range(2)]
    weights = [(torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 32, nb, N), generator=g, device=dev, dtype=torch.int32),
                (0.02 * torch.randn((groups, nb, N), generator=g, device=dev)).half()) for _ in range(2)]
    pair = (native.FusedProblem * 2)()
    for i, (bW, alpha) in enumerate(weights):
        pair[i] = native.FusedProblem(bW.data_ptr(), alpha.data_ptr(), x.data_ptr(), outs[i].data_ptr(), N, K, nb, groups, M, 1, None, None,
                                      1e-5, None, None, None, None, 0)
    return pair, outs, (x, weights)


def _pointer(stream):
    return ctypes.c_void_p(stream.cuda_stream)


def test_a_failed_growth_leaves_no_error_and_the_buffer(gpu_device):
    dev, lib = gpu_device, native.cabi()
    M, N, K = 16, 8192, 8192   # (slices: accumulator words)
    pair, outs, held = _problems(dev, M, N, K)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    lib.lutgemm_release_workspaces()
    assert lib.lutgemm_gemv_rowwise_f16_fused(2, pair, _pointer(stream)) == 0
    torch.cuda.synchronize()
    want = [o.clone() for o in outs]
    for words in (1 << 44, 1 << 60):   # (128 TB and more)
        assert lib.lutgemm_reserve_workspace(_pointer(stream), words) == ENOMEM
        assert lib.lutgemm_gemv_rowwise_f16_fused(2, pair, _pointer(stream)) == 0
        torch.cuda.synchronize()
        assert all(torch.equal(o, w) for o, w in zip(outs, want))
    assert lib.lutgemm_reserve_workspace(_pointer(stream), 1 << 44) == ENOMEM
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):   # (what the stream had before is still there)
        assert lib.lutgemm_gemv_rowwise_f16_fused(2, pair, _pointer(stream)) == 0
    for o in outs:
        o.fill_(7.0)
    graph.replay()
    torch.cuda.synchronize()
    assert all(torch.equal(o, w) for o, w in zip(outs, want))


@pytest.mark.parametrize("M,N,K,slices", [(8, 1024, 1024, False), (16, 8192, 8192, True)])
def test_gated_call_without_words_for_the_product(gpu_device, M, N, K, slices):
    dev, lib = gpu_device, native.cabi()
    pair, outs, held = _problems(dev, M, N, K)
    act = torch.empty_like(outs[0])
    eager, captured_on = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    lib.lutgemm_release_workspaces()
    assert lib.lutgemm_gemv_rowwise_f16_gated(pair, act.data_ptr(), _pointer(eager)) == 0
    torch.cuda.synchronize()
    want = act.clone()
    graph = torch.cuda.CUDAGraph()
    if slices:
        # the two problems' words fill the stream's buffer, which holds a power of two of them
        assert 2 * M * N == 1 << 18
        with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=captured_on):
            assert lib.lutgemm_gemv_rowwise_f16_gated(pair, act.data_ptr(), _pointer(captured_on)) == ECAPTURE
        assert lib.lutgemm_reserve_workspace(_pointer(captured_on), 2 * M * N) == 0
    with torch.cuda.graph(graph, stream=captured_on):
        assert lib.lutgemm_gemv_rowwise_f16_gated(pair, act.data_ptr(), _pointer(captured_on)) == 0
    for _ in range(3):
        for t in (act, *outs):
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(act, want)
        assert torch.isfinite(outs[0]).all()   # (the sums went there: two launches)
