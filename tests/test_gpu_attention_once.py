"""Attention steps that read cached rows past the caches give the bits of those that do not."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,KV,hd,max_pos,positions", [
    (8, 32, 32, 128, 300, (0, 127, 299)),      # 256 workgroups and more: four waves each
    (8, 32, 32, 64, 600, (1, 511, 599)),
    (2, 16, 16, 128, 520, (0, 256, 519)),      # fewer: eight
    (2, 16, 16, 64, 1040, (512, 1039)),
    (3, 40, 10, 128, 1000, (0, 255, 999)),     # query heads that share rows
])
def test_bits_of_the_step(gpu_device, B, H, KV, hd, max_pos, positions):
    lib, dev = native.cabi(), gpu_device
    g = torch.Generator(device=dev).manual_seed(B + H + hd)
    mk = lambda *s: torch.randn(s, generator=g, device=dev).half()
    q, k, v, cos, sin = mk(B, H * hd), mk(B, KV * hd), mk(B, KV * hd), mk(max_pos, hd), mk(max_pos, hd)
    cache = mk(2, B, KV, max_pos, hd)
    plan = native.AttentionPlan()
    assert lib.lutgemm_describe_attention_plan(B, H, KV, hd, max_pos, 1 << 30, ctypes.byref(plan)) == 0 and plan.once == 1
    sp = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for pos in positions:
        results = []
        for step_bytes in (0, 1 << 30):
            own, out, p = cache.clone(), torch.zeros_like(q), torch.tensor([pos], device=dev)
            assert lib.lutgemm_decode_attention_step_f16(*(t.data_ptr() for t in (q, k, v, cos, sin, own[0], own[1], p, out)), B, H, KV, hd,
                                                         max_pos, step_bytes, sp) == 0
            torch.cuda.synchronize()
            results.append((out, own))
        assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
