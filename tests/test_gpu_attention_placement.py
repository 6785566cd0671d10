"""Attention steps whose (sequence, kv head) pairs do not fill the last eight places: nothing is left out, nothing is written by the
workgroups beyond the last pair."""
import ctypes

import pytest
import torch

from shiftaddllm_amd import native
from test_gpu_decode_glue import test_attention_step_routes as check

pytestmark = pytest.mark.gpu

SIZES = [  # B, H, KV, hd, max_pos, pos
    (7, 4, 1, 64, 8000, 199), (3, 6, 3, 128, 2000, 0), (7, 40, 10, 128, 300, 257), (17, 16, 1, 64, 2000, 129), (1, 16, 4, 128, 4200, 700),
    (1, 4, 1, 128, 200, 130), (17, 16, 1, 64, 140, 129), (2, 24, 1, 128, 150, 149), (3, 64, 2, 128, 90, 80),
]


def _plan(B, H, KV, hd, max_pos):
    plan = native.AttentionPlan()
    assert native.cabi().lutgemm_describe_attention_plan(B, H, KV, hd, max_pos, 0, ctypes.byref(plan)) == 0
    return plan


@pytest.mark.parametrize("B,H,KV,hd,max_pos,pos", SIZES)
def test_partial_places(gpu_device, B, H, KV, hd, max_pos, pos):
    assert _plan(B, H, KV, hd, max_pos).placed == 1
    check(gpu_device, B, H, KV, hd, max_pos, pos, 0)


@pytest.mark.parametrize("B,H,KV,hd,max_pos,pos", [(1, 64, 1, 128, 200, 130), (9, 24, 1, 64, 140, 129), (1, 64, 2, 128, 2000, 300)])
def test_pairs_that_would_fill_an_xcd_are_spread(gpu_device, B, H, KV, hd, max_pos, pos):
    assert _plan(B, H, KV, hd, max_pos).placed == 0
    check(gpu_device, B, H, KV, hd, max_pos, pos, 0)


@pytest.mark.parametrize("B,H,KV,hd,max_pos,pos", SIZES)
def test_nothing_beyond_the_last_pair(gpu_device, B, H, KV, hd, max_pos, pos):
    """Outputs and caches with room for eight more pairs behind them."""
    dev, lib = gpu_device, native.cabi()
    g = torch.Generator(device=dev).manual_seed(B * 100 + H + pos)
    mk = lambda *s: torch.randn(s, generator=g, device=dev).half()
    pairs, rep = B * KV, H // KV
    assert _plan(B, H, KV, hd, max_pos).workgroups > pairs * rep
    q, k, v, cos, sin = mk(pairs + 8, rep, hd), mk(pairs + 8, hd), mk(pairs + 8, hd), mk(max_pos, hd), mk(max_pos, hd)
    caches = mk(2, pairs + 8, max_pos, hd)
    before, out = caches.clone(), torch.full((pairs + 8, rep, hd), 777.0, dtype=torch.float16, device=dev)
    p = torch.tensor([pos], device=dev)
    sp = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.lutgemm_decode_attention_f16(*(t.data_ptr() for t in (q, k, v, cos, sin, caches[0], caches[1], p, out)), B, H, KV, hd, max_pos,
                                            sp) == 0
    torch.cuda.synchronize()
    assert (out[pairs:] == 777.0).all() and (out[:pairs] != 777.0).all()
    assert torch.equal(caches[:, pairs:], before[:, pairs:])
    others = torch.arange(max_pos, device=dev) != pos
    assert torch.equal(caches[:, :, others], before[:, :, others])
    assert torch.equal(caches[1, :pairs, pos], v[:pairs])
