"""Attention steps whose (sequence, kv head) pairs do not fill the last eight places: nothing is left out or written twice."""
import pytest

from test_gpu_decode_glue import test_attention_step_routes as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,KV,hd,max_pos,pos", [  # caches of 8 MB and more (placed), and smaller ones
    (7, 4, 1, 64, 8000, 199), (3, 6, 3, 128, 2000, 0), (7, 40, 10, 128, 300, 257), (17, 16, 1, 64, 2000, 129), (1, 16, 4, 128, 4200, 700),
    (1, 4, 1, 128, 200, 130), (17, 16, 1, 64, 140, 129)])
def test_partial_places(gpu_device, B, H, KV, hd, max_pos, pos):
    check(gpu_device, B, H, KV, hd, max_pos, pos, 0)
