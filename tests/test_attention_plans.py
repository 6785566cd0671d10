"""Plans of the attention step without a GPU: lutgemm_describe_attention_plan is pure host arithmetic.  Cached rows are read past the
caches only where what a token reads besides them leaves none of them in the 256 MB memory-side cache."""
import ctypes
import os

import pytest

MB = 1 << 20


@pytest.fixture(scope="module")
def lib():
    from shiftaddllm_amd import native
    if not os.path.exists(native.KERNEL_LIB):
        from shiftaddllm_amd import build
        build.build_kernel_library()
    return native.cabi()


def describe(lib, batch, heads, kv_heads, head_dim=128, max_positions=2048, step_bytes=0):
    from shiftaddllm_amd import native
    plan = native.AttentionPlan()
    rc = lib.lutgemm_describe_attention_plan(batch, heads, kv_heads, head_dim, max_positions, step_bytes, ctypes.byref(plan))
    return rc, plan


def once(lib, *sizes, **kw):
    rc, plan = describe(lib, *sizes, **kw)
    assert rc == 0
    return bool(plan.once)


@pytest.mark.parametrize("batch,heads,kv_heads,max_positions", [(4, 8, 8, 2048), (1, 8, 8, 2048), (8, 8, 2, 2048), (2, 16, 16, 1024), (8, 32, 32, 1024)])
def test_rows_that_are_found_again_are_read_as_usual(lib, batch, heads, kv_heads, max_positions):
    """Caches of 8 to 134 MB a block in networks whose weights leave room for rows beside them, and callers that do not say."""
    for step_bytes in (0, 71 * MB, 200 * MB, 300 * MB, 384 * MB - 1):
        assert not once(lib, batch, heads, kv_heads, max_positions=max_positions, step_bytes=step_bytes)


def test_rows_of_large_networks_are_read_past_the_caches(lib):
    for step_bytes in (384 * MB, 3056 * MB, 1 << 40):
        assert once(lib, 8, 32, 32, max_positions=1024, step_bytes=step_bytes)
        assert once(lib, 2, 16, 16, head_dim=64, step_bytes=step_bytes)
        assert not once(lib, 1, 32, 32, max_positions=256, step_bytes=step_bytes)     # 4 MB a block
        assert once(lib, 8, 32, 8, step_bytes=step_bytes)                             # query heads that share 64 MB of rows
        assert not once(lib, 9, 32, 8, step_bytes=step_bytes)
        assert not once(lib, 8, 32, 32, head_dim=96, step_bytes=step_bytes)           # the kernel for any head size


def test_what_the_call_refuses(lib):
    assert describe(lib, 1, 4, 3)[0] == -1
    assert describe(lib, 0, 4, 4)[0] == -1
    assert describe(lib, 1, 4, 4, head_dim=60)[0] == -1
    assert describe(lib, 1, 4, 4, max_positions=8193)[0] == -1
    assert lib.lutgemm_describe_attention_plan(1, 4, 4, 128, 256, 0, None) == -1
    p = ctypes.c_void_p(0x1000)
    call = lib.lutgemm_decode_attention_step_f16       # (refused on the host: the addresses are never looked at)
    assert call(p, p, p, p, p, p, p, p, p, 1, 4, 3, 64, 16, 0, None) == -1
    assert call(p, p, p, p, p, p, p, None, p, 1, 4, 4, 64, 16, 0, None) == -1
    assert call(p, p, p, p, p, ctypes.c_void_p(0x1008), p, p, p, 1, 4, 4, 64, 16, 0, None) == -2


def test_the_decoder_says_what_a_token_reads():
    from shiftaddllm_amd.decode import DecoderConfig, LutDecoder
    cfg = DecoderConfig(vocab_size=96, hidden=256, intermediate=512, layers=2, heads=2, kv_heads=1, max_positions=16)
    model = LutDecoder(cfg, None, device="cpu", default_bits=3)
    macs = 2 * (256 * 256 * 2 + 256 * 128 * 2 + 3 * 256 * 512)
    assert model.step_bytes == macs * 3 // 8 + macs // 128 * 3 * 2 + 2 * 96 * 256     # signs, one scale per 128 inputs, output matrix


@pytest.mark.parametrize("max_positions", [64, 8192])
def test_no_cu_gets_more_to_do_where_pairs_are_placed(lib, max_positions):
    """32 CUs to an XCD: where query heads of a pair share one, its fullest CU holds no more workgroups than with all spread evenly, and
    the grid has room for every pair and head."""
    for pairs in range(1, 140):
        for rep in (1, 2, 3, 4, 5, 7, 8, 12, 16, 24, 32, 33, 48, 64):
            rc, plan = describe(lib, 1, pairs * rep, pairs, max_positions=max_positions)
            assert rc == 0
            if not plan.placed:
                assert plan.workgroups == pairs * rep
                continue
            fullest, even = -(-pairs // 8) * rep, -(-pairs * rep // 8)
            assert rep > 1 and plan.workgroups == 8 * fullest
            assert -(-fullest // 32) <= -(-even // 32)


def test_pairs_that_share_rows_are_placed_where_it_pays(lib):
    placed = lambda pairs, rep: describe(lib, 1, pairs * rep, pairs)[1].placed == 1
    assert all(placed(pairs, rep) for pairs in (1, 2, 3, 7, 9, 20) for rep in (2, 4, 8)) and placed(140, 4) and placed(64, 4) and placed(8, 64)
    assert not any(placed(*few) for few in ((1, 64), (2, 64), (4, 64), (9, 64), (9, 24), (9, 48), (17, 24), (1, 32), (2, 32), (8, 1)))
