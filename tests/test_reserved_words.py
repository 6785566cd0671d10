"""Which calls need accumulator words, and so a reservation before a capture, is fixed in the sizes: it does not move with
the costs that choose between kernels and cuts.  Checked on the host through the described plans."""
import random

import pytest

from test_launch_plans import BLOCK_F16, BLOCK_I8, GEMM, MATRIX_CORE, ROWWISE, UNIFORM, describe, lib  # noqa: F401


def never_cut(N, K, M):
    """Whether the GEMM kernel, which needs no words, was the choice for a call of more than 32 rows when the line was
    drawn: its time with slices of four waves against rounds of 3 us of the matrix-core kernel."""
    rows = 64 if M <= 64 else 128
    alone, beside = (0.9, 1.6) if rows == 64 else (1.2, 2.1)
    tiles, steps = -(-N // 256) * -(-M // rows), -(-K // 128) * 2
    best = None
    for ks in range(1, 17):
        if ks > 1 and 2 * ks > steps:
            break
        own = (-(-steps // ks) + 1) // 2 * 2
        if -(-steps // own) != ks:
            continue
        if ks > 1 and (tiles * ks > 512 or ks * M * N * 4 > 64 << 20):
            break
        full, rest = divmod(tiles * ks, 512)
        us = full * (own * beside + 5) + (4 + 2 * ks * M * N / 1e6 if ks > 1 else 0)
        us += own * (beside if rest > 256 else alone) + 5 if rest else 0
        if best is None or us < 0.99 * best:
            best = us
    return best < 5 + 3 * -(-N // 64) * -(-M // 32) * -(-K // 1024) / 256


@pytest.mark.parametrize("fmt,N,K,nb,M", [(ROWWISE, 4096, 14336, 1, 33), (ROWWISE, 3904, 17536, 2, 33), (UNIFORM, 3536, 26240, 1, 40),
                                          (ROWWISE, 512, 49152, 1, 512), (UNIFORM, 3860, 25984, 1, 64)])
def test_calls_that_once_needed_a_reservation_by_mistake(lib, fmt, N, K, nb, M):  # noqa: F811
    rc, p = describe(lib, fmt, N, K, nb, K // 128, M)
    assert rc == 0 and not p.needs_workspace and never_cut(N, K, M)


def test_calls_of_many_rows_that_need_words(lib):  # noqa: F811
    rng = random.Random(7)
    needed = 0
    for i in range(20000):
        K, N = (128 * rng.randint(1, 400), 16 * rng.randint(4, 600)) if i % 2 else (32 * rng.randint(4, 1400), 4 * rng.randint(16, 2400))
        M, nb, fmt = rng.randint(33, 600) if i % 3 else rng.randint(33, 64), rng.randint(1, 4), rng.choice((ROWWISE, UNIFORM, BLOCK_I8))
        rc, p = describe(lib, fmt, N, K, nb, 1 if fmt == BLOCK_I8 else K // 32, M)
        assert rc == 0 and p.kernel in (MATRIX_CORE, GEMM)
        if p.needs_workspace:
            needed += 1
            assert not never_cut(N, K, M), (fmt, N, K, nb, M)
    assert needed > 500


@pytest.mark.parametrize("fmt,N,K,nb,M,rows,slices", [(ROWWISE, 4096, 28672, 4, 64, 32, 2), (ROWWISE, 512, 49152, 1, 512, 32, 2),
                                                      (BLOCK_I8, 5120, 13824, 2, 48, 16, 1), (UNIFORM, 2048, 16384, 3, 40, 32, 4)])
def test_without_the_gemm_kernel_calls_are_cut(lib, fmt, N, K, nb, M, rows, slices):  # noqa: F811
    from shiftaddllm_amd import native
    assert lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], 1 << 20) == 0
    try:
        rc, p = describe(lib, fmt, N, K, nb, 8 if fmt == BLOCK_I8 else K // 128, M)
    finally:
        lib.lutgemm_set_option(native.OPTIONS["TILE_MIN_M"], -1)
    assert rc == 0 and (p.kernel, p.rows_per_pass, p.k_slices) == (MATRIX_CORE, rows, slices)


@pytest.mark.parametrize("fmt,N,K,nb,groups,M,kernel", [
    # (us measured, matrix-core / GEMM kernel)
    (BLOCK_F16, 20864, 1408, 3, 8, 64, MATRIX_CORE),   # 32.5 / 51.6
    (BLOCK_F16, 7360, 4864, 4, 8, 48, MATRIX_CORE),    # 34.3 / 53.6
    (BLOCK_I8, 4480, 4608, 4, 8, 72, MATRIX_CORE),     # 24.5 / 33.0
    (UNIFORM, 21888, 1024, 4, 8, 72, MATRIX_CORE),     # 39.9 / 53.0
    (ROWWISE, 6464, 4096, 3, 32, 65, MATRIX_CORE),     # 18.0 / 22.8
    (BLOCK_I8, 10688, 1792, 4, 8, 256, GEMM),          # 78.6 / 42.7
    (ROWWISE, 4352, 17408, 4, 136, 64, GEMM),          # 75.4 / 48.3
    (UNIFORM, 5312, 7168, 3, 56, 112, GEMM),           # 52.7 / 40.9
    (ROWWISE, 13800, 64, 3, 2, 128, GEMM),             # 15.5 / 10.9
    (ROWWISE, 1820, 64, 3, 1, 100, MATRIX_CORE),       # 4.1 / 9.6
    (ROWWISE, 6028, 64, 4, 1, 33, GEMM),               # 6.4 / 8.6: calls of up to 64 inputs keep the line they had
])
def test_the_faster_kernel_where_they_differ_much(lib, fmt, N, K, nb, groups, M, kernel):  # noqa: F811
    rc, p = describe(lib, fmt, N, K, nb, groups, M)
    assert rc == 0 and p.kernel == kernel


@pytest.mark.parametrize("N,K,nb,M,kernel", [
    # us measured, one launch of the matrix-core kernel / the GEMM kernel's slices / those in turn
    (13920, 2560, 2, 75, MATRIX_CORE),    # 26.3 / 35.2 / 93
    (4480, 12800, 3, 34, MATRIX_CORE),    # 27.1 / 29.1 / 261
    (10848, 3200, 4, 50, MATRIX_CORE),    # 26.6 / 32.4 / 110
    (9120, 9984, 3, 64, GEMM),            # 49.8 / 37.6 / 194
    (12816, 3072, 3, 123, GEMM),          # 47.4 / 34.2 / 74
])
def test_one_launch_is_given_up_for_slices_only_for_a_gain(lib, N, K, nb, M, kernel):  # noqa: F811
    """Slices are taken in turn where their sums have no place, as under a capture with nothing reserved."""
    rc, p = describe(lib, ROWWISE, N, K, nb, K // 128, M)
    assert rc == 0 and p.kernel == kernel and not p.needs_workspace and (p.k_slices > 1) == (kernel == GEMM) and not never_cut(N, K, M)
