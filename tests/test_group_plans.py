"""The shares of grouped look-up launches, through the described plans (host arithmetic, no GPU): which launches need
accumulator words, how many workgroups a shader engine is dealt, and what unlike widths get."""
import ctypes
import random

import pytest

from shiftaddllm_amd import native

LOOKUP, MATRIX_CORE = 0, 1
COLS = SET = 256      # outputs and inputs of an item


@pytest.fixture(scope="module")
def lib():
    return native.cabi()


def _problems(K, outs, M, norm):
    """Problems of [(N, planes), ...]: addresses that are never read, in ranges of their own."""
    arr = (native.FusedProblem * len(outs))()
    at = 1 << 40
    def take(size):
        nonlocal at
        first, at = at, at + (size + 255) // 256 * 256
        return first
    x, weight = take(2 * M * K), take(2 * K) if norm else None
    for i, (N, nb) in enumerate(outs):
        arr[i] = native.FusedProblem(take(K // 8 * nb * N), take(K // 32 * nb * N * 2), x, take(2 * M * N), N, K, nb, 1, M, 1, weight, None, 1e-5,
                                     None, None, None, None, 0)
    return arr


def _describe(lib, K, outs, M, norm=True):
    plan = native.GroupPlan()
    assert lib.lutgemm_describe_group_plan(len(outs), _problems(K, outs, M, norm), ctypes.byref(plan)) == 0
    n = len(outs)
    return plan, list(plan.workgroups[:n]), list(plan.units_per_workgroup[:n])


def _whole_rows(K, outs, M):
    """Whether a launch had ranges of whole rows of items alone when the line was drawn: 256 workgroups up to 24 MB of
    signs, 512 beyond, shared in proportion to 0.45 + 0.13 * planes."""
    sets = -(-K // SET)
    items = [-(-N // COLS) * sets for N, _ in outs]
    cost = [0.45 + 0.13 * nb for _, nb in outs]
    budget = 256 if sum(N * (K // 8) * nb * M for N, nb in outs) <= 24 << 20 else 512
    lo, hi = 0.0, max(i * c for i, c in zip(items, cost))
    for _ in range(50):
        mid = 0.5 * (lo + hi)
        per = [int(mid / c) for c in cost]
        if all(p >= 1 for p in per) and sum(-(-i // p) * M for i, p in zip(items, per)) <= budget:
            hi = mid
        else:
            lo = mid
    least = (sets + 38) // 39
    for i, c in zip(items, cost):
        per = max(1, int(hi / c))
        per = min(i, max(least, -(-i // -(-i // per))))
        if per % sets:
            return False
    return True


def test_launches_that_once_needed_a_reservation_by_mistake(lib):
    for K, outs, M in ((4608, [(10192, 1), (40784, 3)], 8), (6144, [(22272, 1), (20736, 1)], 6), (9472, [(25856, 4), (6656, 4)], 8)):
        assert _whole_rows(K, outs, M)
        plan, _, units = _describe(lib, K, outs, M)
        assert plan.kernel == LOOKUP and not plan.needs_workspace and all(u % -(-K // SET) == 0 for u in units)


def test_launches_that_need_words(lib):
    rng = random.Random(5)
    without = 0
    for i in range(6000):
        K = 32 * rng.randint(16, 320) if i % 2 else 256 * rng.randint(8, 40)
        outs = [(4 * rng.randint(16, 12000 if i % 3 else 2000), rng.randint(1, 4)) for _ in range(rng.randint(1, 4))]
        M = rng.choice((1, 2, 2, 4, 8))
        plan, workgroups, units = _describe(lib, K, outs, M)
        assert plan.kernel == LOOKUP and plan.launches == 1
        for (N, _), n, u in zip(outs, workgroups, units):
            items = -(-N // COLS) * -(-K // SET)
            assert u >= 1 and (n // M - 1) * u < items
        if _whole_rows(K, outs, M):
            without += 1
            assert not plan.needs_workspace, (K, outs, M)
    assert without > 30


def _most_on_an_engine(workgroups):
    dealt = [0] * 32
    widest = max(workgroups)
    for i, n in enumerate(workgroups):
        for b in range(n):
            dealt[(i * widest + b) % 32] += 1
    return max(dealt)


def test_no_engine_is_dealt_more_than_it_holds(lib):
    rng = random.Random(3)
    seen = 0
    for _ in range(1500):
        K = rng.choice((4096, 4608, 5120, 6656, 8192))
        outs = [(128 * rng.randint(8, 120), rng.randint(1, 4)) for _ in range(rng.choice((2, 3)))]
        M = rng.choice((1, 2))
        plan, workgroups, units = _describe(lib, K, outs, M)
        # (at most 512: two per CU; below half of that no engine is near its limit)
        if plan.needs_workspace and sum(workgroups) > 256:
            seen += 1
            assert _most_on_an_engine(workgroups) <= 16, (K, outs, M, workgroups)
    assert seen > 700


@pytest.mark.parametrize("K,outs,M,units", [
    (4096, [(4096, 2), (4096, 1), (4096, 4)], 2, [4, 4, 2]),          # within tiles of 16 items
    (5120, [(5120, 3), (5120, 2), (5120, 2)], 2, [5, 5, 5]),          # of 20
    (4096, [(4096, 3), (4096, 3), (4096, 3)], 1, [2, 2, 2]),
    (3072, [(8192, 2), (8192, 4)], 2, [4, 3]),                        # inputs shorter than 4096
    (2048, [(5632, 2), (5632, 4)], 1, [2, 2]),                        # a workgroup per CU
])
def test_shares(lib, K, outs, M, units):
    assert _describe(lib, K, outs, M)[2] == units


def test_other_routes_and_refusals(lib):
    outs = [(4096, 3), (4096, 2)]
    assert _describe(lib, 4096, outs, 8, norm=False)[0].kernel == MATRIX_CORE
    assert _describe(lib, 4096, outs, 1, norm=False)[0].kernel == LOOKUP
    plan = native.GroupPlan()
    arr = _problems(4096, outs, 1, True)
    assert lib.lutgemm_describe_group_plan(0, arr, ctypes.byref(plan)) == lib.lutgemm_describe_group_plan(2, arr, None) == -1
    arr[1].out_f16 = arr[0].out_f16
    assert lib.lutgemm_describe_group_plan(2, arr, ctypes.byref(plan)) == -1
    arr = _problems(4096, outs, 1, True)
    arr[1].norm_weight_f16 = None
    assert lib.lutgemm_describe_group_plan(2, arr, ctypes.byref(plan)) != 0
