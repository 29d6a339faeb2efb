"""Columns admitted through the pool's staging block: more admissions in a row than it holds, a
record larger than it, slots reused right after a removal, and results fetched between. A
column's bits depend on its own data alone, so each must equal the same column run by itself.
"""
import numpy as np
import pytest

from femorax_amd import core
from femorax_amd import synthetic as S

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = core.Context(0)
    yield c
    c.close()


def column(seed, nelem):
    return core.pimy_materials(S.soil_layers(S.Lcg(seed), 3)), S.column_layer_of(nelem, 3)


def alone(ctx, seed, nelem, record, iterations):
    pool = core.ColumnPool(ctx, nelem, 1, 0.005, max_record=11 * len(record))
    cid = pool.add(*column(seed, nelem), len(record), record, record=False)
    pool.run(iterations)
    out = pool.fetch(cid)
    pool.close()
    return out


def test_more_admissions_than_the_staging_block_holds(ctx):
    steps = 20000  # 160 kB each: the 1 MB block wraps
    record = np.resize(S.ground_motion(400, 0.005, 7)[100:], steps)
    pool = core.ColumnPool(ctx, 2000, 64, 0.005, max_record=64 * steps)
    sizes = [1 + (7 * k) % 31 for k in range(60)]
    ids = [pool.add(*column(k, n), steps, record * (1.0 + 0.01 * k), record=False) for k, n in enumerate(sizes)]
    pool.run(6)
    for k in (0, 25, 26, 59):
        got, want = pool.fetch(ids[k]), alone(ctx, k, sizes[k], record * (1.0 + 0.01 * k), 6)
        for f in ("u", "v", "a"):
            np.testing.assert_array_equal(got[f], want[f])
        assert np.any(got["u"])
    pool.close()


def test_a_record_larger_than_the_staging_block(ctx):
    steps = 600000
    record = np.resize(S.ground_motion(400, 0.005, 7)[100:], steps)
    pool = core.ColumnPool(ctx, 40, 2, 0.005, max_record=2 * steps)
    small = pool.add(*column(1, 9), 50, record[:50], record=False)
    large = pool.add(*column(2, 13), steps, record, record=False)
    pool.run(8)
    for cid, seed, n in ((small, 1, 9), (large, 2, 13)):
        want = alone(ctx, seed, n, record[:50], 8)
        got = pool.fetch(cid)
        for f in ("u", "v", "a"):
            np.testing.assert_array_equal(got[f], want[f])
    pool.close()


def test_slots_reused_after_removal(ctx):
    record = S.ground_motion(400, 0.005, 9)[100:112]
    pool = core.ColumnPool(ctx, 30, 2, 0.005, max_record=4000)
    first = pool.add(*column(3, 30), 12, record)
    assert pool.add(*column(4, 5), 12, record) is None  # no room
    pool.run(5)
    pool.remove(first)
    second = pool.add(*column(5, 17), 12, record)
    third = pool.add(*column(6, 13), 12, record)
    while pool.run(4):
        pass
    assert sorted(pool.finished()) == sorted([second, third])
    got = [pool.fetch(second), pool.fetch(third)]
    for g, seed, n in zip(got, (5, 6), (17, 13)):
        one = core.ColumnPool(ctx, n, 1, 0.005, max_record=400)
        cid = one.add(*column(seed, n), 12, record)
        while one.run(4):
            pass
        want = one.fetch(cid)
        for f in ("u", "v", "a", "history"):
            np.testing.assert_array_equal(g[f], want[f])
        assert one.status(cid)["steps"] == 12
        one.close()
    pool.close()
