"""Eq tables described together (dps_eq_build_many): the first reader of one builds them all in one launch, whatever reads first --
a download, a product that takes its table in closed form, a sum that reads entries -- and whichever of them are still there."""
import importlib

import numpy as np
import pytest

from util import rand_base, rand_e2

pytestmark = pytest.mark.gpu
ONE = np.array([1, 0], dtype=np.uint64)


@pytest.fixture(scope="module")
def dp():
    return importlib.import_module("deep-prove_amd")


@pytest.fixture()
def ctx(dp):
    c = dp.Context(0)
    yield c
    c.close()


def _eq_launches(ctx, work):
    ctx.profile(True)
    try:
        ctx.profile_reset()
        work()
        return ctx.profile_read()["eq"]["launches"]
    finally:
        ctx.profile(False)


def _prove(dp, ctx, orc, n, mles, host, terms):
    tr, otr = dp.Transcript(b"eq"), orc.OracleTranscript(b"eq")
    got, want = ctx.sumcheck_prove(n, mles, terms, tr), orc.sc_prove(n, host, terms, otr)
    assert all((a == b).all() for a, b in zip(got, want)) and tr.state() == otr.state()


def test_downloads_come_out_of_one_launch(ctx, orc):
    points = [rand_e2(m, 100 + i) for i, m in enumerate((0, 1, 7, 8, 9, 12, 16, 16))]
    tables = ctx.eq_build_many(points)

    def read():
        for t, p in zip(tables, points):
            assert (t.download() == orc.eq_evals(p)).all()

    assert _eq_launches(ctx, read) == 1
    assert _eq_launches(ctx, read) == 0


@pytest.mark.parametrize("n", [8, 12, 16])
def test_products_with_a_table_each(dp, ctx, orc, n):
    f, g, points = rand_base(1 << n, 1), rand_base(1 << n, 2), [rand_e2(n, 200 + i) for i in range(5)]
    mf, mg, host = ctx.mle_from_base(f), ctx.mle_from_base(g), [orc.embed_base(f), orc.embed_base(g)]
    tables = ctx.eq_build_many(points)

    def prove():
        for t, p in zip(tables, points):
            _prove(dp, ctx, orc, n, [mf, mg, t], host + [orc.eq_evals(p)], [(ONE, [0, 1, 2])])

    assert _eq_launches(ctx, prove) == 1


def test_some_gone_and_some_read_before(dp, ctx, orc):
    points = [rand_e2(m, 300 + i) for i, m in enumerate((9, 9, 9, 9, 17, 9, 10))]
    tables = ctx.eq_build_many(points)
    tables[1].free()
    # a sum over products of eq tables reads entries of three of them
    _prove(dp, ctx, orc, 9, [tables[0], tables[2], tables[3]], [orc.eq_evals(points[i]) for i in (0, 2, 3)], [(ONE, [0, 1]), (ONE, [1, 2]), (ONE, [0, 0, 2])])
    # ... a product takes one of these in closed form, and then one that nothing has read
    f = rand_e2(1 << 9, 310)
    for i in (2, 5):
        _prove(dp, ctx, orc, 9, [ctx.mle_from_ext2(f), tables[i]], [f, orc.eq_evals(points[i])], [(ONE, [0, 1])])
    view = tables[6].view(512, 9)
    assert (view.download() == orc.eq_evals(points[6])[512:]).all()
    for i in (0, 2, 3, 4, 5, 6):
        assert (tables[i].download() == orc.eq_evals(points[i])).all()


def test_more_tables_than_a_launch_stages(ctx, orc):
    points = [rand_e2(8, 400 + i) for i in range(300)]
    tables = ctx.eq_build_many(points)
    for i in (299, 0, 137):
        assert (tables[i].download() == orc.eq_evals(points[i])).all()
