"""dps_mle_evaluate against the CPU checker on both sides of every size at which its kernel changes what it does: tables
shorter than a row of 2^11 entries, one row, a row per workgroup, several rows per workgroup, and the first size (2^24)
whose rows need a third small table of the point's coordinates."""
import importlib

import numpy as np
import pytest

from util import rand_base, rand_e2, rand_i64

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dp():
    return importlib.import_module("deep-prove_amd")


@pytest.fixture(scope="module")
def ctx(dp):
    c = dp.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("n", [0, 1, 2, 8, 9, 10, 11, 12, 16, 17, 18, 21, 22])
def test_evaluate_every_kind(ctx, orc, n):
    pt = rand_e2(n, 41000 + n)
    ext, base = rand_e2(1 << n, 41100 + n), rand_base(1 << n, 41200 + n)
    assert (ctx.mle_from_ext2(ext).evaluate(pt) == orc.mle_evaluate(ext, pt)).all()
    assert (ctx.mle_from_base(base).evaluate(pt) == orc.mle_evaluate(orc.embed_base(base), pt)).all()
    v = rand_i64(1 << n, 41300 + n, -32768, 32767)
    want = orc.mle_evaluate(orc.embed_i64(v), pt)
    assert (ctx.tensor_from_i64(v).evaluate(pt) == want).all()
    assert (ctx.tensor_from_i16(v).evaluate(pt) == want).all()


@pytest.mark.parametrize("n", [23, 24, 25])
def test_evaluate_large(ctx, orc, n):
    base, pt = rand_base(1 << n, 42000 + n), rand_e2(n, 42100 + n)
    assert (ctx.mle_from_base(base).evaluate(pt) == orc.mle_evaluate(orc.embed_base(base), pt)).all()


def test_evaluate_views_and_eq_tables(ctx, orc):
    # a view that starts in the middle of a row of its parent; an eq table whose entries nobody has read
    whole, pt = rand_e2(1 << 13, 43001), rand_e2(9, 43002)
    assert (ctx.mle_from_ext2(whole).view(514, 9).evaluate(pt) == orc.mle_evaluate(whole[514:514 + 512], pt)).all()
    rho, z = rand_e2(20, 43003), rand_e2(20, 43004)
    eq = ctx.eq_build(rho)
    want = orc.identity_eval(rho, z)
    assert (eq.evaluate(z) == want).all()
    half = eq.view(1 << 19, 19)  # reads entries: the table is built
    assert (half.evaluate(z[:19]) == orc.mle_evaluate(orc.eq_evals(rho)[1 << 19:], z[:19])).all()
    assert (eq.evaluate(z) == want).all()
    with pytest.raises(Exception):
        eq.evaluate(rand_e2(19, 1))
