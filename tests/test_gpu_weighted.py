"""Sums over two or three eq factors, each times a polynomial of its own over shared tables (what ties an activation to its lookups,
zkml/src/lookup/operation/inputs/variant.rs:222-348, written out as terms), against the CPU checker: sizes around the edges of the
launches (a sum of one variable, all rounds resident, one launch before the resident ones, factored weights), base and extension
tables, rounds that evaluate t = 1, and no room for resident launches."""
import importlib

import numpy as np
import pytest

from util import rand_base, rand_e2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dp():
    return importlib.import_module("deep-prove_amd")


@pytest.fixture(scope="module")
def ctx(dp):
    c = dp.Context(0)
    yield c
    c.close()


def _prove(dp, ctx, orc, n, kinds, polys, seed, zero_at=()):
    """polys: one per eq factor, a list of the table lists of its terms; kinds: a letter a table (b, e)"""
    dev, host = [], []
    for i, k in enumerate(kinds):
        x = rand_base(1 << n, seed + i) if k == "b" else rand_e2(1 << n, seed + i)
        dev.append(ctx.mle_from_base(x) if k == "b" else ctx.mle_from_ext2(x))
        host.append(orc.embed_base(x) if k == "b" else x)
    terms = []
    for g, poly in enumerate(polys):
        point = rand_e2(n, seed + 50 + g)
        for j in zero_at:
            point[j] = 0
        dev.append(ctx.eq_build(point))
        host.append(orc.eq_evals(point))
        coeffs = [np.array(c, dtype=np.uint64) for c in ([1, 0], [dp.P - 1, 0], [12345, 0])]
        for k, tabs in enumerate(poly):
            terms.append((coeffs[k] if k < 3 and g == 0 else rand_e2(1, seed + 70 + 10 * g + k)[0], list(tabs) + [len(kinds) + g]))
    tr, otr = dp.Transcript(b"weighted"), orc.OracleTranscript(b"weighted")
    proof, point, finals = ctx.sumcheck_prove(n, dev, terms, tr)
    oproof, opoint, ofinals = orc.sc_prove(n, host, terms, otr)
    assert (proof == oproof).all() and (point == opoint).all() and (finals == ofinals).all() and tr.state() == otr.state()


LINKING = [[[0], [0, 1, 1], [1, 1], [1]], [[0], [1]]]
THREE = [[[0, 1, 2, 2], [2, 3], [], [3]], [[0, 3], [1]], [[2], []]]


@pytest.mark.parametrize("n", [1, 2, 5, 9, 13, 16, 17, 18])
def test_two_factors(dp, ctx, orc, n):
    _prove(dp, ctx, orc, n, "bb", LINKING, 100 + n)
    _prove(dp, ctx, orc, n, "be", LINKING, 300 + n)


@pytest.mark.parametrize("n", [1, 4, 10, 17])
def test_three_factors(dp, ctx, orc, n):
    _prove(dp, ctx, orc, n, "beeb", THREE, 500 + n)
    _prove(dp, ctx, orc, n, "bb", [[[0, 1], [0]], [[1, 1], [0]]], 600 + n)


@pytest.mark.parametrize("n,zero_at", [(6, (0, 3)), (11, (2,)), (17, (0, 1, 5))])
def test_rounds_that_evaluate_at_one(dp, ctx, orc, n, zero_at):
    _prove(dp, ctx, orc, n, "bb", LINKING, 700 + n, zero_at)
    _prove(dp, ctx, orc, n, "beeb", THREE, 800 + n, zero_at)


def test_without_resident_launches(dp, orc):
    ctx = dp.Context(0)
    dp.set_resident_budget(0, 0)
    try:
        for n in (3, 12, 18):
            _prove(dp, ctx, orc, n, "bb", LINKING, 900 + n)
            _prove(dp, ctx, orc, n, "beeb", THREE, 950 + n)
    finally:
        dp.set_resident_budget(0, -1)
        ctx.close()
