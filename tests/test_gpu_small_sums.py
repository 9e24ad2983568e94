"""Sums of several products whose rounds are all resident, against the CPU checker: pairs and terms around the sizes at which a sum is
cut into one more workgroup, with a common eq factor and without, tables of all kinds."""
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


def _prove(dp, ctx, orc, n, n_terms, with_eq):
    dev, host, terms = [], [], []
    for i in range(2 * n_terms):
        base = i % 3 == 0
        x = rand_base(1 << n, 1000 * n + i) if base else rand_e2(1 << n, 1000 * n + i)
        dev.append(ctx.mle_from_base(x) if base else ctx.mle_from_ext2(x))
        host.append(orc.embed_base(x) if base else x)
    if with_eq:
        point = rand_e2(n, 77 + n)
        dev.append(ctx.eq_build(point))
        host.append(orc.eq_evals(point))
    for k in range(n_terms):
        coeff = np.array([1, 0], dtype=np.uint64) if k % 2 else rand_e2(1, 5 * n + k)[0]
        terms.append((coeff, [2 * k, 2 * k + 1] + ([2 * n_terms] if with_eq else [])))
    tr, otr = dp.Transcript(b"small sums"), orc.OracleTranscript(b"small sums")
    proof, point, finals = ctx.sumcheck_prove(n, dev, terms, tr)
    oproof, opoint, ofinals = orc.sc_prove(n, host, terms, otr)
    assert (proof == oproof).all() and (point == opoint).all() and (finals == ofinals).all() and tr.state() == otr.state(), n


@pytest.mark.parametrize("n_terms", [1, 2, 3, 8, 16])
@pytest.mark.parametrize("with_eq", [False, True])
def test_sums_of_products(dp, ctx, orc, n_terms, with_eq):
    # (the first round's pairs times terms from a quarter of a workgroup's share to more than 32 workgroups take at the smallest one)
    for n in (3, 4, 6, 7, 8, 9, 10, 11, 12, 13):
        _prove(dp, ctx, orc, n, n_terms, with_eq)


@pytest.mark.parametrize("n_terms", [1, 3, 16])
@pytest.mark.parametrize("with_eq", [False, True])
def test_no_place_for_the_resident_launch(dp, orc, n_terms, with_eq):
    # every round is a launch of its own, whose descriptors the session has not worked out when it began
    ctx = dp.Context(0)
    dp.set_resident_budget(0, 0)
    try:
        for n in (1, 3, 5, 8, 11):
            _prove(dp, ctx, orc, n, n_terms, with_eq)
    finally:
        dp.set_resident_budget(0, -1)
        ctx.close()
