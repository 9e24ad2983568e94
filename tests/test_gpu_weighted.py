"""Sums over two or three eq factors, each times a polynomial of its own over shared tables (what ties an activation to its lookups,
zkml/src/lookup/operation/inputs/variant.rs:222-348, written out as terms), against the CPU checker: sizes around the edges of the
launches (a sum of one variable, all rounds resident, one launch before the resident ones, factored weights), base and extension
tables, rounds that evaluate t = 1, and no room for resident launches."""
import importlib
import time

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


def _instance(dp, ctx, orc, n, kinds, polys, seed, zero_at=(), one_at=()):
    """polys: one per eq factor, a list of the table lists of its terms; kinds: a letter a table (b, e); zero_at, one_at: those coordinates
    of the eq factors' points"""
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
        for j in one_at:
            point[j] = (1, 0)
        dev.append(ctx.eq_build(point))
        host.append(orc.eq_evals(point))
        coeffs = [np.array(c, dtype=np.uint64) for c in ([1, 0], [dp.P - 1, 0], [12345, 0])]
        for k, tabs in enumerate(poly):
            terms.append((coeffs[k] if k < 3 and g == 0 else rand_e2(1, seed + 70 + 10 * g + k)[0], list(tabs) + [len(kinds) + g]))
    return dev, host, terms


def _prove(dp, ctx, orc, n, kinds, polys, seed, zero_at=(), claimed=False):
    dev, host, terms = _instance(dp, ctx, orc, n, kinds, polys, seed, zero_at)
    tr, otr = dp.Transcript(b"weighted"), orc.OracleTranscript(b"weighted")
    oproof, opoint, ofinals = orc.sc_prove(n, host, terms, otr)
    claim = orc.e2_add(oproof[0, 0], oproof[0, 1]) if claimed else None
    proof, point, finals = ctx.sumcheck_prover(n, dev, terms, claim=claim)(tr) if claimed else ctx.sumcheck_prove(n, dev, terms, tr)
    assert (proof == oproof).all() and (point == opoint).all() and (finals == ofinals).all() and tr.state() == otr.state()


LINKING = [[[0], [0, 1, 1], [1, 1], [1]], [[0], [1]]]
THREE = [[[0, 1, 2, 2], [2, 3], [], [3]], [[0, 3], [1]], [[2], []]]
TWO_QUADRATIC = [[[0, 1], [0]], [[1, 1], [0]]]
THREE_LOW = [[[0, 1], [2]], [[0], [1]], [[2], []]]  # (three factors whose sums leave room for trips of two rounds)


@pytest.mark.parametrize("n", [1, 2, 5, 9, 13, 16, 17, 18])
def test_two_factors(dp, ctx, orc, n):
    _prove(dp, ctx, orc, n, "bb", LINKING, 100 + n)
    _prove(dp, ctx, orc, n, "be", LINKING, 300 + n)


@pytest.mark.parametrize("n", [1, 4, 10, 17])
def test_three_factors(dp, ctx, orc, n):
    _prove(dp, ctx, orc, n, "beeb", THREE, 500 + n)
    _prove(dp, ctx, orc, n, "bb", TWO_QUADRATIC, 600 + n)


@pytest.mark.parametrize("n", [1, 2, 5, 9, 13, 17])
def test_three_factors_in_trips_of_two_rounds(dp, ctx, orc, n):
    _prove(dp, ctx, orc, n, "beb", THREE_LOW, 1000 + n)


@pytest.mark.parametrize("zero_at", [(), (0,), (1,), (2,)])
@pytest.mark.parametrize("kinds,polys", [("be", LINKING), ("bb", TWO_QUADRATIC), ("beeb", THREE), ("bb", LINKING[:1])])
def test_lanes_that_take_several_pairs(dp, ctx, orc, kinds, polys, zero_at):
    # 2^20 entries: up to three pairs a lane in the first round, factored weights in the first four, folded from the second on; rounds that evaluate t = 1
    # unfolded and folded
    _prove(dp, ctx, orc, 20, kinds, polys, 1100, zero_at)


@pytest.mark.parametrize("n", [3, 8, 13, 18])
def test_claim_known_before_round_one(dp, ctx, orc, n):
    _prove(dp, ctx, orc, n, "be", LINKING, 1200 + n, claimed=True)
    _prove(dp, ctx, orc, n, "beeb", THREE, 1300 + n, zero_at=(0,), claimed=True)
    _prove(dp, ctx, orc, n, "beb", THREE_LOW, 1400 + n, zero_at=(1,), claimed=True)


@pytest.mark.parametrize("kinds,polys", [("be", LINKING), ("beb", THREE_LOW), ("beeb", THREE), ("be", LINKING[:1])])
@pytest.mark.parametrize("n,at", [(8, 0), (8, 1), (8, 2), (8, 3), (19, 0), (19, 1), (19, 2)])
def test_challenge_that_makes_the_eq_factors_vanish(dp, ctx, orc, kinds, polys, n, at):
    # the points' coordinate `at` is 1 and so is nothing of eq(rho, .) left at the challenge 0: the messages that follow take p(1) from a first factor of scalar zero,
    # and a launch made ahead that leaves t = 1 out is not the one that is needed
    dev, tables, terms = _instance(dp, ctx, orc, n, kinds, polys, 1500 + n + at, one_at=(at,))
    s, challenge = ctx.session(n, dev, terms), None
    for j in range(n):
        message = orc.sc_round_poly(n - j, tables, [n - j] * len(tables), terms)
        assert (s.round(challenge) == message).all(), j
        challenge = np.zeros(2, dtype=np.uint64) if j == at else rand_e2(1, 1600 + j)[0]
        tables = [orc.mle_fix_low(t, challenge[None]) for t in tables]
    assert (s.finish(challenge) == np.concatenate([t.reshape(1, 2) for t in tables])).all()


@pytest.mark.parametrize("kinds,polys", [("be", LINKING), ("beeb", THREE)])
@pytest.mark.parametrize("how", ["other call", "slow caller"])
def test_launch_made_ahead_steps_aside(dp, ctx, orc, kinds, polys, how):
    # rounds 1 .. 3 of 19 variables (more than 2^15 pairs) are launches, the rest resident: before each of them has its challenge another call needs the context, or the caller
    # takes longer than the launch waits
    n = 19
    dev, host, terms = _instance(dp, ctx, orc, n, kinds, polys, 1700)
    proof, point, finals = orc.sc_prove(n, host, terms, orc.OracleTranscript(b"aside"))
    for after in (1, 2, 3):
        s, challenge = ctx.session(n, dev, terms), None
        for j in range(n):
            assert (s.round(challenge) == proof[j]).all(), (after, j)
            challenge = point[j]
            if j + 1 == after and how == "other call":
                assert (ctx.eq_build(point[:3]).download() == orc.eq_evals(point[:3])).all()
            elif j + 1 == after:
                time.sleep(0.3)
        assert (s.finish(challenge) == finals).all()
        del s


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
