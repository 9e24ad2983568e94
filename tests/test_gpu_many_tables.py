"""Sums of several terms over more tables than a group of the multi-term kernels holds, and over tables of fewer variables,
through the resident launches: the numbers of tables and terms at which a launch still takes them and the next ones, sums of
one round and of a few, sums whose first rounds are launches of their own, tables one and several variables short (down to a
constant), and the same sums when no launch may wait on the GPU."""
import importlib

import numpy as np
import pytest

from util import py_rng, rand_base, rand_e2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dp():
    return importlib.import_module("deep-prove_amd")


@pytest.fixture(scope="module")
def ctx(dp):
    c = dp.Context(0)
    yield c
    c.close()


def _instance(ctx, orc, seed, table_vars, base, n_terms, max_deg):
    rng = py_rng(seed)
    gpu, host = [], []
    for k, m in enumerate(table_vars):
        if k in base:
            v = rand_base(1 << m, seed * 100 + k)
            gpu.append(ctx.mle_from_base(v))
            host.append(orc.embed_base(v))
        else:
            v = rand_e2(1 << m, seed * 100 + k)
            gpu.append(ctx.mle_from_ext2(v))
            host.append(v)
    terms = []
    for i in range(n_terms):
        # every table is in some term
        fs = [(i * max_deg + d) % len(table_vars) if i * max_deg + d < len(table_vars) + max_deg else rng.randrange(len(table_vars)) for d in range(max_deg)]
        coeff = np.array([rng.randrange(1, 1 << 62), rng.randrange(0, 1 << 62)], dtype=np.uint64)
        terms.append((coeff, fs))
    return gpu, host, terms


def _check(dp, ctx, orc, n, gpu, host, terms):
    tr, otr = dp.Transcript(b"many"), orc.OracleTranscript(b"many")
    proof, point, finals = ctx.sumcheck_prove(n, gpu, terms, tr)
    oproof, opoint, ofinals = orc.sc_prove(n, host, terms, otr)
    assert (proof == oproof).all() and (point == opoint).all() and (finals == ofinals).all()
    assert tr.state() == otr.state()


CASES = [
    # n, variables of the tables, base-field tables, terms, degree
    (6, [6] * 24, [0, 5], 12, 2),
    (8, [8] * 32, [], 16, 2),
    (8, [8] * 33, [], 17, 2),           # a table too many for a launch
    (9, [9] * 20, list(range(20)), 64, 3),
    (9, [9] * 20, [], 65, 3),           # a term too many
    (1, [1] * 18, [], 9, 2),
    (2, [2] * 17, [3], 9, 2),
    (12, [12] * 25, [], 15, 3),         # several workgroups
    (17, [17] * 9 + [16, 14, 3, 0], [0, 1], 9, 3),   # two groups of tables, the first rounds launches of their own
    (10, [10, 10, 9, 8, 5, 1, 0], [2, 5], 6, 3),
    (14, [14] * 6 + [13] * 6 + [12] * 4 + [7] * 4, [1, 8], 14, 3),
    (5, [4, 4, 3], [], 3, 2),           # no table has the sum's first variable
]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_many_tables_match_checker(dp, ctx, orc, case):
    n, table_vars, base, n_terms, deg = CASES[case]
    gpu, host, terms = _instance(ctx, orc, 700 + case, table_vars, base, n_terms, deg)
    _check(dp, ctx, orc, n, gpu, host, terms)
    _check(dp, ctx, orc, n, gpu, host, terms)


@pytest.mark.parametrize("case", [0, 8, 9, 10])
def test_many_tables_without_resident_launches(dp, ctx, orc, case):
    n, table_vars, base, n_terms, deg = CASES[case]
    gpu, host, terms = _instance(ctx, orc, 700 + case, table_vars, base, n_terms, deg)
    dp.set_resident_budget(0, 0)
    try:
        _check(dp, ctx, orc, n, gpu, host, terms)
    finally:
        dp.set_resident_budget(0, -1)


@pytest.mark.parametrize("case", [0, 1, 3, 7, 8, 9, 10, 11])
@pytest.mark.parametrize("budget", [1, 2, 5])
def test_many_tables_in_few_workgroups(dp, ctx, orc, case, budget):
    # the resident launch in as many workgroups as there are places, behind rounds that are launches: tables one and several variables short of its first round too
    n, table_vars, base, n_terms, deg = CASES[case]
    gpu, host, terms = _instance(ctx, orc, 700 + case, table_vars, base, n_terms, deg)
    dp.set_resident_budget(0, budget)
    try:
        _check(dp, ctx, orc, n, gpu, host, terms)
    finally:
        dp.set_resident_budget(0, -1)


@pytest.mark.parametrize("tables,n_terms,eq,short", [(16, 24, False, False), (17, 24, False, False), (16, 25, False, False), (16, 24, True, False),
                                                     (17, 25, True, False), (4, 3, True, True), (16, 24, False, True)])
def test_sizes_of_the_arguments(dp, ctx, orc, tables, n_terms, eq, short):
    """A launch's arguments have room for 16 tables and 24 terms or for 32 and 64, and only the larger ones take tables of fewer
    variables: sums on both sides, in one workgroup and in several."""
    for n, deg in ((5, 2), (12, 2 if eq else 3)):
        table_vars = [n] * tables
        if short:
            table_vars[1] = n - 2
        gpu, host, terms = _instance(ctx, orc, 900 + tables + n_terms + n, table_vars, [0], n_terms, deg)
        if eq:
            rho = rand_e2(n, 950 + n)
            gpu.append(ctx.eq_build(rho))
            host.append(orc.eq_evals(rho))
            terms = [(c, fs + [tables]) for c, fs in terms]
        _check(dp, ctx, orc, n, gpu, host, terms)
