"""Sums of products that share factors, which run over fewer tables (one product with a combined table, or one product per eq
table), against the CPU checker: eq tables on both sides of the row length (2^11) and of the sizes whose rows need two and
three small tables, base and extension tables, zero-padded tables down to one entry, constants, stated sums, tables no term
uses, and sums on either side of the rule that decides (2^16 and 2^17 entries, 32 and 33 tables)."""
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


class Sum:
    def __init__(self, ctx, orc, n, seed, marked=False):
        # (marked: full-size tables are zero-padded to their own size, as the opening of committed polynomials passes all of its tables)
        self.ctx, self.orc, self.n, self.seed, self.rng, self.marked = ctx, orc, n, seed, py_rng(seed), marked
        self.gpu, self.host, self.terms, self.k = [], [], [], 0

    def _pad(self, v, h, m):
        if m < self.n or self.marked:
            h = h.zero_pad(self.n)
        if m < self.n:
            v = np.concatenate([v, np.zeros(((1 << self.n) - (1 << m), 2), dtype=np.uint64)])
        self.gpu.append(h)
        self.host.append(v)
        return len(self.gpu) - 1

    def table(self, m=None, base=False):
        m = self.n if m is None else m
        self.k += 1
        v = rand_base(1 << m, self.seed * 100 + self.k) if base else rand_e2(1 << m, self.seed * 100 + self.k)
        return self._pad(self.orc.embed_base(v) if base else v, self.ctx.mle_from_base(v) if base else self.ctx.mle_from_ext2(v), m)

    def eqs(self, ms):
        points = [rand_e2(m, self.seed * 100 + 50 + self.k + i) for i, m in enumerate(ms)]
        self.k += len(ms)
        return [self._pad(self.orc.eq_evals(p), h, m) for p, h, m in zip(points, self.ctx.eq_build_many(points), ms)]

    def coeff(self):
        return np.array([self.rng.randrange(1, 1 << 62), self.rng.randrange(0, 1 << 62)], dtype=np.uint64)

    def term(self, *factors):
        self.terms.append((self.coeff(), list(factors)))

    def check(self, dp):
        for claimed in (False, True):
            tr, otr = dp.Transcript(b"c"), self.orc.OracleTranscript(b"c")
            oproof, opoint, ofinals = self.orc.sc_prove(self.n, self.host, self.terms, otr)
            if claimed:
                claim = self.orc.e2_add(oproof[0][0], oproof[0][1])
                got = self.ctx.sumcheck_prover(self.n, self.gpu, self.terms, claim=claim)(tr)
            else:
                got = self.ctx.sumcheck_prove(self.n, self.gpu, self.terms, tr)
            assert (got[0] == oproof).all() and (got[1] == opoint).all() and (got[2] == ofinals).all()
            assert tr.state() == otr.state()


@pytest.mark.parametrize("n,k,base", [(1, 2, False), (2, 6, True), (3, 3, True), (3, 4, False), (5, 4, False), (5, 3, True), (6, 4, False), (7, 2, False), (10, 5, True), (11, 2, False), (12, 4, True), (16, 3, True),
                                      (17, 2, False), (18, 9, True), (20, 4, True)])
def test_claims_on_one_table(dp, ctx, orc, n, k, base):
    s = Sum(ctx, orc, n, 1000 + 10 * n + k)
    x = s.table(base=base)
    for e in s.eqs([n] * k):
        s.term(x, e) if e % 2 else s.term(e, x)
    s.check(dp)


@pytest.mark.parametrize("n", [16, 17, 18])
def test_a_table_times_several(dp, ctx, orc, n):
    s = Sum(ctx, orc, n, 2000 + n)
    x, y, z = s.table(base=True), s.table(), s.table(base=True)
    unused = s.table(base=True)
    s.term(x, y)
    s.term(z, x)
    s.term(x, y)
    s.terms.append((s.coeff(), []))  # a constant
    assert unused == 3
    s.check(dp)


@pytest.mark.parametrize("n,ms", [(4, [0, 1, 4]), (9, [9, 3]), (12, [11, 12, 5, 0]), (13, [10, 12, 11, 2])])
def test_zero_padded_tables_times_one(dp, ctx, orc, n, ms):
    s = Sum(ctx, orc, n, 3000 + n)
    e = s.eqs([n])[0]
    for i, m in enumerate(ms):
        s.term(s.table(m, base=i % 2 == 1), e)
    s.check(dp)


@pytest.mark.parametrize("n,polys,claims", [(5, [5, 5, 3, 3, 0], 2), (10, [10] * 28, 5), (10, [10] * 27, 5), (11, [11, 11, 10, 10, 10, 7, 0], 3), (14, [14, 12, 13], 3)])
def test_claims_at_several_points(dp, ctx, orc, n, polys, claims):
    # every polynomial at one point of its own number of variables, or at two of them (28 + 5 tables are more than a launch takes)
    s = Sum(ctx, orc, n, 4000 + n + len(polys))
    tables = [s.table(m, base=i % 3 == 2) for i, m in enumerate(polys)]
    sizes = sorted(set(polys), reverse=True)
    eqs = {m: s.eqs([m] * (1 + (claims - 1) // len(sizes))) for m in sizes}
    for i, (t, m) in enumerate(zip(tables, polys)):
        s.term(t, eqs[m][i % len(eqs[m])])
        if i % 4 == 1:
            s.term(eqs[m][(i + 1) % len(eqs[m])], t)
    used = {f for _, fs in s.terms for f in fs}
    for e in [e for m in sizes for e in eqs[m]]:
        if e not in used:
            s.term(tables[0], e)
    s.check(dp)


def test_session_given_up_and_errors(dp, ctx, orc):
    s = Sum(ctx, orc, 12, 5000)
    x = s.table(base=True)
    for e in s.eqs([12] * 3):
        s.term(x, e)
    se = ctx.session(s.n, s.gpu, s.terms)
    first = se.round(None)
    with pytest.raises(dp.DpsError):
        se.round(None)  # round 2 needs a challenge
    with pytest.raises(dp.DpsError):
        se.finish(rand_e2(1, 1)[0])  # 11 rounds to go
    se.abort()
    with pytest.raises(dp.DpsError):
        se.round(rand_e2(1, 2)[0])
    del se
    # rounds with another call on the context between them, from scratch, and a whole proof after it
    oproof, opoint, ofinals = orc.sc_prove(s.n, s.host, s.terms, orc.OracleTranscript(b"c"))
    assert (first == oproof[0]).all()
    s.check(dp)
    se = ctx.session(s.n, s.gpu, s.terms)
    chal = None
    for j in range(s.n):
        assert (se.round(chal) == oproof[j]).all()
        chal = opoint[j]
    assert (se.finish(chal) == ofinals).all()


# rows of 512 and of 1024 entries on either side of 2^18; descriptors beyond what the kernel arguments hold, read from the host's
# memory (up to 256 workgroups) and from a copy (2^19); more than 64 items of one table
@pytest.mark.parametrize("n,k", [(8, 3), (9, 4), (10, 70), (13, 66), (18, 20), (19, 14)])
def test_many_claims_on_one_table(dp, ctx, orc, n, k):
    s = Sum(ctx, orc, n, 6000 + 10 * n + k)
    x = s.table(base=True)
    for e in s.eqs([n] * k):
        s.term(x, e)
    s.check(dp)


# full-size tables at several points: combined up to eight points, as they stand beyond that while their groups of tables fit side by
# side, combined again where they do not (34 points) and for large tables
@pytest.mark.parametrize("n,polys,points", [(9, 40, 8), (9, 40, 9), (11, 60, 17), (8, 80, 34), (17, 40, 17)])
def test_claims_at_many_points(dp, ctx, orc, n, polys, points):
    s = Sum(ctx, orc, n, 8000 + n + points)
    tables = [s.table(base=i % 2 == 0) for i in range(polys)]
    eqs = s.eqs([n] * points)
    for i, t in enumerate(tables):
        s.term(t, eqs[i % points])
    s.check(dp)


# full-size tables that carry the mark of padding run like the others: resident launches for the products that are left (up to 16
# points; 17 as they stand, and from 2^12 entries on combined), and for a small sum as it stands
@pytest.mark.parametrize("n,polys,points", [(6, 40, 4), (10, 40, 8), (10, 60, 15), (10, 60, 16), (10, 60, 17), (11, 60, 17), (12, 60, 17), (7, 60, 16), (9, 12, 4)])
def test_marked_claims_at_several_points(dp, ctx, orc, n, polys, points):
    s = Sum(ctx, orc, n, 9000 + n + points, marked=True)
    tables = [s.table(base=i % 2 == 0) for i in range(polys)]
    eqs = s.eqs([n] * points)
    for i, t in enumerate(tables):
        s.term(t, eqs[i * points // polys])
    s.check(dp)
    ctx.profile(True)
    try:
        ctx.profile_reset()
        s.ctx.sumcheck_prove(s.n, s.gpu, s.terms, dp.Transcript(b"c"))
        resident = ctx.profile_read()["tail"]["launches"]
    finally:
        ctx.profile(False)
    assert (resident > 0) == (points <= 16), resident


def test_marked_products_of_one_table(dp, ctx, orc):
    s = Sum(ctx, orc, 13, 9500, marked=True)
    x, y = s.table(base=True), s.table()
    for e in s.eqs([13] * 2):
        s.term(x, e)
    s.term(x, y)
    s.check(dp)
