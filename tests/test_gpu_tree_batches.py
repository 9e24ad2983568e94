"""Fraction trees built together, against the CPU checker: more trees than a launch takes, trees whose larger levels are launches of
their own beside trees of one level, several columns, multiplicities."""
import importlib

import numpy as np
import pytest

from util import rand_base, rand_e2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,columns,table", [((2,), 1, False), ((3, 2), 2, True), ((13, 12, 12, 11, 3, 3, 2, 2), 1, False),
                                                 ((12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2), 2, False), ((6,) * 17, 1, True)])
def test_batches(orc, sizes, columns, table):
    dp = importlib.import_module("deep-prove_amd")
    ctx = dp.Context(0)
    host, dev = [], []
    for i, n in enumerate(sizes):
        cols = [rand_base(1 << n, 7000 + 10 * i + k) for k in range(columns)]
        numer = rand_base(1 << n, 7500 + i) if table else None
        c, beta = rand_e2(1, 7600 + i)[0], rand_e2(1, 7700 + i)[0]
        host.append(dict(cols=cols, numer=numer, c=c, beta=beta))
        dev.append(dict(cols=[ctx.mle_from_base(x) for x in cols], numer=None if numer is None else ctx.mle_from_base(numer), c=c, beta=beta))
    tr, otr = dp.Transcript(), orc.OracleTranscript()
    want = orc.logup_batch_prove(host, otr)
    got = dp.logup_batch_prove(ctx, dev, tr)
    assert got.shape == want.shape and (got == want).all() and tr.state() == otr.state()
    ctx.close()


def test_one_bad_tree_refuses_the_batch(orc):
    dp = importlib.import_module("deep-prove_amd")
    ctx = dp.Context(0)
    c, beta = rand_e2(1, 1)[0], rand_e2(1, 2)[0]
    good = dict(cols=[ctx.mle_from_base(rand_base(16, 3))], numer=None, c=c, beta=beta)
    bad = dict(good, c=np.array([dp.P, 0], dtype=np.uint64))
    with pytest.raises(Exception):
        dp.logup_batch_prove(ctx, [good, bad], dp.Transcript())
    ref = orc.logup_batch_prove([dict(cols=[rand_base(16, 3)], numer=None, c=c, beta=beta)], orc.OracleTranscript())
    assert (dp.logup_batch_prove(ctx, [good], dp.Transcript()) == ref).all()
    ctx.close()
