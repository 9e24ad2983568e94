"""Partial evaluations of tensors in one launch, against the CPU checker: contractions at the edges of what a wavefront, a
workgroup's weights and a step of a row hold (63 .. 65, 255 .. 257, 511 .. 513 values), outputs on either side of the tile of 64
and of the size below which lanes go over the contracted axis (31, 32), shares of one tile or row between workgroups, rows that
need padding, every kind of entry, and calls without an axis to contract."""
import importlib

import numpy as np
import pytest

from util import rand_base, rand_e2, rand_i64

pytestmark = pytest.mark.gpu
C_, O_, S_ = 0, 1, 2


@pytest.fixture(scope="module")
def dp():
    return importlib.import_module("deep-prove_amd")


@pytest.fixture(scope="module")
def ctx(dp):
    c = dp.Context(0)
    yield c
    c.close()


def _pad(shape):
    return [1 << max(0, (d - 1).bit_length()) for d in shape]


def _padded(t):
    out = np.zeros(_pad(t.shape), dtype=np.int64)
    out[tuple(slice(0, d) for d in t.shape)] = t
    return out


CASES = (
    # lanes over the outputs: contracted axis, then outputs
    [((k, c), [O_, C_]) for k in (1, 2, 31, 32, 33, 255, 257, 700) for c in (32, 65)] +
    # lanes over the contracted axis
    [((c, k), [C_, O_]) for k in (1, 2, 63, 65, 511, 512, 513, 2049, 5000) for c in (1, 3, 31)] +
    # one and two outputs of a long row (several workgroups each, more than 64 steps), more rows than share a workgroup
    [((1, 70000), [C_, O_]), ((70000,), [O_]), ((2, 300000), [S_, O_]), ((4100, 600), [C_, O_]), ((4097, 33), [C_, O_]), ((70000, 31), [O_, C_])] +
    # more tiles than are shared, stacked rows with padding, several axes
    [((3, 40, 20000), [S_, O_, C_]), ((12, 197, 197), [S_, O_, C_]), ((12, 197, 64), [S_, C_, O_]), ((3, 5, 7, 9), [O_, S_, O_, C_]), ((33, 2, 40), [O_, C_, O_])] +
    # tiles that are shared between workgroups, more than one a compute unit of them (257, 266), and that are not (few values; 1025)
    [((512, 16448), [O_, C_]), ((520, 17000), [O_, C_]), ((300, 30000), [O_, C_]), ((40, 65600), [O_, C_])] +
    # a thread an output: on both sides of 4096 outputs a value, with rows to pad, several axes, more outputs than a pass
    [((1, 4095), [O_, C_]), ((1, 4096), [O_, C_]), ((2, 8191), [O_, C_]), ((2, 8193), [O_, C_]), ((9, 36865), [O_, C_]), ((30, 131000), [O_, C_]),
     ((33, 135300), [O_, C_]), ((3, 600007), [O_, C_]), ((600, 4, 40), [C_, O_, C_]), ((300, 2, 33), [S_, O_, C_])] +
    # several outputs a wavefront: on both sides of 4096 outputs, of 64, 128 and 256 values, and adjacent outputs
    [((c, k), [C_, O_]) for c, k in ((4095, 64), (4096, 64), (4097, 1), (70001, 64), (4099, 65), (4096, 128), (5000, 129), (4097, 256), (4096, 257))] +
    [((2050, 100, 2), [S_, O_, C_]), ((137, 60, 31), [C_, O_, C_])] +
    # a second contraction, of the first one's extension entries, over rows that several workgroups share and over tiles that they share
    [((2, 3000, 5), [C_, O_, O_]), ((1, 70000, 3), [C_, O_, O_]), ((3, 700, 40), [O_, O_, C_]), ((300, 40, 3), [O_, C_, O_])] +
    # one, two and four wavefronts an output of several steps
    [((c, k), [C_, O_]) for c, k in ((300, 513), (2049, 2049), (2048, 2049), (3001, 1100), (4097, 513), (4095, 513))] +
    # nothing to contract
    [((3, 5, 5000), [S_, C_, C_]), ((1,), [C_]), ((768,), [C_]), ((3, 5, 100), [S_, C_, C_])]
)


@pytest.mark.parametrize("case", range(len(CASES)))
def test_shapes(ctx, orc, case):
    shape, kinds = CASES[case]
    t, pd = rand_i64(shape, 500 + case, -32768, 32767), _pad(shape)
    points = [rand_e2(max(0, (p - 1).bit_length()), 600 + 10 * case + a) if k == O_ else None for a, (p, k) in enumerate(zip(pd, kinds))]
    want = orc.partial_eval(_padded(t), pd, list(shape), kinds, points)
    for make in (ctx.tensor_from_i64, ctx.tensor_from_i16):
        for _ in range(2):  # (the second call finds the counters the first one left)
            got = ctx.partial_eval(make(t), pd, list(shape), kinds, points)
            assert len(got) == want.shape[0]
            for g, w in zip(got, want):
                assert (g.download() == w).all()


@pytest.mark.parametrize("rows,cols", [(4, 8), (64, 32), (2, 1024), (512, 64), (4, 16384), (4096, 8), (8192, 64), (4096, 256)])
@pytest.mark.parametrize("first", [True, False])
def test_field_tables(ctx, orc, rows, cols, first):
    """tables of either field, against the definition: sum_k in[k] eq(point, k)"""
    kinds = [O_, C_] if first else [C_, O_]
    k = rows if first else cols
    point = rand_e2(k.bit_length() - 1, 71)
    eq = orc.eq_evals(point)
    for ext in (False, True):
        v = rand_e2(rows * cols, 72) if ext else orc.embed_base(rand_base(rows * cols, 73))
        table = ctx.mle_from_ext2(v) if ext else ctx.mle_from_base(v[:, 0].copy())
        got = ctx.partial_eval(table, [rows, cols], [rows, cols], kinds, [point if x == O_ else None for x in kinds])[0].download()
        grid = v.reshape(rows, cols, 2)
        for i in (0, 1, (cols if first else rows) - 1):
            line = grid[:, i] if first else grid[i]
            want = np.zeros(2, dtype=np.uint64)
            for a, b in zip(line, eq):
                want = orc.e2_add(want, orc.e2_mul(a, b))
            assert (got[i] == want).all()


@pytest.mark.parametrize("rows,cols", [(1, 4096), (2, 65536), (8, 8192), (1, 1 << 18)])
@pytest.mark.parametrize("ext", [False, True])
def test_long_rows_of_field_tables(ctx, orc, rows, cols, ext):
    """rows that several workgroups share, of base and extension entries: a row's value is its evaluation at the point"""
    point = rand_e2(cols.bit_length() - 1, 81)
    v = rand_e2(rows * cols, 82 + rows) if ext else orc.embed_base(rand_base(rows * cols, 83 + rows))
    table = ctx.mle_from_ext2(v) if ext else ctx.mle_from_base(v[:, 0].copy())
    got = ctx.partial_eval(table, [rows, cols], [rows, cols], [C_, O_], [None, point])[0].download()
    for r in range(rows):
        assert (got[r] == orc.mle_evaluate(v[r * cols:(r + 1) * cols], point)).all()


@pytest.mark.parametrize("n,rest", [(12, 0), (14, 2), (17, 4), (18, 1), (13, 5), (16, 15), (18, 13)])
@pytest.mark.parametrize("ext", [False, True])
def test_fix_high_down_to_a_few_entries(ctx, orc, n, rest, ext):
    v = rand_e2(1 << n, 91 + n) if ext else orc.embed_base(rand_base(1 << n, 92 + n))
    point = rand_e2(n - rest, 93 + rest)
    table = ctx.mle_from_ext2(v) if ext else ctx.mle_from_base(v[:, 0].copy())
    got = table.fix_high(point).download()
    assert (got == orc.mle_fix_high(v, point)).all()


def test_points_are_checked(dp, ctx):
    t = ctx.tensor_from_i64(rand_i64((4, 4), 1))
    bad = rand_e2(2, 2)
    bad[1][0] = dp.P
    with pytest.raises(dp.DpsError):
        ctx.partial_eval(t, [4, 4], [4, 4], [O_, C_], [bad, None])
