"""The proofs a layer prover asks of this library, as cases to be timed.

Every case is one statement proved through the package's public entry points the way a prover of a quantised
model calls them: tables and weights lie on the GPU before the proof (or, where the case says so, the tensors come from
host memory), the claim's point is new for every proof, and one call of `run` is the whole proof: eq tables, partial
evaluations, every round with the transcript on the host, final evaluations.  Proofs are integers, so they are compared
bit for bit.

Sizes are the ones of the repository's benchmark and tests (products of 2^24 entries, [512 x 768] by [768 x 3072]
layers, 12 heads of 64, 2^22 lookups into a 2^16-entry table, openings of 14 polynomials, a [512 x 3072] activation), down to
the single row of a decoding step, and ragged sizes in between.
"""
import importlib

import numpy as np

dp = importlib.import_module("deep-prove_amd")

ONE = np.array([1, 0], dtype=np.uint64)
_context = None


def context():
    """The one context a single-threaded prover keeps for its life."""
    global _context
    if _context is None:
        _context = dp.Context(0)
    return _context


# ---- the cases (lists of sizes are written as texts) ----


def _text(sizes):
    return " ".join(str(x) for x in sizes)


def _sizes(text):
    return [int(x) for x in text.split()]


def listed():
    return [
        # a gate times an activation of one token (1024 wide): the smallest proof a layer asks for, all of it latency
        dict(name="hadamard_n10", kind="product", n=10, eq=True, tables="quantised quantised", claimed=True),
        # the same layer over a prompt of 512 tokens
        dict(name="hadamard_n19", kind="product", n=19, eq=True, tables="quantised quantised", claimed=True),
        # the benchmark statement: eq f g over 2^24 uniform base-field entries, the sum not known beforehand
        dict(name="hadamard_n24", kind="product", n=24, eq=True, tables="base base", claimed=False),
        # decoding: one token through an MLP up-projection, weights resident in 16-bit storage
        dict(name="matmul_decode", kind="matmul", rows=1, inner=768, cols=3072, outputs=1, bias=True, bits=16, host=False),
        # prefill of the same projection with 64-bit tensors resident on the device
        dict(name="matmul_prefill", kind="matmul", rows=512, inner=768, cols=3072, outputs=1, bias=False, bits=64, host=False),
        # a ragged prompt through three projections with biases, the tensors handed over from host memory: the three
        # claims on the input are merged by a second sumcheck
        dict(name="qkv_from_host", kind="matmul", rows=300, inner=768, cols=768, outputs=3, bias=True, bits=64, host=True),
        # both products of an attention layer, 12 heads over a ragged prompt
        dict(name="attention_12", kind="attention", heads=12, queries=197, keys=197, width=64, bits=64),
        # the lookups of a short prompt: five batches of different sizes into a small table; the prover verifies its own
        # proofs before it hands them out, which is the path's other direction
        dict(name="lookups_small", kind="lookup", logs="11 10 9 8 7", columns=1, log_table=8, verify=True),
        # the benchmark's lookup argument
        dict(name="lookups_22", kind="lookup", logs="22", columns=2, log_table=16, verify=False),
        # the claims of 14 committed polynomials of 2^10 .. 2^15 entries, in chunks of 2^11, batched for opening (those smaller than
        # a chunk are padded with zeros by the sumcheck that reads them)
        dict(name="opening_14", kind="opening", sizes="13 15 10 14 12 11 13 10 12 11 13 10 12 13", chunk=11),
        # the activation behind an MLP up-projection, tied to its lookups
        dict(name="linking_512x3072", kind="linking", variant="standard", shape="512 3072", value_chunks=1, zero_chunks=1),
        # an activation that four layers read: four evaluations of its table and the sumcheck that merges the claims
        dict(name="merge_n20", kind="merge", n=20, claims=4, table="quantised"),
    ]


def draw(rng):
    """One more case of the same ranges (sizes over their logarithm, ragged where the path allows it)."""

    def size(lo, hi):
        return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))

    kind = rng.choice(["product", "matmul", "attention", "lookup", "opening", "linking", "merge"])
    if kind == "product":
        # (a masked activation is a product of three tables; a table that an earlier sumcheck folded is in the extension field)
        tables = [rng.choice(["quantised", "quantised", "base", "ext2"]) for _ in range(rng.choice([2, 2, 2, 3]))]
        eq = rng.random() < 0.7
        return dict(kind=kind, n=rng.randint(8, 24 if tables in (["quantised"] * 2, ["base"] * 2) else 21), eq=eq, tables=_text(tables),
                    claimed=eq and rng.random() < 0.5)
    if kind == "matmul":
        outputs = rng.choice([1, 1, 3])
        return dict(kind=kind, rows=size(1, 512), inner=size(64, 3072 if outputs == 1 else 1024), cols=size(64, 3072 if outputs == 1 else 1024),
                    outputs=outputs, bias=rng.random() < 0.5, bits=rng.choice([16, 64]), host=rng.random() < 0.3)
    if kind == "attention":
        return dict(kind=kind, heads=rng.choice([1, 4, 8, 12, 16]), queries=size(2, 512), keys=size(16, 512), width=rng.choice([32, 64, 80, 128, 256]),
                    bits=rng.choice([16, 64]))
    if kind == "lookup":
        top = rng.randint(8, 22)
        logs = [top] + sorted((rng.randint(6, top) for _ in range(rng.randint(0, 4 if top <= 18 else 1 if top <= 20 else 0))), reverse=True)
        return dict(kind=kind, logs=_text(logs), columns=rng.randint(1, 2), log_table=rng.randint(6, 16), verify=top <= 12)
    if kind == "opening":
        sizes, chunk = [rng.randint(9, 15) for _ in range(rng.randint(3, 14))], rng.randint(9, 12)
        while sum(2 ** max(0, nv - chunk) for nv in sizes) > 140:
            chunk += 1
        return dict(kind=kind, sizes=_text(sizes), chunk=chunk)
    if kind == "linking":
        if rng.random() < 0.5:
            shape = [size(1, 512), size(64, 3072)]
        else:
            shape = [rng.choice([2, 4, 8, 12]), size(2, 256), rng.choice([64, 128])]
        return dict(kind=kind, variant=rng.choice(["standard", "standard", "glu", "softmax", "normalisation"]), shape=_text(shape),
                    value_chunks=rng.randint(1, 2), zero_chunks=rng.randint(0, 2))
    return dict(kind=kind, n=rng.randint(8, 21), claims=rng.randint(2, 9), table=rng.choice(["quantised", "ext2"]))


# ---- what a prover has in hand ----


def _generator(seed):
    return np.random.Generator(np.random.PCG64(seed))


def _base(g, n):
    return g.integers(0, dp.P, size=n, dtype=np.uint64)


def _ext2(g, n):
    return np.stack([_base(g, n), _base(g, n)], axis=-1)


def _table(ctx, g, kind, n):
    if kind == "quantised":  # 12-bit activations, zero-centred
        return ctx.mle_from_i64(g.integers(-2048, 2048, size=1 << n, dtype=np.int64), n)
    return ctx.mle_from_base(_base(g, 1 << n)) if kind == "base" else ctx.mle_from_ext2(_ext2(g, 1 << n))


def _log2_ceil(x):
    return max(0, (x - 1).bit_length())


def _sum_of(proof):
    """p(0) + p(1) of a proof's first message: the sum it proves"""
    return np.array([(int(proof[0][0][k]) + int(proof[0][1][k])) % dp.P for k in range(2)], dtype=np.uint64)


def _linking_config(case):
    return dict(variant=case["variant"], shape=_sizes(case["shape"]), value_chunks=case["value_chunks"], zero_chunks=case["zero_chunks"], bit_size=8,
                signed=True, min_out=-128, max_out=127, input_sign="positive", norm_sum=case["variant"] == "normalisation",
                has_weight=case["variant"] == "normalisation")


def _linking_chunks(case):
    """(number of chunks, variables of a chunk, tables of a chunk)"""
    shape = _sizes(case["shape"])
    chunks = int(np.prod(shape[:-2], dtype=np.int64)) if len(shape) > 2 else 1
    extra = {"standard": 0, "softmax": 0, "glu": 1, "normalisation": 2}[case["variant"]]
    return chunks, sum(_log2_ceil(d) for d in shape[-2:]), case["value_chunks"] + case["zero_chunks"] + extra


def prepare(case, seed):
    g, ctx, kind = _generator(seed), context(), case["kind"]
    s = dict(case=case)
    if kind == "product":
        n = case["n"]
        s["tables"] = [_table(ctx, g, kind, n) for kind in case["tables"].split()]
        s["point"] = _ext2(g, n)
        factors = list(range(len(s["tables"])))
        s["terms"] = [(ONE, [len(factors)] + factors if case["eq"] else factors)]
        s["claim"] = None
        if case["claimed"]:  # the layer behind this one has left the claim on the product
            eq = ctx.eq_build(s["point"])
            s["claim"] = _sum_of(ctx.sumcheck_prove(n, s["tables"] + [eq], s["terms"], dp.Transcript(b"claim"))[0])
    elif kind == "matmul":
        rows, inner, cols, outputs = (case[k] for k in ("rows", "inner", "cols", "outputs"))
        values = lambda *shape: g.integers(-2048, 2048, size=shape, dtype=np.int64)
        row, out = ("k", "j") if rows == 1 else ("ik", "ij")  # a single row is a vector
        s["ops"] = [(row, "kj", out, "j") if case["bias"] else (row, "kj", out)] * outputs
        lhs, rhs = values(inner) if rows == 1 else values(rows, inner), [values(inner, cols) for _ in range(outputs)]
        biases = [values(cols) for _ in range(outputs)] if case["bias"] else None
        if not case["host"]:
            lhs, rhs = dp.Tensor(ctx, lhs, case["bits"]), [dp.Tensor(ctx, x, case["bits"]) for x in rhs]
            biases = None if biases is None else [dp.Tensor(ctx, b, case["bits"]) for b in biases]
        s["lhs"], s["rhs"], s["biases"] = lhs, rhs, biases
        s["claims"] = [(_ext2(g, _log2_ceil(rows) + _log2_ceil(cols)), ONE) for _ in range(outputs)]
    elif kind == "attention":
        heads, queries, keys, width = (case[k] for k in ("heads", "queries", "keys", "width"))
        tensor = lambda *shape: dp.Tensor(ctx, g.integers(-2048, 2048, size=shape, dtype=np.int64), case["bits"])
        s["q"], s["k"], s["v"] = tensor(heads, queries, width), tensor(heads, keys, width), tensor(heads, keys, width)
        s["probabilities"] = tensor(heads, queries, keys)
        vh, vq, vk, vw = (_log2_ceil(x) for x in (heads, queries, keys, width))
        s["scores_claim"], s["context_claim"] = (_ext2(g, vh + vq + vk), ONE), (_ext2(g, vh + vq + vw), ONE)
    elif kind == "lookup":
        size = 1 << case["log_table"]
        t_in = np.arange(size, dtype=np.uint64)
        columns = [t_in, (t_in * np.uint64(40503) + np.uint64(17)) & np.uint64(0xFFFF)][: case["columns"]]
        tr = dp.Transcript(b"lookup")
        tr.append_u64(seed)
        c, beta = tr.append_and_sample(b"c"), tr.append_and_sample(b"beta")
        count, s["lookups"] = np.zeros(size, dtype=np.int64), []
        for log in _sizes(case["logs"]):
            idx = g.integers(0, size, size=1 << log)
            count += np.bincount(idx, minlength=size)
            s["lookups"].append(dict(cols=[ctx.mle_from_base(col[idx]) for col in columns], numer=None, c=c, beta=beta))
        s["table"] = [dict(cols=[ctx.mle_from_base(col) for col in columns], numer=ctx.mle_from_base(count.astype(np.uint64)), c=c, beta=beta)]
        s["transcript"] = tr
        s["lookup_shapes"] = [(case["columns"], log - 1, c, beta) for log in _sizes(case["logs"])]
        s["table_shapes"] = [(case["columns"], case["log_table"] - 1, c, beta)]
    elif kind == "opening":
        s["polys"], s["claims"] = [], []
        for i, nv in enumerate(_sizes(case["sizes"])):
            whole, m = ctx.mle_from_ext2(_ext2(g, 1 << nv)), min(nv, case["chunk"])
            s["polys"].append([whole.view(k << m, m) for k in range(1 << (nv - m))])
            points = [_ext2(g, nv) for _ in range(2 if i < 5 and i % 2 else 1)]
            s["claims"].append([(p, whole.evaluate(p)) for p in points])
    elif kind == "linking":
        chunks, nv, per_chunk = _linking_chunks(case)
        config = s["config"] = _linking_config(case)
        narrow = lambda: ctx.mle_from_i64(g.integers(-128, 128, size=1 << nv, dtype=np.int64), nv)
        bit = lambda: ctx.mle_from_i64(g.integers(-1, 2, size=1 << nv, dtype=np.int64), nv)
        s["tables"] = []
        for _ in range(chunks):
            s["tables"] += [narrow() for _ in range(case["value_chunks"])] + [bit() for _ in range(case["zero_chunks"])]
        s["tables"] += [narrow() for _ in range(chunks * (per_chunk - case["value_chunks"] - case["zero_chunks"]))]
        s["weight"] = narrow() if config["has_weight"] else None
        s["claim_point"] = _ext2(g, sum(_log2_ceil(d) for d in _sizes(case["shape"])))
        s["logup_point"] = _ext2(g, nv)
    else:
        s["table"] = _table(ctx, g, case["table"], case["n"])
        s["points"] = [_ext2(g, case["n"]) for _ in range(case["claims"])]
    return s


# ---- one proof ----


def _einsum_outputs(r):
    out = [r["proof"], r["evaluations"]]
    if r["aggregation_proof"] is not None:
        out.append(r["aggregation_proof"])
    for point, value in r["claims"]:
        out += [point, value]
    for _, point, value in r["bias_claims"]:
        out += [point, value]
    return out


def run(state):
    ctx, case = context(), state["case"]
    kind = case["kind"]
    if kind == "product":
        tables = list(state["tables"])
        if case["eq"]:
            tables.append(ctx.eq_build(state["point"]))
        if state["claim"] is None:
            return ctx.sumcheck_prove(case["n"], tables, state["terms"], dp.Transcript(b"product"))
        return ctx.sumcheck_prover(case["n"], tables, state["terms"], claim=state["claim"])(dp.Transcript(b"product"))
    if kind == "matmul":
        return _einsum_outputs(dp.einsum_prove(ctx, state["ops"], state["lhs"], state["rhs"], state["claims"], dp.Transcript(b"matmul"), state["biases"]))
    if kind == "attention":
        tr = dp.Transcript(b"attention")
        context_proof = dp.einsum_prove(ctx, [("hst", "htd", "hsd")], state["probabilities"], [state["v"]], [state["context_claim"]], tr)
        scores_proof = dp.einsum_prove(ctx, [("hsd", "htd", "hst")], state["q"], [state["k"]], [state["scores_claim"]], tr)
        return _einsum_outputs(context_proof) + _einsum_outputs(scores_proof)
    if kind == "lookup":
        tr = state["transcript"].clone()
        lookups, table = dp.logup_batch_prove(ctx, state["lookups"], tr), dp.logup_batch_prove(ctx, state["table"], tr)
        if not case["verify"]:
            return lookups, table
        check = state["transcript"].clone()
        ok_l, claims_l, point_l = dp.logup_batch_verify(state["lookup_shapes"], False, lookups, check)
        ok_t, claims_t, point_t = dp.logup_batch_verify(state["table_shapes"], True, table, check)
        return lookups, table, ok_l, claims_l, point_l, ok_t, claims_t, point_t
    if kind == "opening":
        return dp.claims_batching_prove(ctx, state["polys"], state["claims"], dp.Transcript(b"opening"))
    if kind == "linking":
        proof, point, evals, weight, _ = dp.linking_prove(ctx, state["config"], state["tables"], dp.Transcript(b"linking"), state["claim_point"],
                                                          state["logup_point"], state["weight"])
        return (proof, point, evals) if weight is None else (proof, point, evals, weight)
    claims = [(p, state["table"].evaluate(p)) for p in state["points"]]
    return dp.same_poly_prove(ctx, state["table"], claims, dp.Transcript(b"merge")) + tuple(v for _, v in claims)


# ---- what a proof cannot do without ----


def _sumcheck_mults(n, base_tables, ext_tables, per_pair_first, per_pair):
    """Base-field multiply-adds of a sumcheck over 2^n entries: a round's products a pair (the first round's are
    cheaper: its tables are in the base field), and the folds (2 a base entry, 4 an extension entry)."""
    pairs = 2.0 ** (n - 1)
    return pairs * (per_pair_first + 2 * base_tables + 4 * ext_tables) + pairs * (per_pair + 4 * (base_tables + ext_tables))


def work(case):
    """Every input read once, the proof written; operations are 2 a base-field multiply-add (an extension product is 4)."""
    kind, mults = case["kind"], 0.0
    if kind == "product":
        n, kinds, eq = case["n"], case["tables"].split(), 1 if case["eq"] else 0
        k, ext = len(kinds), sum(t == "ext2" for t in kinds)
        nbytes, proof = 8 * (k + ext) * 2.0**n, n * (k + eq + 1) * 16
        # a round evaluates the product of k tables at k points, each weighted where there is an eq factor
        mults = _sumcheck_mults(n, k - ext, ext, k * ((k - 1 + 2 * eq) if not ext else 4 * (k - 1 + eq)), k * 4 * (k - 1 + eq))
    elif kind == "matmul":
        entry = case["bits"] // 8
        one, weights = case["rows"] * case["inner"], case["outputs"] * case["inner"] * case["cols"]
        nv = _log2_ceil(case["inner"])
        nbytes, proof = entry * (one + weights), nv * 3 * 16
        mults = 2.0 * (case["outputs"] * one + weights) + case["outputs"] * _sumcheck_mults(nv, 0, 2, 8, 8)
        if case["outputs"] > 1:
            mults += _sumcheck_mults(_log2_ceil(case["rows"]) + nv, 1, 1, 4, 8)
    elif kind == "attention":
        entry, heads = case["bits"] // 8, case["heads"]
        q, k, p = (heads * a * b for a, b in ((case["queries"], case["width"]), (case["keys"], case["width"]), (case["queries"], case["keys"])))
        nbytes = entry * (q + 2 * k + p)
        mults = 2.0 * (q + 2 * k + p) + heads * sum(_sumcheck_mults(_log2_ceil(x), 0, 2, 8, 8) for x in (case["width"], case["keys"]))
        proof = 3 * 16 * (_log2_ceil(case["width"]) + _log2_ceil(case["keys"]))
    elif kind == "lookup":
        nbytes, proof = 0.0, 0.0
        for log, table in [(x, 0) for x in _sizes(case["logs"])] + [(case["log_table"], 1)]:
            entries, cols = 2.0**log, case["columns"] + table
            nbytes += 8 * cols * entries
            proof += 16 * 4 * log * log / 2
            # the fraction tree: the denominators, then three extension products a node; its layer sums: every layer is a
            # sumcheck of four tables, six products and a weight at two points a pair
            mults += entries * (2 * case["columns"] + 12) + sum(_sumcheck_mults(v, 0, 4, 32, 32) for v in range(1, log - 1))
            mults += _sumcheck_mults(log - 1, 2 * cols, 0, 16, 32)
    elif kind == "opening":
        tables = sum(2.0 ** (nv - min(nv, case["chunk"])) for nv in _sizes(case["sizes"]))
        nbytes, proof = sum(16 * 2.0**nv for nv in _sizes(case["sizes"])), 3 * 16 * case["chunk"] + 16 * tables
        mults = sum(2.0 ** (nv - min(nv, case["chunk"])) * _sumcheck_mults(min(nv, case["chunk"]), 0, 1, 8, 8) for nv in _sizes(case["sizes"]))
    elif kind == "linking":
        chunks, nv, per_chunk = _linking_chunks(case)
        tables = chunks * per_chunk + (1 if case["variant"] == "normalisation" else 0)
        nbytes, proof = tables * 8 * 2.0**nv, nv * 5 * 16 + tables * 16
        mults = _sumcheck_mults(nv, tables, 0, 6 * tables, 12 * tables)
    else:
        n, base = case["n"], case["table"] != "ext2"
        nbytes, proof = (8 if base else 16) * 2.0**n, n * 3 * 16
        mults = case["claims"] * (2 if base else 4) * 2.0**n + _sumcheck_mults(n, 1 if base else 0, 1 if base else 2, 4 if base else 8, 8)
    return {"bytes": float(nbytes + proof), "flops": 2.0 * mults}


def tolerance(case):
    """Field elements: any correct implementation gives the same bits."""
    return "exact"
