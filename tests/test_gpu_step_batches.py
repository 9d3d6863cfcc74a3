"""Batches of linear-transform steps against the oracle's stage by stage form:
more (step, ciphertext) pairs than one launch sequence takes (32), pieces that
end inside a step, single ciphertexts, missing terms and no giant step 0, both
evaluators, digit counts with and without the folded key product (the QP stage
against the oracle, the Q stage against the sequential form that the reference
vectors pin)."""
import numpy as np
import pytest

import oracle as O
from helpers import product, rand_residues

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("evaluator", ["qp", "q"])
@pytest.mark.parametrize("dnum,count,bs,index", [
    (3, 1, 4, [0, 1, 3, 4, 6, 9]),
    (3, 7, 8, list(range(1, 8)) + [8, 11, 24, 40]),    # 49 baby pairs: 32 + 17; giants 0, 1, 3, 5
    (2, 5, 4, [5, 6, 9, 11, 14]),                      # no giant step 0
    (6, 3, 4, [0, 2, 5, 7, 13]),                       # five digits at this level
    (3, 3, 20, [0, 3, 17, 19, 20, 36, 39]),            # baby steps beyond 16
])
def test_stage_batches_match_the_oracle(evaluator, dnum, count, bs, index, monkeypatch):
    M = product()
    N = 1 << 11
    p, q = O.find_primes([61, 50, 50], [36, 61, 42, 50, 38, 38], N)
    ctx, octx = M.Context(N, q, p, dnum), O.Ctx(N, q, p, dnum)
    level = 4
    Q, basis = list(q[: level + 1]), list(q) + list(p)
    rng = np.random.default_rng(count + 10 * bs)
    dmod = Q + list(p) if evaluator == "qp" else Q
    diags = [rand_residues(rng, dmod, N) for _ in index]
    rots = sorted(({d % bs for d in index} | {d - d % bs for d in index}) - {0})
    keys = {r: np.concatenate([rand_residues(rng, basis, N) for _ in range(2 * octx.parts(len(q) - 1))]) for r in rots}
    cts = [(rand_residues(rng, Q, N), rand_residues(rng, Q, N)) for _ in range(count)]
    W = (level + 1) * N
    outs = [(M.to_dev(np.zeros(W, np.uint64)), M.to_dev(np.zeros(W, np.uint64))) for _ in cts]
    ctx.linear_transform_qp_batch(level, [(M.to_dev(a), M.to_dev(b)) for a, b in cts], index,
                                  [M.to_dev(d) for d in diags], bs, {r: M.to_dev(k) for r, k in keys.items()}, outs,
                                  q_evaluator=evaluator == "q")
    single = [(M.to_dev(np.zeros(W, np.uint64)), M.to_dev(np.zeros(W, np.uint64))) for _ in cts]
    # one ciphertext per call, the key products in their separate, step-by-step form
    monkeypatch.setenv("MICKKS_FUSE_MAC", "0")
    plain = M.Context(N, q, p, dnum)
    fn = plain.linear_transform_q if evaluator == "q" else plain.linear_transform_qp
    for (a, b), (oa, ob) in zip(cts, single):
        fn(level, M.to_dev(a), M.to_dev(b), index, [M.to_dev(d) for d in diags], bs,
           {r: M.to_dev(k) for r, k in keys.items()}, oa, ob)
    for k, ((oa, ob), (sa, sb)) in enumerate(zip(outs, single)):
        assert np.array_equal(M.from_dev(oa), M.from_dev(sa)) and np.array_equal(M.from_dev(ob), M.from_dev(sb)), k
    if evaluator == "qp":
        for (a, b), (oa, ob) in zip(cts[:2], outs[:2]):
            wa, wb = octx.lt_stage_qp(level, a, b, index, np.concatenate(diags), bs, keys)
            assert np.array_equal(M.from_dev(oa), wa) and np.array_equal(M.from_dev(ob), wb)


@pytest.mark.parametrize("kind", ["both", "integer", "double"])
@pytest.mark.parametrize("dnum,level,count,bs,giants", [
    (6, 5, 1, 4, 2), (6, 5, 3, 4, 5),  # six digits: one after the other
    (3, 5, 1, 4, 5),                   # one ciphertext, more giant steps than four
    (3, 5, 3, 4, 8), (2, 3, 5, 2, 6),  # five to eight giant steps, an odd last ciphertext
    (3, 4, 2, 4, 9), (4, 5, 3, 2, 16),  # nine to sixteen, more than one ciphertext
    (2, 3, 2, 2, 17),                  # a second launch of giant steps
    (3, 5, 2, 18, 17),                 # and of baby steps
    (3, 3, 2, 1, 10),                  # no baby step
    (6, 5, 105, 2, 9),                 # more than 850,000 coefficients
])
def test_qp_stage_shapes_match_the_oracle(kind, dnum, level, count, bs, giants):
    """The QP evaluator's fused kernel in each of its shapes (giant steps at a
    time, ciphertexts at a time, digits unrolled or not), over moduli below and
    above 2^50 in one basis and of one kind alone; a term of every second
    diagonal is missing, giant step 1 is whole."""
    M = product()
    N = 1 << 10
    p_bits, q_bits = {"both": ([61, 50], [36, 61, 42, 50, 38, 60]), "integer": ([61, 55], [60, 61, 52, 55, 58, 60]),
                      "double": ([50, 49], [36, 50, 42, 50, 38, 27])}[kind]
    p, q = O.find_primes(p_bits, q_bits, N)
    ctx, octx = M.Context(N, q, p, dnum), O.Ctx(N, q, p, dnum)
    assert (ctx.parts(level) > 5) == (dnum == 6)
    rng = np.random.default_rng(dnum + 10 * giants + 1000 * count)
    Q, basis, T = list(q[: level + 1]), list(q) + list(p), list(q[: level + 1]) + list(p)
    index = [d for d in range(bs * giants) if bs == 1 or d // bs == 1 or d % 2 == 0 or d == bs * giants - 1]
    assert {d // bs for d in index} == set(range(giants))
    pool = [rand_residues(rng, T, N) for _ in range(5)]
    diags = [pool[i % 5] for i in range(len(index))]
    rots = sorted(({d % bs for d in index} | {d - d % bs for d in index}) - {0})
    made = [np.concatenate([rand_residues(rng, basis, N) for _ in range(2 * octx.parts(len(q) - 1))]) for _ in range(3)]
    keys = {r: made[i % 3] for i, r in enumerate(rots)}
    cts = [(rand_residues(rng, Q, N), rand_residues(rng, Q, N)) for _ in range(count)]
    dev = {id(x): M.to_dev(x) for x in pool + made}
    W = (level + 1) * N
    outs = [(M.to_dev(np.zeros(W, np.uint64)), M.to_dev(np.zeros(W, np.uint64))) for _ in cts]
    ctx.linear_transform_qp_batch(level, [(M.to_dev(a), M.to_dev(b)) for a, b in cts], index,
                                  [dev[id(d)] for d in diags], bs, {r: dev[id(k)] for r, k in keys.items()}, outs)
    for i in {0, count - 1}:
        wa, wb = octx.lt_stage_qp(level, *cts[i], index, np.concatenate(diags), bs, keys)
        assert np.array_equal(M.from_dev(outs[i][0]), wa) and np.array_equal(M.from_dev(outs[i][1]), wb), i


def _sequential(M, N, q, p, dnum, monkeypatch):
    """A context that runs the Q evaluator's steps one after the other."""
    monkeypatch.setenv("MICKKS_FUSE_MAC", "0")
    ctx = M.Context(N, q, p, dnum)
    monkeypatch.delenv("MICKKS_FUSE_MAC")
    return ctx


def test_one_ciphertext_keeps_its_scratch_small(monkeypatch):
    """31 baby steps of one ciphertext at N = 2^16, 30 + 10 limbs: the steps run
    in batches of nine pairs (2^25 words of two polynomials), not of 31 with
    152 MB of scratch each; the result is the sequential form's."""
    M = product()
    N, level, bs = 1 << 16, 29, 32
    p, q = O.find_primes([50] * 10, [50] * 30, N)
    ctx = M.Context(N, q, p, 3)
    rng = np.random.default_rng(5)
    key = np.tile(rand_residues(rng, list(q) + list(p), N), 2 * ctx.parts(level))
    ct, diag = [rand_residues(rng, q, N) for _ in range(2)], M.to_dev(rand_residues(rng, q, N))
    dkey, index = M.to_dev(key), list(range(bs))
    results = []
    for c in (ctx, _sequential(M, N, q, p, 3, monkeypatch)):
        out = [M.to_dev(np.zeros((level + 1) * N, np.uint64)) for _ in range(2)]
        before = c.device_bytes()
        c.linear_transform_q(level, M.to_dev(ct[0]), M.to_dev(ct[1]), index, [diag] * bs, bs,
                             {r: dkey for r in range(1, bs)}, out[0], out[1])
        results.append([M.from_dev(o) for o in out])
        if c is ctx:
            LN, pair = 30 * N, (3 * 40 + 30 + 20 + 120) * N
            babies = 2 * (bs - 1) * LN
            assert c.device_bytes() - before <= 8 * (9 * pair + babies + 2 * LN)
    assert all(np.array_equal(x, y) for x, y in zip(*results))


def test_steps_fit_the_workspace_of_a_capture(monkeypatch):
    """A captured transform whose stream holds enough for one ciphertext's steps
    one at a time, but not for a batch of them, runs them one at a time."""
    import torch
    M = product()
    N, level, bs = 1 << 12, 5, 13
    p, q = O.find_primes([50] * 3, [50] * 6, N)
    ctx = M.Context(N, q, p, 3)
    rng = np.random.default_rng(6)
    key = M.to_dev(np.concatenate([rand_residues(rng, list(q) + list(p), N) for _ in range(6)]))
    a, b, diag = (M.to_dev(rand_residues(rng, q, N)) for _ in range(3))
    new = lambda: M.to_dev(np.zeros(6 * N, np.uint64))  # noqa: E731
    out, want, st = [new(), new()], [new(), new()], torch.cuda.Stream()
    args = (list(range(bs)), [diag] * bs, bs, {r: key for r in range(1, bs)})
    _sequential(M, N, q, p, 3, monkeypatch).linear_transform_q(level, a, b, *args, want[0], want[1])
    torch.cuda.synchronize()
    # eight key switches at once: 408 limbs of workspace, where the transform's
    # steps take 219 one at a time and 900 as one batch
    ctx.keyswitch_batch([(level, a, key, new(), new(), 0, 1) for _ in range(8)], stream=st)
    st.synchronize()
    ctx.graph_begin(st)
    ctx.linear_transform_q(level, a, b, *args, out[0], out[1], stream=st)
    graph = ctx.graph_end(st)
    try:
        for r in range(3):
            out[0].zero_(), out[1].zero_()
            torch.cuda.synchronize()
            graph.launch(st)
            st.synchronize()
            assert all(np.array_equal(M.from_dev(o), M.from_dev(w)) for o, w in zip(out, want)), r
            ctx.keyswitch_batch([(level, a, key, new(), new(), 0, 1)], stream=st)
            st.synchronize()
    finally:
        graph.destroy()
