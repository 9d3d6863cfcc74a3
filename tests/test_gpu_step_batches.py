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
    (6, 3, 4, [0, 2, 5, 7, 13]),                       # six digits: one after the other
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
