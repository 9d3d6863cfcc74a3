"""Moduli below 2^50 are computed in integer-valued doubles, larger ones in
integers: both sides of that line, and the values that bring the doubles
closest to 2^53, against the oracle (whose arithmetic is integer throughout).
Residues are exact, so every comparison is equality."""
import numpy as np
import pytest

import oracle as O
from helpers import product, rand_residues

pytestmark = pytest.mark.gpu

# above and below 2^50 (integers / doubles) and 2^44 (reductions inside a pass)
BITS = [50, 51, 49, 45, 44, 43, 36, 27, 61, 50, 38]


def _pattern(kind, rng, moduli, N):
    if kind == "random":
        return rand_residues(rng, moduli, N)
    out = []
    for m in moduli:
        m = int(m)
        x = np.full(N, m - 1, dtype=np.uint64)
        if kind == "alternating":
            x[1::2] = 0
        elif kind == "halves":
            x[: N // 2], x[N // 2:] = m // 2, m // 2 + 1
        out.append(x)
    return np.concatenate(out)


@pytest.mark.parametrize("kind", ["random", "largest", "alternating", "halves"])
@pytest.mark.parametrize("logn", [10, 11, 12, 13, 14, 15, 16])
def test_transforms_on_both_sides_of_the_line(logn, kind):
    M = product()
    N = 1 << logn
    p, q = O.find_primes([61], BITS, N)
    assert any(int(v) < 1 << 50 for v in q) and any(int(v) >= 1 << 50 for v in q)
    ctx, octx = M.Context(N, q, p, 2), O.Ctx(N, q, p, 2)
    host = _pattern(kind, np.random.default_rng(logn), q, N)
    d = M.to_dev(host)
    ctx.ntt_forward(d, 1, len(q))
    assert np.array_equal(M.from_dev(d), octx.ntt_fwd(host, len(q)))
    ctx.ntt_inverse(d, 1, len(q))
    assert np.array_equal(M.from_dev(d), host)
    # the inverse of extreme evaluations, and the forward one back
    d = M.to_dev(host)
    ctx.ntt_inverse(d, 1, len(q))
    ctx.ntt_forward(d, 1, len(q))
    assert np.array_equal(M.from_dev(d), host)


@pytest.mark.parametrize("kind", ["random", "largest"])
@pytest.mark.parametrize("p_bits,q_bits,dnum", [
    ([50] * 3, [50] * 8, 3),                    # doubles throughout
    ([61] * 4, [36, 61, 42, 42, 38, 38, 50], 2),  # both kinds in one digit
    ([50], [50, 51, 50, 49], 4),                # one limb per digit
])
@pytest.mark.parametrize("mont", [True, False])
def test_key_switch_and_rescale(p_bits, q_bits, dnum, kind, mont):
    M = product()
    N = 1 << 12
    p, q = O.find_primes(p_bits, q_bits, N)
    ctx, octx = M.Context(N, q, p, dnum), O.Ctx(N, q, p, dnum)
    rng = np.random.default_rng(len(q_bits) + 10 * dnum)
    basis = list(q) + list(p)
    top = len(q) - 1
    key = np.concatenate([_pattern(kind, rng, basis, N) for _ in range(2 * octx.parts(top))])
    dkey = M.to_dev(key)
    for level in (top, top // 2):
        Q = q[: level + 1]
        kt, b, a = (_pattern(kind, rng, Q, N) for _ in range(3))
        ob, oa = octx.keyswitch(level, kt, key, b, a, 0, 1, montgomery=mont)
        db, da = M.to_dev(b), M.to_dev(a)
        ctx.keyswitch(level, M.to_dev(kt), dkey, db, da, 0, 1, montgomery=mont)
        assert np.array_equal(M.from_dev(db), ob) and np.array_equal(M.from_dev(da), oa), level
        x = M.to_dev(b)
        ctx.rescale(level, x, 1)
        want = octx.rescale(level, b.reshape(1, -1))
        assert np.array_equal(M.from_dev(x)[: level * N], want[0]), level


@pytest.mark.parametrize("bits", [50, 49, 43, 38])
@pytest.mark.parametrize("over", [False, True])
@pytest.mark.parametrize("mont", [True, False])
def test_walsh_sum_at_the_line_of_exact_doubles(bits, over, mont):
    """A row of Walsh coefficients whose magnitudes sum to the largest value
    that keeps a combination and its constant below 2^53 (doubles), and to one
    more (integers), over residues all q - 1."""
    M = product()
    N = 1 << 10
    p, q = O.find_primes([61], [bits, bits], N)
    ctx, octx = M.Context(N, q, p, 1), O.Ctx(N, q, p, 1)
    rng = np.random.default_rng(bits)
    Q = [int(v) for v in q]
    most = (1 << 53) // max(Q) - 1 + (1 if over else 0)
    row = np.zeros(16, dtype=np.int64)
    row[1:] = most // 15
    row[1: 1 + most % 15] += 1
    cr = np.stack([row if h % 2 == 0 else -row for h in range(16)])
    ci = np.stack([-row if h % 3 == 0 else row for h in range(16)])
    big = _pattern("largest", rng, Q, N)
    low = [np.stack([big, big]) for _ in range(15)]
    high = [np.stack([big, rand_residues(rng, Q, N)]) for _ in range(15)]
    pt = _pattern("largest", rng, Q, N)
    consts = [(-1, (1 << 90) + h) for h in range(16)]  # constants of q - 1 and of many words
    acc_o, raw_o = octx.walsh_product_sum(1, low, high, cr, ci, consts, pt, mont)
    dev = lambda x: [M.to_dev(x[0]), M.to_dev(x[1])]  # noqa: E731
    new = lambda: M.to_dev(np.zeros(2 * N, np.uint64))  # noqa: E731
    acc, raw = [new(), new()], [new(), new(), new()]
    ctx.walsh_product_sum(1, [dev(x) for x in low], [dev(x) for x in high], cr, ci, consts, M.to_dev(pt), acc, raw,
                          pt_montgomery=mont)
    assert all(np.array_equal(M.from_dev(a), o) for a, o in zip(acc, acc_o))
    assert all(np.array_equal(M.from_dev(r), o) for r, o in zip(raw, raw_o))


# A prime below 2^50 whose rounded inverse is a little below 1/q by almost half
# a unit in the last place, a residue x and a word y in [3q, 4q) for which the
# products of the double path leave x y - k q = 1.4956 q, odd: five of them and
# q - 1 are an odd number above 2^53.
WORST_Q, WORST_X, WORST_Y = 1125899894996993, 1122752751754747, 4501000844983853


@pytest.mark.parametrize("mont", [True, False])
@pytest.mark.parametrize("keys", ["largest", "worst"])
@pytest.mark.parametrize("parts", [1, 3, 4, 5, 6])
def test_fused_baby_steps_at_their_largest(parts, keys, mont):
    """QP linear transforms whose key products are the largest that the double
    path meets: digits of q - 1 (a polynomial that is a small negative constant
    is one in every digit) against keys of 4q - 1, and the digits and keys above,
    whose sum over five digits is not a double.  Diagonals of 4q - 1, b of q - 1,
    against the oracle on the reduced values."""
    M = product()
    N = 1 << 11
    p, q = O.find_primes([50], [50] * 5, N)
    q = [WORST_Q] + [int(v) for v in q]
    p = [int(v) for v in p]
    assert len(set(q + p)) == 7 and (WORST_Q - 1) % (2 * N) == 0
    ctx, octx = M.Context(N, q, p, 6), O.Ctx(N, q, p, 6)
    level = parts - 1
    assert ctx.parts(level) == parts
    minus = 1 if keys == "largest" else WORST_Q - WORST_X
    full = lambda moduli, value: np.concatenate([np.full(N, value(int(m)), np.uint64) for m in moduli])  # noqa: E731
    Q, basis, T = q[: level + 1], q + p, q[: level + 1] + p
    a, b = full(Q, lambda m: m - minus), full(Q, lambda m: m - 1)
    raw = full(basis, lambda m: WORST_Y if keys == "worst" and m == WORST_Q else 4 * m - 1)
    raw = np.concatenate([raw] * (2 * octx.parts(len(q) - 1)))
    mods = np.repeat(np.array(basis, np.uint64), N)
    key = raw % np.concatenate([mods] * (2 * octx.parts(len(q) - 1)))
    index = [0, 1, 2, 3, 5, 6]
    lifted = full(T, lambda m: 4 * m - 1)
    diags = [lifted % np.repeat(np.array(T, np.uint64), N)] * len(index)
    rots = [1, 2, 3, 4]
    wa, wb = octx.lt_stage_qp(level, a, b, index, np.concatenate(diags), 4, {r: key for r in rots}, montgomery=mont)
    dkey, ddiag = M.to_dev(raw), M.to_dev(lifted)
    for count in (1, 3):
        outs = [(M.to_dev(np.zeros(len(a), np.uint64)), M.to_dev(np.zeros(len(a), np.uint64))) for _ in range(count)]
        ctx.linear_transform_qp_batch(level, [(M.to_dev(a), M.to_dev(b))] * count, index, [ddiag] * len(index), 4,
                                      {r: dkey for r in rots}, outs, montgomery=mont)
        for oa, ob in outs:
            assert np.array_equal(M.from_dev(oa), wa) and np.array_equal(M.from_dev(ob), wb), count


@pytest.mark.parametrize("kind", ["random", "largest", "halves"])
@pytest.mark.parametrize("first", [49, 50, 51, 60])
def test_modraise_from_either_side(first, kind):
    """The q_0 limb, below or above 2^50, centred and lifted to limbs of both
    sides; values around q_0 / 2, where the sign changes, among them."""
    M = product()
    N = 1 << 11
    p, q = O.find_primes([61], [first, 50, 51, 36, 61, 27], N)
    ctx, octx = M.Context(N, q, p, 2), O.Ctx(N, q, p, 2)
    coeff = _pattern(kind, np.random.default_rng(first), q[:1], N)
    x = M.to_dev(coeff)
    ctx.ntt_forward(x, 1, 1)
    host = M.from_dev(x)
    out = M.to_dev(np.zeros(len(q) * N, np.uint64))
    ctx.modraise(len(q) - 1, x, out)
    assert np.array_equal(M.from_dev(out), octx.modraise(len(q) - 1, host))
