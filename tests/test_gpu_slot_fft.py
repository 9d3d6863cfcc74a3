"""The special FFTs of encoding and decoding run in two passes (a block of 2048
points, then columns): every ring dimension, so every number of column stages
from none to five, bit for bit against the host's stage-by-stage form."""
import numpy as np
import pytest

from helpers import host

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("logn", [10, 11, 12, 13, 14, 15, 16])
def test_encode_and_decode_equal_the_host_form(logn):
    H = host()
    c = H.CKKSParamsConfig()
    c.N = 1 << logn
    c.mult_depth = 2
    c.q0_bit = 50
    c.q_bit = 40
    c.p_bits = [50]
    c.dnum = 3
    c.secure = False
    c.seed = logn
    ctx = H.CKKSContext(H.CKKSParams(c))
    P = ctx.getParams()
    rng = np.random.default_rng(logn)
    v = rng.uniform(-1, 1, P.getSlots()) + 1j * rng.uniform(-1, 1, P.getSlots())
    for level in (0, 2):
        got = H.ckks_encode(ctx, v, level).getPlaintext()
        want = H.encode_slots_custom_basis(ctx, v, P.getScale(), list(P.getModuli()[: level + 1]))
        assert np.array_equal(np.asarray(got), np.asarray(want)), level
    ct = H.ckks_encrypt(ctx, v, 2)
    got, want = H.ckks_decrypt(ctx, ct), H.ckks_decrypt_host_decode(ctx, ct)
    assert np.array_equal(np.asarray(got), np.asarray(want))
    assert np.max(np.abs(np.asarray(got) - v)) < 1e-5
