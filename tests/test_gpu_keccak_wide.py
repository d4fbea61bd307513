"""FrodoKEM-976 calls whose sponges run on 16 lanes per request against the lane-pair
form of a larger call (and, for a few requests, the CPU oracle)."""
import numpy as np
import pytest

from tests import oracle_lib as O

pytestmark = pytest.mark.gpu

CT, SS = 15744, 24


def test_frodo_16_lane_calls_equal_pair_call_and_oracle():
    import pqc_amd
    n = 4100  # above the 16-lane form's limit
    rng = np.random.default_rng(11)
    pk, sk = O.frodo_keypair(rng.integers(0, 256, 64, dtype=np.uint8).tobytes())
    pk, sk = np.frombuffer(pk, np.uint8).copy(), np.frombuffer(sk, np.uint8).copy()
    mu = rng.integers(0, 256, (n, 24), dtype=np.uint8)
    ctx = pqc_amd.Context(["frodo976"], max_batch=n)
    print("frodo pairs", n, flush=True)
    ct, ss = ctx.frodo_enc_host(pk, mu)
    ct[::5, rng.integers(0, CT)] ^= 1
    want = ctx.frodo_dec_host(sk, ct)
    assert (want[1::5] == ss[1::5]).all() and (want[::5] != ss[::5]).any(axis=1).all()
    for m in (1, 3, 4, 5, 63, 1025, 4096):
        print("frodo 16 lanes", m, flush=True)
        c2, s2 = ctx.frodo_enc_host(pk, mu[:m])
        assert (s2 == ss[:m]).all() and (c2[1:5] == ct[1:5][: len(c2) - 1]).all()
        assert (ctx.frodo_dec_host(sk, ct[:m]) == want[:m]).all()
    for i in range(3):
        oc, os_ = O.frodo_enc(pk.tobytes(), mu[i].tobytes())
        assert ss[i].tobytes() == os_
        assert want[i].tobytes() == O.frodo_dec(ct[i].tobytes(), sk.tobytes())
    ctx.close()
