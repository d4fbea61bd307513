"""The fused NewHope CPA kernels (FP32 transforms, four elements per workgroup) against the
per-operation kernels at batch sizes around a workgroup's edge, on valid keys and on
arbitrary bytes, whose 14-bit coefficients reach past q."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1024, 512])
def test_fused_equals_plain_at_workgroup_edges(N):
    import pqc_amd
    rng = np.random.default_rng(N)
    pkb, skb, ctb = 14 * N // 8 + 32, 14 * N // 8, 17 * N // 8
    ctx = pqc_amd.Context([f"newhope{N}cpa"], max_batch=300)
    rand = lambda n, b: rng.integers(0, 256, (n, b), dtype=np.uint8)  # noqa: E731
    for n in (1, 2, 3, 4, 5, 7, 257):
        print("newhope fused", N, n, flush=True)
        seed, msg, coin, rpk, rsk, rct = (rand(n, b) for b in (32, 32, 32, pkb, skb, ctb))
        out = []
        for plain in (False, True):
            pk, sk = np.empty((n, pkb), np.uint8), np.empty((n, skb), np.uint8)
            ct, ct2 = np.empty((n, ctb), np.uint8), np.empty((n, ctb), np.uint8)
            m, m2 = np.empty((n, 32), np.uint8), np.empty((n, 32), np.uint8)
            kw = dict(host=True, N=N, plain=plain)
            ctx.newhope_keypair(n, pk, sk, seed, **kw)
            ctx.newhope_enc(n, ct, msg, pk, coin, **kw)
            ctx.newhope_dec(n, m, ct, sk, **kw)
            assert (m == msg).all()
            ctx.newhope_enc(n, ct2, msg, rpk, coin, **kw)
            ctx.newhope_dec(n, m2, rct, rsk, **kw)
            out.append((pk, sk, ct, ct2, m2))
        for a, b in zip(*out):
            assert (a == b).all()
    ctx.close()
