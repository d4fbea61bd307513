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


@pytest.mark.parametrize("N", [1024, 512])
def test_cca_16_lane_hashes_equal_larger_call(N):
    """Calls whose hashes run on 16 lanes per element against the rows of a call above that
    form's limit, a differing byte in every part of the ciphertext included."""
    import pqc_amd
    n, alg = 8200, f"newhope{N}"
    rng = np.random.default_rng(N + 1)
    kc = rng.integers(0, 256, (n, 64), dtype=np.uint8)
    ec = rng.integers(0, 256, (n, 32), dtype=np.uint8)
    ctx = pqc_amd.Context([alg], max_batch=n)
    print("newhope cca large", N, flush=True)
    pk, sk = ctx.keypair_host(alg, kc)
    ct, ss = ctx.enc_host(alg, pk, ec)
    bad = ct.copy()
    for i, col in enumerate((0, 14 * N // 8 - 1, 14 * N // 8, 17 * N // 8 - 1, 17 * N // 8, 17 * N // 8 + 31)):
        bad[i::7, col] ^= 0x80 >> i
    want = ctx.dec_host(alg, bad, sk)
    ok = (bad == ct).all(axis=1)
    assert ok.any() and (want[ok] == ss[ok]).all() and (want[~ok] != ss[~ok]).any(axis=1).all()
    for m in (1, 3, 4, 5, 63, 1025, 4097, 8192):
        print("newhope cca 16 lanes", N, m, flush=True)
        pk2, sk2 = ctx.keypair_host(alg, kc[:m])
        ct2, ss2 = ctx.enc_host(alg, pk[:m], ec[:m])
        assert (pk2 == pk[:m]).all() and (sk2 == sk[:m]).all()
        assert (ct2 == ct[:m]).all() and (ss2 == ss[:m]).all()
        assert (ctx.dec_host(alg, bad[:m], sk[:m]) == want[:m]).all()
    ctx.close()
