"""Kyber contexts whose memory budget leaves short passes, or none, for the staged kernels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ALG = {2: "kyber512", 3: "kyber768", 4: "kyber1024"}


def budget_for(pqc, algs, kmax, n, passes_of):
    """Budget of a context for n requests of `algs` (largest K kmax) whose stages hold
    passes_of requests (0: no stages)."""
    full = pqc.Context(algs, max_batch=n)
    total = full.device_bytes
    full.close()
    ld = (n + 63) // 64 * 64

    def scratch(stage):
        rows = stage + 128 if stage else 0
        return (2 * kmax + 1) * 128 * max(ld, rows) + rows * (512 * kmax * kmax + 128)

    return total - scratch(ld) + scratch(passes_of)


def best_ms(pqc, st, run, reps=5):
    run()
    st.synchronize()
    out = []
    for _ in range(reps):
        a, b = pqc.Event(), pqc.Event()
        a.record(st)
        run()
        b.record(st)
        b.synchronize()
        out.append(a.elapsed_ms(b))
    return min(out)


def test_a_small_budget_is_no_slower_than_none_for_stages():
    """A budget with room for passes of 256 requests must not cost more time than one with
    room for no stages at all (64 passes of at least ~0.1 ms against one tile launch)."""
    import pqc_amd as pqc
    n, k = 16384, 3
    rng = np.random.default_rng(1)
    st = pqc.Stream()
    coins = pqc.DeviceBuffer.from_array(rng.integers(0, 256, (n, 64), dtype=np.uint8))
    ec = pqc.DeviceBuffer.from_array(rng.integers(0, 256, (n, 32), dtype=np.uint8))
    pk, sk, ct = pqc.DeviceBuffer(n * 1184), pqc.DeviceBuffer(n * 2400), pqc.DeviceBuffer(n * 1088)
    ss, ss2 = pqc.DeviceBuffer(n * 32), pqc.DeviceBuffer(n * 32)
    ms = {}
    for stage in (0, 256):
        ctx = pqc.Context([ALG[k]], max_batch=n, hbm_budget=budget_for(pqc, [ALG[k]], k, n, stage))
        ms[stage] = [best_ms(pqc, st, lambda: ctx.keypair_derand(ALG[k], n, pk, sk, coins, stream=st)),
                     best_ms(pqc, st, lambda: ctx.enc_derand(ALG[k], n, ct, ss, pk, ec, stream=st)),
                     best_ms(pqc, st, lambda: ctx.dec(ALG[k], n, ss2, ct, sk, stream=st))]
        assert (ss2.download((n, 32)) == ss.download((n, 32))).all()
        ctx.close()
        print("passes of", stage, ["%.3f ms" % t for t in ms[stage]], flush=True)
    assert all(a <= 1.5 * b for a, b in zip(ms[256], ms[0]))


@pytest.mark.parametrize("k", [2, 3, 4])
def test_several_passes_give_the_bytes_of_one(k):
    """3000 requests in passes of 1472 (two and a ragged third) and, with no room for stages,
    in tiles, against one pass."""
    import pqc_amd as pqc
    from pqc_amd import tuner as T
    n, rng = 3000, np.random.default_rng(20 + k)
    kc, ec = (rng.integers(0, 256, (n, b), dtype=np.uint8) for b in (64, 32))
    want = None
    for stage in (3008, 1472, 0):
        print("passes k", k, "of", stage, flush=True)
        ctx = pqc.Context([ALG[k]], max_batch=n, hbm_budget=budget_for(pqc, [ALG[k]], k, n, stage))
        T.put_tuning(ctx, lowlat_max=-1)
        bufs = [pqc.DeviceBuffer(n * b) for b in (*pqc.sizes(ALG[k]), 32)]
        pk, sk, ct, ss, ss2 = bufs
        ctx.keypair_derand(ALG[k], n, pk, sk, pqc.DeviceBuffer.from_array(kc))
        ctx.enc_derand(ALG[k], n, ct, ss, pk, pqc.DeviceBuffer.from_array(ec))
        damaged = ct.download((n, ct.nbytes // n))
        damaged[5::7, 11] ^= 8
        bad = pqc.DeviceBuffer.from_array(damaged)
        ctx.dec(ALG[k], n, ss2, bad, sk)
        assert ctx.take_status() == 0
        got = [b.download((n, b.nbytes // n)) for b in bufs]
        ctx.close()
        if want is None:
            want = got
            ok = np.ones(n, bool)
            ok[5::7] = False
            assert (got[4][ok] == got[3][ok]).all() and (got[4][~ok] != got[3][~ok]).any(axis=1).all()
        assert all((a == b).all() for a, b in zip(want, got))


def test_mixed_batch_in_several_passes():
    """A mixed batch in passes of 1472 and in tiles, against one pass: descriptors of a set
    the context does not hold, in the first and the last pass, are skipped and reported."""
    import pqc_amd as pqc
    from pqc_amd import tuner as T
    n, rng, algs = 3000, np.random.default_rng(31), ["kyber512", "kyber768", "kyber1024"]
    lay = pqc.MixedLayout(np.array([1, 2, 2, 3] * (n // 4), np.int32)[rng.permutation(n)], rng)
    fill = {kind: rng.integers(0, 256, lay.nbytes[kind], dtype=np.uint8) for kind in ("pk", "sk", "coins")}
    wrong = [3, 1500, 2944, n - 1]
    want = None
    for stage in (3008, 1472, 0):
        print("mixed passes of", stage, flush=True)
        ctx = pqc.Context(algs, max_batch=n, hbm_budget=budget_for(pqc, algs, 4, n, stage))
        T.put_tuning(ctx, lowlat_max=-1)
        ar = pqc.DeviceArenas(lay)
        for kind, v in fill.items():
            ar.buf[kind].upload(v)
        for kind in ("ct", "ss"):
            ar.buf[kind].upload(np.zeros(lay.nbytes[kind], np.uint8))
        out = []
        for key, call in (("pk", lambda r: ctx.kem_enc_mixed(n, r, ar.buf["ct"], ar.buf["pk"], ar.buf["ss"],
                                                             ar.buf["coins"])),
                          ("sk", lambda r: ctx.kem_dec_mixed(n, r, ar.buf["ct"], ar.buf["sk"], ar.buf["ss"]))):
            reqs = lay.requests(key)
            call(pqc.DeviceBuffer.from_array(reqs))
            assert ctx.take_status() == 0
            out += [ar.download("ct"), ar.download("ss")]
            reqs["alg"][wrong] = 5
            ar.buf["ss"].upload(np.zeros(lay.nbytes["ss"], np.uint8))
            call(pqc.DeviceBuffer.from_array(reqs))
            assert ctx.take_status() == 2
            out.append(ar.download("ss"))
            assert all(not lay.element(out[-1], "ss", i).any() for i in wrong)
            assert all((lay.element(out[-1], "ss", i) == lay.element(out[-2], "ss", i)).all() for i in (0, 1499, 2999 - 1))
        ctx.close()
        want = want or out
        assert all((a == b).all() for a, b in zip(want, out))


def test_batch_above_one_full_pass():
    """65600 Kyber-512 requests: a pass of 65536 and one of 64, against calls of the last 128
    rows alone."""
    import pqc_amd as pqc
    n, alg, rng = 65600, "kyber512", np.random.default_rng(41)
    ctx = pqc.Context([alg], max_batch=n)
    pkb, skb, ctb, _ = pqc.sizes(alg)
    coins, ec = (rng.integers(0, 256, (n, b), dtype=np.uint8) for b in (64, 32))
    pk, sk, ct, ss, ss2 = (pqc.DeviceBuffer(n * b) for b in (pkb, skb, ctb, 32, 32))
    print("full pass and one more", n, flush=True)
    ctx.keypair_derand(alg, n, pk, sk, pqc.DeviceBuffer.from_array(coins))
    ctx.enc_derand(alg, n, ct, ss, pk, pqc.DeviceBuffer.from_array(ec))
    ctx.dec(alg, n, ss2, ct, sk)
    assert ctx.take_status() == 0
    s = ss.download((n, 32))
    assert (ss2.download((n, 32)) == s).all()
    pk2, sk2 = ctx.keypair_host(alg, coins[-128:])
    ct2, s2 = ctx.enc_host(alg, pk2, ec[-128:])
    assert (pk.download((n, pkb))[-128:] == pk2).all() and (sk.download((n, skb))[-128:] == sk2).all()
    assert (ct.download((n, ctb))[-128:] == ct2).all() and (s[-128:] == s2).all()
    ctx.close()
