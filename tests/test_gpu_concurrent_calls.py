"""Calls of several contexts on streams of their own share the GPU: a call that fills the
SIMDs with one wave each leaves room for the others' waves."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_four_frodo_encapsulation_calls_overlap():
    """4096 FrodoKEM-976 encapsulations are 1024 serial chains on 16 lanes each, one per
    SIMD.  A wave issues in under a quarter of its SIMD's cycles, so four calls side by
    side take well below the time of four in a row (where a wave keeps its SIMD to itself,
    just that time)."""
    import pqc_amd
    n, calls = 4096, 4
    rng = np.random.default_rng(3)
    pk = pqc_amd.DeviceBuffer(15632)
    sk = pqc_amd.DeviceBuffer(31296)
    # streams are put on four hardware queues, and two on one queue do not overlap: the best
    # of some sets of four counts
    streams = [pqc_amd.Stream() for _ in range(8)]
    sets = [streams[:4], streams[4:], streams[::2], streams[1::2]]
    runs, keep = [], []
    for i in range(calls):
        ctx = pqc_amd.Context(["frodo976"], max_batch=n)
        if i == 0:
            ctx.frodo_keypair(1, pk, sk, pqc_amd.DeviceBuffer.from_array(rng.integers(0, 256, 64, dtype=np.uint8)))
        ctx.frodo_load_key(pk, False)
        mu = pqc_amd.DeviceBuffer.from_array(rng.integers(0, 256, (n, 24), dtype=np.uint8))
        ct, ss = pqc_amd.DeviceBuffer(n * 15744), pqc_amd.DeviceBuffer(n * 24)
        keep.append((ctx, mu, ct, ss))
        runs.append(lambda st, ctx=ctx, mu=mu, ct=ct, ss=ss: ctx.frodo_enc(n, ct, ss, mu, stream=st))

    def in_a_row(sts):
        t = time.perf_counter()
        for run, st in zip(runs, sts):
            run(st)
            st.synchronize()
        return time.perf_counter() - t

    def side_by_side(sts):
        t = time.perf_counter()
        for run, st in zip(runs, sts):
            run(st)
        for st in sts:
            st.synchronize()
        return time.perf_counter() - t

    print("frodo enc", calls, "x", n, flush=True)
    for _ in range(8):
        side_by_side(sets[0])
    row = min(in_a_row(sets[0]) for _ in range(5))
    side = [min(side_by_side(sts) for _ in range(5)) for sts in sets]
    print("in a row %.2f ms, side by side" % (row * 1e3), ["%.2f" % (t * 1e3) for t in side], flush=True)
    assert min(side) < 0.85 * row
    for k in keep:
        k[0].close()


def test_sixteen_lane_calls_of_every_workgroup_shape():
    """FrodoKEM-976 and NewHope CCA calls around the batch sizes where a workgroup's waves
    go from one to four to eight, against the rows of one larger call."""
    import pqc_amd
    rng = np.random.default_rng(4)
    n = 4096
    ctx = pqc_amd.Context(["frodo976"], max_batch=n)
    pk, sk = ctx.frodo_keypair_host(rng.integers(0, 256, (1, 64), dtype=np.uint8))
    mu = rng.integers(0, 256, (n, 24), dtype=np.uint8)
    ct, ss = ctx.frodo_enc_host(pk[0], mu)
    ct[::9, 77] ^= 2
    want = ctx.frodo_dec_host(sk[0], ct)
    assert (want[1:9] == ss[1:9]).all() and (want[::9] != ss[::9]).any(axis=1).all()
    for m in (1024, 1025, 1029, 2048, 2049, 2053, 4093):
        print("frodo", m, flush=True)
        ct2, ss2 = ctx.frodo_enc_host(pk[0], mu[:m])
        assert (ss2 == ss[:m]).all() and (ct2[1:9] == ct[1:9]).all()
        assert (ctx.frodo_dec_host(sk[0], ct[:m]) == want[:m]).all()
    ctx.close()
    n = 8200
    ctx = pqc_amd.Context(["newhope512"], max_batch=n)
    kc, ec = (rng.integers(0, 256, (n, b), dtype=np.uint8) for b in (64, 32))
    pk, sk = ctx.keypair_host("newhope512", kc)
    ct, ss = ctx.enc_host("newhope512", pk, ec)
    ct[::9, 77] ^= 2
    want = ctx.dec_host("newhope512", ct, sk)
    for m in (2048, 2049, 2061, 4096, 4097, 4109, 8191):
        print("newhope512", m, flush=True)
        pk2, sk2 = ctx.keypair_host("newhope512", kc[:m])
        ct2, ss2 = ctx.enc_host("newhope512", pk[:m], ec[:m])
        assert (pk2 == pk[:m]).all() and (sk2 == sk[:m]).all()
        assert (ss2 == ss[:m]).all() and (ct2[1:9] == ct[1:9]).all()
        assert (ctx.dec_host("newhope512", ct[:m], sk[:m]) == want[:m]).all()
    ctx.close()
