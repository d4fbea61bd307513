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
