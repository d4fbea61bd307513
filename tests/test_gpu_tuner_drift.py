"""The autotuner on a workload whose first runs are slower than the later ones, as a GPU's
are after an idle phase."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_slow_first_runs_do_not_change_the_pick():
    """The configuration in use does 10 units of work a run, every other one 11; the first
    8 runs do a third more.  Measured first and once, the configuration in use would look
    slower than those measured after the slow phase."""
    import pqc_amd as pqc
    from pqc_amd import tuner as T
    rng = np.random.default_rng(2)
    ctx, st = pqc.Context(["kyber768"], max_batch=64), pqc.Stream()
    pk, sk, ct, ss = (pqc.DeviceBuffer(64 * b) for b in (1184, 2400, 1088, 32))
    ctx.keypair_derand("kyber768", 64, pk, sk, pqc.DeviceBuffer.from_array(rng.integers(0, 256, (64, 64), dtype=np.uint8)))
    ct.upload(rng.integers(0, 256, (64, 1088), dtype=np.uint8))
    start = T.get_tuning(ctx).fused_waves_per_cu
    runs = []

    def run(s):
        mine = T.get_tuning(ctx).fused_waves_per_cu
        units = 30 if mine == start else 33  # one unit: a call of 64 requests, whose kernel the knob does not touch
        runs.append(mine)
        for _ in range(units * 4 // 3 if len(runs) <= 8 else units):
            ctx.dec("kyber768", 64, ss, ct, sk, stream=s)

    res = T.autotune(ctx, T.request("fused_kyber", 64, k=3, op=2, budget=0, reps=3), run, st)
    x, y = T.samples(ctx)
    print("runs", len(runs), "ms", np.exp(y), "pick", res.best.fused_waves_per_cu, flush=True)
    assert res.measured == 4 and len(y) == 4
    assert res.best.fused_waves_per_cu == start
    assert T.get_tuning(ctx).fused_waves_per_cu == start
    ctx.close()


def test_a_failing_run_keeps_the_samples_before_it():
    """A workload that fails in the third candidate's first run: the error is reported, the
    configuration in use stays, and the two candidates timed before it stay as samples."""
    import pqc_amd as pqc
    from pqc_amd import tuner as T
    ctx, st = pqc.Context(["kyber768"], max_batch=1), pqc.Stream()
    sk, ct, ss = (pqc.DeviceBuffer.from_array(np.zeros(b, np.uint8)) for b in (2400, 1088, 32))
    start = T.get_tuning(ctx).as_dict()
    seen = []

    def run(s):
        w = T.get_tuning(ctx).fused_waves_per_cu
        if w not in seen:
            seen.append(w)
            if len(seen) == 3:
                raise ValueError("no")
        ctx.dec("kyber768", 1, ss, ct, sk, stream=s)

    with pytest.raises(ValueError):
        T.autotune(ctx, T.request("fused_kyber", 1, k=3, op=2, budget=0, reps=3), run, st)
    assert len(T.samples(ctx)[1]) == 2
    assert T.get_tuning(ctx).as_dict() == start
    ctx.close()
