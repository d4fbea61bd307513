"""Mixed Kyber batches a little above the dense per-request limits take the faster form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_mixed_decapsulation_of_1400_takes_the_faster_form():
    import pqc_amd as pqc
    from pqc_amd import tuner as T
    n, rng = 1400, np.random.default_rng(7)
    lay = pqc.MixedLayout(np.array([1, 2, 2, 3] * (n // 4), np.int32)[rng.permutation(n)])
    ctx, st = pqc.Context(["kyber512", "kyber768", "kyber1024"], max_batch=n), pqc.Stream()
    ct, sk = (pqc.DeviceBuffer.from_array(rng.integers(0, 256, lay.nbytes[k], dtype=np.uint8)) for k in ("ct", "sk"))
    ss = pqc.DeviceBuffer.from_array(np.zeros(lay.nbytes["ss"], np.uint8))
    reqs = pqc.DeviceBuffer.from_array(np.frombuffer(lay.requests("sk").tobytes(), np.uint8))
    forms = {"default": 0, "per request": 65536, "stages": -1}
    ms, out = {name: [] for name in forms}, {}
    for _ in range(40):  # in turn: clocks that settle meanwhile favour none
        for name, lim in forms.items():
            T.put_tuning(ctx, lowlat_max=lim)
            a, b = pqc.Event(), pqc.Event()
            a.record(st)
            ctx.kem_dec_mixed(n, reqs, ct, sk, ss, stream=st)
            b.record(st)
            b.synchronize()
            ms[name].append(a.elapsed_ms(b))
            out[name] = ss.download((lay.nbytes["ss"],))
    ms = {name: min(t) for name, t in ms.items()}
    print({name: "%.1f us" % (t * 1e3) for name, t in ms.items()}, flush=True)
    assert (out["default"] == out["stages"]).all() and (out["default"] == out["per request"]).all()
    assert ms["default"] <= 1.12 * min(ms["per request"], ms["stages"])
    ctx.close()
