"""The Keccak lane layout of FrodoKEM-976's decapsulation stream: which one the tuning knob
selects (host code), and the same bytes under each of them."""
import numpy as np
import pytest


def test_knob_selects_the_layout():
    """frodo_lane_min: 0 and thresholds leave calls of up to 4096 requests on 16 lanes per
    state, -1 is lane pairs at every size."""
    from pqc_amd import tuner as T
    t = T.Tuning(plain_block=256, newhope_block=128, fused_waves_per_cu=4, frodo_stream_block=64)
    # lane_min, n -> (16 lanes, one lane)
    for lane_min, n, want in ((0, 1, (1, 0)), (0, 4096, (1, 0)), (0, 4097, (0, 0)), (0, 49152, (0, 1)),
                              (-1, 1, (0, 0)), (-1, 4096, (0, 0)), (-1, 65536, (0, 0)),
                              (1, 1, (0, 1)), (2000, 1999, (1, 0)), (2000, 2000, (0, 1))):
        t.frodo_lane_min = lane_min
        f = T.features(T.request("frodo", n, op=2), t)
        assert (f[9], f[10]) == want, (lane_min, n)


@pytest.mark.gpu
def test_layouts_give_the_same_bytes_and_the_tuner_measures_each():
    import pqc_amd as pqc
    from pqc_amd import tuner as T
    n, rng = 2050, np.random.default_rng(6)
    ctx, st = pqc.Context(["frodo976"], max_batch=n), pqc.Stream()
    pk, sk = ctx.frodo_keypair_host(rng.integers(0, 256, (1, 64), dtype=np.uint8))
    ct, ss = ctx.frodo_enc_host(pk[0], rng.integers(0, 256, (n, 24), dtype=np.uint8))
    ct[::7, 40] ^= 1
    want = ctx.frodo_dec_host(sk[0], ct)
    assert (want[1:7] == ss[1:7]).all() and (want[::7] != ss[::7]).any(axis=1).all()
    for lane_min in (-1, 1, 0):
        T.put_tuning(ctx, frodo_lane_min=lane_min)
        for m in (1, 33, n):
            print("frodo layout", lane_min, m, flush=True)
            assert (ctx.frodo_dec_host(sk[0], ct[:m]) == want[:m]).all()
    # six candidates at 512 requests, one of them on 16 lanes, whose block size plays no part
    d_ct, d_ss = pqc.DeviceBuffer.from_array(ct[:512]), pqc.DeviceBuffer(512 * 24)
    res = T.autotune(ctx, T.request("frodo", 512, op=2, budget=0, reps=3),
                     lambda s: ctx.frodo_dec(512, d_ss, d_ct, stream=s), st)
    x, y = T.samples(ctx)
    print("ms", np.exp(y), res.best.frodo_lane_min, flush=True)
    assert res.measured == len(np.unique(x, axis=0)) == 6
    assert x[:, 9].sum() == 1 and x[:, 10].sum() == 2
    assert (d_ss.download((512, 24)) == want[:512]).all()
    ctx.close()
