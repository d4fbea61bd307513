"""Staged Kyber kernels (sponge stages, matrix-core product stages) at the edges of
their groups of 16, tiles of 64 and persistent grids, and the one-workgroup-per-request
kernels, bit-exact against the CPU oracle."""
import sys

import numpy as np
import pytest

from tests import oracle_lib as O

pytestmark = pytest.mark.gpu

ALG = {2: "kyber512", 3: "kyber768", 4: "kyber1024"}
SIZES = [1, 15, 16, 17, 63, 64, 65, 193]


@pytest.fixture(scope="module")
def pqc():
    import pqc_amd
    return pqc_amd


def staged_ctx(pqc, k, n, grid):
    from pqc_amd import tuner as T
    ctx = pqc.Context([ALG[k]], max_batch=n)
    T.put_tuning(ctx, lowlat_max=-1)  # no batch is too small for the stages
    ctx.set_tuning(grid=grid)
    return ctx


def inputs(k, n, seed):
    """Valid key pairs and ciphertexts, a third of the ciphertexts damaged, and every
    fourth secret key and ciphertext of arbitrary bytes (12-bit values up to 4095)."""
    rng = np.random.default_rng(seed)
    pk, sk = O.kyber_batch("keypair", k, [rng.integers(0, 256, (n, 64), dtype=np.uint8)])
    ct, _ = O.kyber_batch("enc", k, [pk, rng.integers(0, 256, (n, 32), dtype=np.uint8)])
    ct[::3, rng.integers(0, ct.shape[1])] ^= 1 << int(rng.integers(0, 8))
    sk[3::4] = rng.integers(0, 256, sk[3::4].shape, dtype=np.uint8)
    ct[3::8] = rng.integers(0, 256, ct[3::8].shape, dtype=np.uint8)
    pk[3::4] = rng.integers(0, 256, pk[3::4].shape, dtype=np.uint8)
    return pk, sk, ct


@pytest.mark.parametrize("grid", [0, 1])
@pytest.mark.parametrize("k", [2, 3, 4])
def test_staged_decaps_vs_oracle(pqc, k, grid):
    ctx = staged_ctx(pqc, k, max(SIZES), grid)
    for n in SIZES:
        print("staged decaps k", k, "n", n, "grid", grid, flush=True)
        sys.stdout.flush()
        _, sk, ct = inputs(k, n, 1000 * k + n)
        want = O.kyber_batch("dec", k, [ct, sk])
        got = ctx.dec_host(ALG[k], ct, sk)
        assert (got == want).all(), np.nonzero((got != want).any(axis=1))[0][:8]
    ctx.close()


@pytest.mark.parametrize("grid", [0, 1])
@pytest.mark.parametrize("k", [2, 3, 4])
def test_staged_keypair_and_encaps_vs_oracle(pqc, k, grid):
    ctx = staged_ctx(pqc, k, max(SIZES), grid)
    for n in SIZES:
        print("staged keypair and encaps k", k, "n", n, "grid", grid, flush=True)
        rng = np.random.default_rng(2000 * k + n)
        coins = rng.integers(0, 256, (n, 64), dtype=np.uint8)
        pk, sk = ctx.keypair_host(ALG[k], coins)
        opk, osk = O.kyber_batch("keypair", k, [coins])
        assert (pk == opk).all() and (sk == osk).all()
        pk, _, _ = inputs(k, n, 3000 * k + n)  # every fourth public key of arbitrary bytes
        coins = rng.integers(0, 256, (n, 32), dtype=np.uint8)
        ct, ss = ctx.enc_host(ALG[k], pk, coins)
        oct_, oss = O.kyber_batch("enc", k, [pk, coins])
        assert (ct == oct_).all() and (ss == oss).all()
    ctx.close()


@pytest.mark.parametrize("k", [2, 3, 4])
def test_per_request_kernels_vs_oracle(pqc, k):
    sizes = [1, 5, 200]
    ctx = pqc.Context([ALG[k]], max_batch=max(sizes))
    for n in sizes:
        print("per-request kernels k", k, "n", n, flush=True)
        pk, sk, ct = inputs(k, n, 4000 * k + n)
        rng = np.random.default_rng(5000 * k + n)
        coins = rng.integers(0, 256, (n, 64), dtype=np.uint8)
        assert all((a == b).all() for a, b in zip(ctx.keypair_host(ALG[k], coins), O.kyber_batch("keypair", k, [coins])))
        c32 = np.ascontiguousarray(coins[:, :32])
        assert all((a == b).all() for a, b in zip(ctx.enc_host(ALG[k], pk, c32), O.kyber_batch("enc", k, [pk, c32])))
        assert (ctx.dec_host(ALG[k], ct, sk) == O.kyber_batch("dec", k, [ct, sk])).all()
    ctx.close()


@pytest.mark.parametrize("k", [2, 3, 4])
def test_hash_forms_agree_across_batch_sizes(pqc, k):
    """The stages hash on one lane, a lane pair or 16 lanes per request, by batch size: the
    rows of a call in one form against calls in the others, and against the oracle."""
    n, rng = 32800, np.random.default_rng(40 + k)
    ctx = staged_ctx(pqc, k, n, 0)
    kc = rng.integers(0, 256, (n, 64), dtype=np.uint8)
    ec = rng.integers(0, 256, (n, 32), dtype=np.uint8)
    print("hash forms k", k, "n", n, flush=True)
    pk, sk = ctx.keypair_host(ALG[k], kc)
    ct, ss = ctx.enc_host(ALG[k], pk, ec)
    bad = ct.copy()
    bad[::5, int(rng.integers(0, ct.shape[1]))] ^= 4
    want = ctx.dec_host(ALG[k], bad, sk)
    ok = (bad == ct).all(axis=1)
    assert (want[ok] == ss[ok]).all() and (want[~ok] != ss[~ok]).any(axis=1).all()
    for m in (5, 1027, 8192, 8193, 32768):
        print("hash forms k", k, "n", m, flush=True)
        pk2, sk2 = ctx.keypair_host(ALG[k], kc[:m])
        ct2, ss2 = ctx.enc_host(ALG[k], pk[:m], ec[:m])
        assert (pk2 == pk[:m]).all() and (sk2 == sk[:m]).all()
        assert (ct2 == ct[:m]).all() and (ss2 == ss[:m]).all()
        assert (ctx.dec_host(ALG[k], bad[:m], sk[:m]) == want[:m]).all()
    assert (O.kyber_batch("dec", k, [bad[:8], sk[:8]]) == want[:8]).all()
    ctx.close()


@pytest.mark.parametrize("k", [2, 4])
def test_budget_limits_staged_scratch(pqc, k):
    """A budget below the full scratch gets shorter passes, one that holds only the noise
    rows 64-request tiles, with the same bytes; less is refused."""
    n = 2000
    _, sk, ct = inputs(k, n, 70 + k)
    full = pqc.Context([ALG[k]], max_batch=n)
    total = full.device_bytes
    want = full.dec_host(ALG[k], ct, sk)
    full.close()
    d_ct, d_sk = pqc.DeviceBuffer.from_array(ct), pqc.DeviceBuffer.from_array(sk)
    ld = (n + 63) // 64 * 64
    stage = (ld + 128) * (512 * k * k + 128) + 128 * 128 * (2 * k + 1)
    for budget in (total, total - 1, total - stage // 3, total - stage):
        print("budget k", k, budget, flush=True)
        ctx = pqc.Context([ALG[k]], max_batch=n, hbm_budget=budget)
        assert ctx.device_bytes <= budget
        d_ss = pqc.DeviceBuffer(n * 32)
        ctx.dec(ALG[k], n, d_ss, d_ct, d_sk)
        ctx.take_status()
        assert (d_ss.download((n, 32)) == want).all()
        ctx.close()
    with pytest.raises(Exception):
        pqc.Context([ALG[k]], max_batch=n, hbm_budget=total - stage - 1)
