"""Graph mode of the serving loop with batches that alternate between sizes whose kernels
differ: every batch's results against a direct call, with the executables of the other
sizes kept and updated in between."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("alg,sizes", [("kyber768", (900, 2000, 1, 1537, 1536, 3000)),
                                       ("frodo976", (3, 1030, 520, 1500, 4))])
def test_graph_batches_of_alternating_sizes(alg, sizes):
    import pqc_amd as pqc
    from pqc_amd.server import RequestSet, Server
    keys, rng = 8, np.random.default_rng(9)
    srv = Server([alg], keys_per_alg=keys, max_batch=max(sizes), slots=1, arena_bytes=64 << 20, max_wait_us=10000,
                 graph=True)
    sks = np.stack([srv.key(alg, i)[1] for i in range(keys)])
    ctx = pqc.Context([alg], max_batch=max(sizes))
    skb, ctb, ssb = sks.shape[1], pqc.sizes(alg)[2], pqc.sizes(alg)[3]
    sets = []
    for n in sizes:
        kid = rng.integers(0, keys, n).astype(np.uint32)
        rs = RequestSet.random(np.full(n, pqc.kem.alg_id(alg), np.int32), np.full(n, 2, np.int32), kid, rng)
        ct = rs.inbuf[:n * ctb].reshape(n, ctb)
        if alg == "frodo976":  # one key per call: its rows
            want = np.empty((n, ssb), np.uint8)
            for i in range(keys):
                if (kid == i).any():
                    want[kid == i] = ctx.frodo_dec_host(sks[i], ct[kid == i])
        else:
            want = ctx.dec_host(alg, ct, sks[kid].reshape(n, skb))
        sets.append((rs, want))
    for rep in range(4):
        for rs, want in sets:
            rs.outbuf[:] = 0
            print(alg, "rep", rep, "n", rs.n, flush=True)
            srv.submit(rs.reqs)
            srv.drain()
            done = srv.poll(8192)
            assert len(done) == rs.n and all(c.status == 0 for c in done)
            assert (rs.outbuf[:rs.n * ssb].reshape(rs.n, ssb) == want).all()
    srv.close()
    ctx.close()
