"""The measured work: batched KEM calls as a program that uses this library makes them.

A server or a batch job holds keys, ciphertexts and coins on the GPU and calls the
engine's batch entry points (pqc_amd.Context) on them: a handful of requests where
latency counts, some hundreds to thousands where a serving loop closes a batch, tens of
thousands where a job works through a backlog.  Outputs are bytes, equal on every path.
"""
import math

import torch

import pqc_amd

FRODO = (15632, 31296, 15744, 24)  # pk, sk, ct, ss of FrodoKEM-976
KECCAK_OPS = 7440                  # two-input 32-bit operations of one Keccak-f[1600]
KYBER_K = {"kyber512": 2, "kyber768": 3, "kyber1024": 4}


class Buf:
    """A torch uint8 tensor on the GPU as the binding takes a device buffer."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel()


def listed():
    return [
        # one ciphertext of a handshake that waits for it: latency and launches only
        {"name": "kyber768_dec_1", "kind": "kyber", "op": "dec", "alg": "kyber768", "n": 1},
        # the batch a serving loop closes at some million requests/s, never a round number
        {"name": "kyber768_dec_761", "kind": "kyber", "op": "dec", "alg": "kyber768", "n": 761},
        # a middle batch of the largest parameter set
        {"name": "kyber1024_dec_6000", "kind": "kyber", "op": "dec", "alg": "kyber1024", "n": 6000},
        # the headline batch: a backlog of decapsulations, each under its own key
        {"name": "kyber768_dec_65536", "kind": "kyber", "op": "dec", "alg": "kyber768", "n": 65536},
        # clients' encapsulations, smallest set, ragged middle batch
        {"name": "kyber512_enc_2501", "kind": "kyber", "op": "enc", "alg": "kyber512", "n": 2501},
        # the large encapsulation batch
        {"name": "kyber768_enc_65536", "kind": "kyber", "op": "enc", "alg": "kyber768", "n": 65536},
        # key pairs made ahead of use
        {"name": "kyber1024_keypair_16384", "kind": "kyber", "op": "keypair", "alg": "kyber1024", "n": 16384},
        # mixed parameter sets 1:2:1, each request named by a descriptor: encapsulate, then decapsulate
        {"name": "kyber_mixed_65536", "kind": "mixed", "n": 65536},
        # FrodoKEM-976 ciphertexts under one resident key
        {"name": "frodo976_dec_4096", "kind": "frodo", "op": "dec", "n": 4096},
        # a small batch of FrodoKEM-976 encapsulations to one public key
        {"name": "frodo976_enc_501", "kind": "frodo", "op": "enc", "n": 501},
        # NewHope-1024 CPA: key pair, encryption and decryption of every element
        {"name": "newhope1024_cpa_16384", "kind": "newhope_cpa", "N": 1024, "n": 16384},
        # NewHope-512 CCA-KEM: encapsulation and decapsulation, ragged middle batch
        {"name": "newhope512_cca_3001", "kind": "newhope_cca", "N": 512, "n": 3001},
    ]


def _size(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(["kyber", "kyber", "kyber", "kyber", "mixed", "frodo", "newhope_cpa", "newhope_cca"])
    if kind == "kyber":
        alg = rng.choice(["kyber512", "kyber768", "kyber1024"])
        return {"kind": kind, "op": rng.choice(["dec", "dec", "enc", "keypair"]), "alg": alg,
                "n": _size(rng, 1, 65536 if alg != "kyber1024" else 49152)}
    if kind == "mixed":
        return {"kind": kind, "n": _size(rng, 3, 65536)}
    if kind == "frodo":
        return {"kind": kind, "op": rng.choice(["dec", "enc"]), "n": _size(rng, 1, 4096)}
    return {"kind": kind, "N": rng.choice([512, 1024]), "n": _size(rng, 1, 16384)}


def _bytes(gen, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, generator=gen).cuda()


def _empty(*shape):
    return torch.empty(shape, dtype=torch.uint8, device="cuda")


def _damage(gen, ct):
    """One ciphertext in 64 does not decrypt to what was sent (implicit rejection)."""
    n = ct.shape[0]
    hit = torch.randint(0, 64, (n,), generator=gen) == 0
    pos = torch.randint(0, ct.shape[1], (n,), generator=gen)
    rows = hit.nonzero().flatten().cuda()
    if rows.numel():
        cols = pos[hit].cuda()
        ct[rows, cols] ^= 1


def prepare(case, seed):
    gen = torch.Generator().manual_seed(seed)
    return {"kyber": _prepare_kyber, "mixed": _prepare_mixed, "frodo": _prepare_frodo,
            "newhope_cpa": _prepare_newhope_cpa, "newhope_cca": _prepare_newhope_cca}[case["kind"]](case, gen)


def _prepare_kem(alg, op, n, gen):
    """Inputs of one batched KEM operation with a key pair per element."""
    pkb, skb, ctb, ssb = pqc_amd.sizes(alg)
    ctx = pqc_amd.Context([alg], max_batch=n)
    st = {"ctx": ctx, "alg": alg, "op": op, "n": n}
    coins, pk, sk = _bytes(gen, n, 64), _empty(n, pkb), _empty(n, skb)
    st["coins"], st["pk"], st["sk"] = Buf(coins), Buf(pk), Buf(sk)
    if op != "keypair":
        ctx.keypair_derand(alg, n, st["pk"], st["sk"], st["coins"])
        st["coins"], st["ct"], st["ss"] = Buf(_bytes(gen, n, 32)), Buf(_empty(n, ctb)), Buf(_empty(n, ssb))
        if op in ("dec", "enc_dec"):
            ctx.enc_derand(alg, n, st["ct"], st["ss"], st["pk"], st["coins"])
        if op == "dec":
            _damage(gen, st["ct"].t)
        st["ss2"] = Buf(_empty(n, ssb))
    torch.cuda.synchronize()
    return st


def _prepare_kyber(case, gen):
    return dict(_prepare_kem(case["alg"], case["op"], case["n"], gen), kind="kem")


def _prepare_newhope_cca(case, gen):
    return dict(_prepare_kem("newhope%d" % case["N"], "enc_dec", case["n"], gen), kind="kem")


def _prepare_mixed(case, gen):
    n = case["n"]
    algs = torch.tensor([1, 2, 2, 3], dtype=torch.int32).repeat(n // 4 + 1)[:n][torch.randperm(n, generator=gen)]
    lay = pqc_amd.MixedLayout(algs.numpy())
    ctx = pqc_amd.Context(["kyber512", "kyber768", "kyber1024"], max_batch=n)
    st = {"kind": "mixed", "ctx": ctx, "n": n}
    for k in ("pk", "sk", "ct", "ss", "kcoins", "coins"):
        fill = _bytes(gen, lay.nbytes[k]) if k in ("coins", "kcoins") else torch.zeros(
            lay.nbytes[k], dtype=torch.uint8, device="cuda")
        st[k] = Buf(fill)
    st["ss2"] = Buf(torch.zeros_like(st["ss"].t))
    for a, cnt in lay.count.items():
        if cnt:
            part = [Buf(st[k].t[lay.region[k][a][0]:lay.region[k][a][0] + cnt * lay.elem[k][a]])
                    for k in ("pk", "sk", "kcoins")]
            ctx.keypair_derand(a, cnt, *part)
    for k, key in (("enc_reqs", "pk"), ("dec_reqs", "sk")):
        r = torch.frombuffer(bytearray(lay.requests(key).tobytes()), dtype=torch.uint8)
        st[k] = Buf(r.cuda())
    torch.cuda.synchronize()
    return st


def _prepare_frodo(case, gen):
    n, op = case["n"], case["op"]
    pkb, skb, ctb, ssb = FRODO
    ctx = pqc_amd.Context(["frodo976"], max_batch=n)
    pk, sk = Buf(_empty(1, pkb)), Buf(_empty(1, skb))
    ctx.frodo_keypair(1, pk, sk, Buf(_bytes(gen, 1, 64)))
    ctx.frodo_load_key(sk, True)
    st = {"kind": "frodo", "op": op, "ctx": ctx, "n": n, "pk": pk, "sk": sk, "mu": Buf(_bytes(gen, n, 24)),
          "ct": Buf(_empty(n, ctb)), "ss": Buf(_empty(n, ssb))}
    if op == "dec":
        ctx.frodo_enc(n, st["ct"], st["ss"], st["mu"])
        _damage(gen, st["ct"].t)
    torch.cuda.synchronize()
    return st


def _prepare_newhope_cpa(case, gen):
    n, N = case["n"], case["N"]
    poly = 14 * N // 8
    ctx = pqc_amd.Context(["newhope%dcpa" % N], max_batch=n)
    st = {"kind": "newhope_cpa", "ctx": ctx, "n": n, "N": N}
    for k in ("seeds", "msgs", "coins"):
        st[k] = Buf(_bytes(gen, n, 32))
    for k, b in (("pk", poly + 32), ("sk", poly), ("ct", poly + 3 * N // 8), ("out", 32)):
        st[k] = Buf(_empty(n, b))
    torch.cuda.synchronize()
    return st


def run(st):
    ctx, n, kind = st["ctx"], st["n"], st["kind"]
    if kind == "kem":
        alg, op = st["alg"], st["op"]
        if op == "keypair":
            ctx.keypair_derand(alg, n, st["pk"], st["sk"], st["coins"])
            return [st["pk"].t, st["sk"].t]
        if op == "dec":
            ctx.dec(alg, n, st["ss2"], st["ct"], st["sk"])
            return [st["ss2"].t]
        ctx.enc_derand(alg, n, st["ct"], st["ss"], st["pk"], st["coins"])
        if op == "enc":
            return [st["ct"].t, st["ss"].t]
        ctx.dec(alg, n, st["ss2"], st["ct"], st["sk"])
        return [st["ct"].t, st["ss"].t, st["ss2"].t]
    if kind == "mixed":
        ctx.kem_enc_mixed(n, st["enc_reqs"], st["ct"], st["pk"], st["ss"], st["coins"])
        ctx.kem_dec_mixed(n, st["dec_reqs"], st["ct"], st["sk"], st["ss2"])
        return [st["ct"].t, st["ss"].t, st["ss2"].t]
    if kind == "frodo":
        if st["op"] == "enc":
            ctx.frodo_enc(n, st["ct"], st["ss"], st["mu"])
            return [st["ct"].t, st["ss"].t]
        ctx.frodo_dec(n, st["ss"], st["ct"])
        return [st["ss"].t]
    N = st["N"]
    ctx.newhope_keypair(n, st["pk"], st["sk"], st["seeds"], N=N)
    ctx.newhope_enc(n, st["ct"], st["msgs"], st["pk"], st["coins"], N=N)
    ctx.newhope_dec(n, st["out"], st["ct"], st["sk"], N=N)
    return [st["pk"].t, st["sk"].t, st["ct"].t, st["out"].t]


def _perms_kyber(k, op):
    """Keccak-f[1600] permutations of one Kyber operation (a matrix entry takes four SHAKE128 blocks)."""
    pkb, _, ctb, _ = pqc_amd.sizes({2: "kyber512", 3: "kyber768", 4: "kyber1024"}[k])
    mat, hpk, hct = 4 * k * k, pkb // 136 + 1, ctb // 136 + 1
    if op == "keypair":
        return 1 + mat + 2 * k + hpk
    if op == "enc":
        return 1 + hpk + 1 + mat + 2 * k + 1 + hct + 1
    return 1 + mat + 2 * k + 1 + hct + 1


def work(case):
    """Bytes: inputs and outputs once.  Operations: the Keccak permutations' 32-bit operations, and
    for FrodoKEM-976 the product by the shared matrix."""
    n, kind = case["n"], case["kind"]
    if kind == "kyber":
        pkb, skb, ctb, ssb = pqc_amd.sizes(case["alg"])
        b = {"keypair": pkb + skb + 64, "enc": pkb + ctb + ssb + 32, "dec": ctb + skb + ssb}[case["op"]]
        return {"bytes": n * b, "flops": n * _perms_kyber(KYBER_K[case["alg"]], case["op"]) * KECCAK_OPS}
    if kind == "mixed":
        b = f = 0.0
        for share, alg in ((0.25, "kyber512"), (0.5, "kyber768"), (0.25, "kyber1024")):
            pkb, skb, ctb, ssb = pqc_amd.sizes(alg)
            b += share * (pkb + ctb + ssb + 32 + ctb + skb + ssb)
            f += share * (_perms_kyber(KYBER_K[alg], "enc") + _perms_kyber(KYBER_K[alg], "dec"))
        return {"bytes": int(n * b), "flops": int(n * f * KECCAK_OPS)}
    if kind == "frodo":
        pkb, skb, ctb, ssb = FRODO
        perms = 1 + 231 + ctb // 136 + 1
        mac = 2 * 8 * 976 * 976 + 2 * 8 * 976 * 8 * (2 if case["op"] == "dec" else 1)
        b = n * (ctb + ssb + (0 if case["op"] == "dec" else 24)) + (skb if case["op"] == "dec" else pkb) + 2 * 976 * 976
        return {"bytes": b, "flops": n * (perms * KECCAK_OPS + mac)}
    N = case["N"]
    poly, ct = 14 * N // 8, 14 * N // 8 + 3 * N // 8
    s = N // 64  # SHAKE streams of one polynomial
    if kind == "newhope_cpa":
        b = (32 + 2 * poly + 32) + (32 + 32 + poly + 32 + ct) + (ct + poly + 32)
        return {"bytes": n * b, "flops": n * (1 + 3 * s + 4 * s) * KECCAK_OPS}
    pkb, skb, ctb, ssb = pqc_amd.sizes("newhope%d" % N)
    b = (pkb + 32 + ctb + ssb) + (ctb + skb + ssb)
    hashes = 1 + pkb // 136 + 1 + 1 + ctb // 136 + 1 + 1 + 1 + ctb // 136 + 1 + 1
    return {"bytes": n * b, "flops": n * (8 * s + hashes) * KECCAK_OPS}
