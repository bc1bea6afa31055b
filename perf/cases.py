"""Performance cases of the Groth16 prover core: what a prover, a KZG
committer or a caller of the transforms and multi-scalar products has this
library do, through the Python front end of the C ABI.

listed() names the fixed cases, draw(rng) gives one more of the same ranges,
prepare(case, seed) makes a case's inputs on the GPU, run(state) is one pass,
work(case) the bytes and operations a pass cannot do without, tolerance(case)
how close two implementations have to be (all results are whole numbers: field
elements, curve points, proof bytes), and exact(case, seed) the result in
Python integers where that takes seconds.
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuda-zkml_amd"))
import zkml_amd  # noqa: E402

R = zkml_amd.R_INT
Q = 0x30644E72E131A029B85045B68181585D97816A916871CA8D3C208C16D87CFD47
MONT = 1 << 256
MAD = 136  # 32-bit multiply-adds of one 256-bit Montgomery product (2 * 8^2 + 8)

_ctx = None


def context():
    """The process's context on GPU 0, which a program keeps."""
    global _ctx
    if _ctx is None:
        _ctx = zkml_amd.Context(0)
    return _ctx


class Buf:
    """A torch tensor as the front end's device buffer."""

    def __init__(self, t):
        self.t = t
        self.ptr = t.data_ptr()
        self.nbytes = t.numel() * t.element_size()


def device(words):
    """(n, k) uint64 words on the GPU."""
    return Buf(torch.from_numpy(np.ascontiguousarray(words).view(np.int64)).cuda())


def empty(*shape):
    return Buf(torch.empty(shape, dtype=torch.int64, device="cuda"))


# ------------------------------------------------------------------ cases
def listed():
    return [
        # one small transform: latency and launches (a 4096-row statement's domain)
        {"name": "ntt 2^12", "kind": "ntt", "log_n": 12, "op": "forward", "batch": 1},
        # the three coset inverses of a 2^16 domain in one call
        {"name": "coset inverse 2^16 x3", "kind": "ntt", "log_n": 16, "op": "coset inverse", "batch": 3},
        # the largest transform of the benchmark's configurations
        {"name": "ntt 2^22", "kind": "ntt", "log_n": 22, "op": "forward", "batch": 1},
        # a small G1 product, ragged: a statement of a few hundred rows
        {"name": "msm g1 1000", "kind": "msm", "n": 1000, "g2": False, "scalars": "uniform", "prepared": False},
        # one query of a 2^16 proof by itself
        {"name": "msm g1 2^16", "kind": "msm", "n": 1 << 16, "g2": False, "scalars": "uniform", "prepared": False},
        # witness values over a base set kept as records, ragged
        {"name": "msm g1 300007 witness", "kind": "msm", "n": 300007, "g2": False, "scalars": "witness",
         "prepared": True},
        # the benchmark's headline product
        {"name": "msm g1 2^20", "kind": "msm", "n": 1 << 20, "g2": False, "scalars": "uniform", "prepared": False},
        # the G2 query of a 2^16 proof by itself, ragged
        {"name": "msm g2 62779", "kind": "msm", "n": 62779, "g2": True, "scalars": "uniform", "prepared": False},
        # a KZG opening: synthetic division and a G1 product
        {"name": "kzg open 100000", "kind": "kzg", "degree": 100000},
        # a proof of the quantized MLP statement (domain 2^13)
        {"name": "prove mlp 2^13", "kind": "prove", "statement": "mlp", "constraints": 7933},
        # a proof of the private CNN statement (domain 2^16): the benchmark's headline proof
        {"name": "prove cnn 2^16", "kind": "prove", "statement": "cnn", "constraints": 62692},
        # a proof over uniform witness values, ragged, domain 2^18: bounded by its total work
        {"name": "prove synthetic 200001", "kind": "prove", "statement": "synthetic", "constraints": 200001},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ntt", "msm", "msm", "kzg", "prove"])
    if kind == "ntt":
        log_n = rng.randint(8, 22)
        batch = rng.choice([b for b in (1, 2, 3, 5) if b << log_n <= 1 << 22])
        op = rng.choice(["forward", "inverse", "coset forward", "coset inverse"])
        return {"kind": "ntt", "log_n": log_n, "op": op, "batch": batch}
    if kind == "msm":
        g2 = rng.random() < 0.35
        n = _log_uniform(rng, 300, 150000 if g2 else 1 << 20)
        return {"kind": "msm", "n": n, "g2": g2, "scalars": rng.choice(["uniform", "witness"]),
                "prepared": rng.random() < 0.5}
    if kind == "kzg":
        return {"kind": "kzg", "degree": _log_uniform(rng, 300, 400000)}
    return {"kind": "prove", "statement": "synthetic", "constraints": _log_uniform(rng, 1500, 200000)}


# ------------------------------------------------------------------ inputs
def words(vals):
    """Python ints below 2^256 as (n, 4) uint64 words."""
    b = b"".join(v.to_bytes(32, "little") for v in vals)
    return np.frombuffer(b, dtype=np.uint64).reshape(-1, 4).copy()


def ints(w):
    b = np.ascontiguousarray(w).tobytes()
    return [int.from_bytes(b[i:i + 32], "little") for i in range(0, len(b), 32)]


_small = None


def witness_scalars(n, rng):
    """What a witness holds (Montgomery words): 70% below 2^16, 10% small
    negatives, the rest uniform."""
    global _small
    if _small is None:
        _small = words([v * MONT % R for v in range(1 << 16)]), words([-v * MONT % R for v in range(1 << 16)])
    s = zkml_amd.random_fr(n, rng)
    u = rng.random(n)
    m = u < 0.7
    s[m] = _small[0][rng.integers(0, 1 << 16, size=int(m.sum()))]
    m = (u >= 0.7) & (u < 0.8)
    s[m] = _small[1][rng.integers(1, 1 << 16, size=int(m.sum()))]
    return s


def msm_inputs(case, seed):
    """(k, s): the points are k_i times the generator, s_i the scalars."""
    rng = np.random.default_rng([seed, case["n"]])
    k = zkml_amd.random_fr(case["n"], rng)
    s = (witness_scalars if case["scalars"] == "witness" else zkml_amd.random_fr)(case["n"], rng)
    return k, s


def ntt_inputs(case, seed):
    rng = np.random.default_rng([seed, case["log_n"], case["batch"]])
    return zkml_amd.random_fr(case["batch"] << case["log_n"], rng)


def kzg_inputs(case, seed):
    """tau, the coefficients (Montgomery words) and the point z (Montgomery words)."""
    rng = np.random.default_rng([seed, case["degree"]])
    tau = ints(zkml_amd.random_fr(1, rng))[0]
    return tau, zkml_amd.random_fr(case["degree"], rng), zkml_amd.random_fr(1, rng)[0]


COSET = 5  # the prover's coset shift


def statement(case, seed):
    """(num_constraints, num_variables, num_public, A, B, C, witness)."""
    rng = np.random.default_rng([seed, case["constraints"]])
    z = zkml_amd
    if case["statement"] == "synthetic":
        A, B, C, w = z.synthetic_r1cs(case["constraints"], 8, 1000, int(rng.integers(1 << 40)))
        return case["constraints"], w.shape[0], 8, A, B, C, w
    if case["statement"] == "mlp":
        # quantized 64 -> 32 -> 10, int8 weights, int32 biases, three samples
        def lin(i, o):
            return z.layer_linear(i, o, rng.integers(-127, 128, i * o), rng.integers(-2**31, 2**31, o))
        st = z.statement_v2([lin(64, 32), z.layer_relu_exact(32, 34, 8), lin(32, 10), z.layer_softmax(10)],
                            rng.integers(0, 17, (3, 64)))
    else:
        # 1x6x6 -> two 3x3 filters -> exact ReLU -> 4 scores, private model, inputs and outputs, routed
        st = z.statement_v2([z.layer_conv2d(1, 6, 6, 2, 3, 3, 1, 1, rng.integers(-3, 4, 18), rng.integers(-4, 5, 2)),
                             z.layer_relu_exact(72, 24, 2),
                             z.layer_linear(72, 4, rng.integers(-4, 5, 288), rng.integers(-4, 5, 4)),
                             z.layer_softmax(4)],
                            rng.integers(-8, 9, (2, 36)), model_tag=0xC0FFEE, private_input=True,
                            input_blinding=[int(v) for v in rng.integers(1, 1 << 40, 2)], private_model=True,
                            private_outputs=True, route_threshold=5)
    return st.nc, st.nv, st.npub, st.A, st.B, st.C, st.w


def points(k, n, g2):
    """The generator's multiples by the n scalars of k, complete on return (k
    is torch's memory, used on the context's stream)."""
    ctx = context()
    pts = empty(n, 16 if g2 else 8)
    (ctx.g2_generator_mul if g2 else ctx.g1_generator_mul)(k, n, pts)
    ctx.sync()
    return pts


def prepare(case, seed):
    ctx = context()
    if case["kind"] == "ntt":
        a = ntt_inputs(case, seed)
        return {"case": case, "in": device(a), "out": empty(*a.shape)}
    if case["kind"] == "msm":
        k, s = msm_inputs(case, seed)
        n, g2 = case["n"], case["g2"]
        st = {"case": case, "points": points(device(k), n, g2), "scalars": device(s)}
        if case["prepared"]:
            st["records"] = ctx.msm_prepare(st["points"], n, g2)
            ctx.sync()
        return st
    if case["kind"] == "kzg":
        tau, f, z = kzg_inputs(case, seed)
        p, powers = MONT % R, []
        for _ in range(case["degree"]):
            powers.append(p)
            p = p * tau % R
        srs = points(device(words(powers)), case["degree"], False)
        return {"case": case, "srs": srs, "f": device(f), "z": z}
    nc, nv, npub, A, B, C, w = statement(case, seed)
    r1cs = ctx.r1cs(nc, nv, npub, A, B, C)
    with tempfile.TemporaryDirectory() as td:
        pk_path = os.path.join(td, "pk.bin")
        ctx.setup(r1cs, 0xDEADBEEF42 + seed, pk_path, os.path.join(td, "vk.bin"))
        pk = ctx.load_pk(pk_path)
    ctx.sync()
    return {"case": case, "r1cs": r1cs, "pk": pk, "w": w, "npub": npub, "blind": 0xCAFEBABE + seed}


def run(st):
    ctx, case = context(), st["case"]
    if case["kind"] == "ntt":
        inv = "inverse" in case["op"]
        if case["op"].startswith("coset"):
            ctx.coset_ntt(st["out"], st["in"], case["log_n"], COSET, inverse=inv, batch=case["batch"])
        else:
            ctx.ntt(st["out"], st["in"], case["log_n"], inverse=inv, batch=case["batch"])
        return st["out"].t
    if case["kind"] == "msm":
        if case["prepared"]:
            f = ctx.msm_g2_prepared if case["g2"] else ctx.msm_g1_prepared
            return f(st["records"], st["scalars"], case["n"])
        return (ctx.msm_g2 if case["g2"] else ctx.msm_g1)(st["points"], st["scalars"], case["n"])
    if case["kind"] == "kzg":
        return ctx.kzg_open(st["srs"], st["f"], case["degree"], st["z"])
    proof, _ = ctx.prove(st["pk"], st["r1cs"], st["w"], st["npub"], st["blind"])
    return np.frombuffer(proof, dtype=np.uint8)


# ------------------------------------------------------------------ work
def msm_mults(n, g2=False):
    """Field multiplications of a signed-window product (the best window): 10
    per mixed addition, 14 per bucket-reduction addition, the combination; a
    multiplication over Fq2 is three over Fq."""
    def at(c):
        w = -(-255 // c)
        return n * w * 10 + w * (1 << (c - 1)) * 2 * 14 + w * (6 * c + 14)
    return min(at(c) for c in range(4, 22)) * (3 if g2 else 1)


def ntt_mults(log_n, batch, coset):
    return batch * ((1 << log_n) // 2 * log_n + (1 << log_n if coset else 0))


def work(case):
    if case["kind"] == "ntt":
        mults = ntt_mults(case["log_n"], case["batch"], case["op"] != "forward")
        return {"bytes": 64 * (case["batch"] << case["log_n"]), "flops": 2 * MAD * mults}
    if case["kind"] == "msm":
        return {"bytes": case["n"] * (32 + (128 if case["g2"] else 64)),
                "flops": 2 * MAD * msm_mults(case["n"], case["g2"])}
    if case["kind"] == "kzg":
        return {"bytes": case["degree"] * (32 + 64), "flops": 2 * MAD * (msm_mults(case["degree"]) + case["degree"])}
    m = case["constraints"]
    log_n = (m - 1).bit_length()
    mults = 3 * msm_mults(m) + msm_mults(m, True) + msm_mults(1 << log_n) + ntt_mults(log_n, 7, True)
    # the witness, five point queries, the rows' terms (about five of 36 bytes)
    return {"bytes": m * (32 + 4 * 64 + 128 + 5 * 36), "flops": 2 * MAD * mults}


def tolerance(case):
    return "exact"  # field elements, points and proof bytes are whole numbers


# ------------------------------------------------------------------ exact results
def _fft(a, w):
    """DFT of a list over Fr, natural order in and out."""
    n = len(a)
    if n == 1:
        return a
    half = n // 2
    tw, t = [1] * half, 1
    for i in range(half):
        tw[i] = t
        t = t * w % R
    log_n = n.bit_length() - 1
    out = [a[int(format(i, "0%db" % log_n)[::-1], 2)] for i in range(n)]
    h = 1
    while h < n:
        step = half // h
        for s in range(0, n, 2 * h):
            for j in range(h):
                u, v = out[s + j], out[s + j + h] * tw[j * step] % R
                out[s + j], out[s + j + h] = (u + v) % R, (u - v) % R
        h *= 2
    return out


def _f2(a, b):
    return (a[0] * b[0] - a[1] * b[1]) % Q, (a[0] * b[1] + a[1] * b[0]) % Q


class _Fq:
    mul = staticmethod(lambda a, b: a * b % Q)
    sub = staticmethod(lambda a, b: (a - b) % Q)
    inv = staticmethod(lambda a: pow(a, -1, Q))
    words = staticmethod(lambda a: [a])


class _Fq2:
    mul = staticmethod(_f2)
    sub = staticmethod(lambda a, b: ((a[0] - b[0]) % Q, (a[1] - b[1]) % Q))
    words = staticmethod(lambda a: list(a))

    @staticmethod
    def inv(a):
        d = pow(a[0] * a[0] + a[1] * a[1], -1, Q)
        return a[0] * d % Q, -a[1] * d % Q


G1_GEN = (1, 2)
G2_GEN = ((10857046999023057135944570762232829481370756359578518086990519993285655852781,
           11559732032986387107991004021392285783925812861821192530917403151452391805634),
          (8495653923123431417604973247489272438418190587263600148770280649306958101930,
           4082367875863433681332203403145435568316851327593401208105741076214120093531))


def _add(F, p, q):
    if p is None or q is None:
        return p or q
    if p[0] == q[0]:
        if p != q:
            return None
        x2 = F.mul(p[0], p[0])
        zero = F.sub(x2, x2)
        three = F.sub(F.sub(x2, F.sub(zero, x2)), F.sub(zero, x2))
        lam = F.mul(three, F.inv(F.sub(p[1], F.sub(zero, p[1]))))
    else:
        lam = F.mul(F.sub(q[1], p[1]), F.inv(F.sub(q[0], p[0])))
    x = F.sub(F.sub(F.mul(lam, lam), p[0]), q[0])
    return x, F.sub(F.mul(lam, F.sub(p[0], x)), p[1])


def _times(F, p, k):
    acc = None
    for b in bin(k % R)[2:]:
        acc = _add(F, acc, acc)
        if b == "1":
            acc = _add(F, acc, p)
    return acc


def _affine_words(F, p, g2=False):
    """The front end's affine layout: Montgomery words, all zero at infinity."""
    if p is None:
        return np.zeros(16 if g2 else 8, dtype=np.uint64)
    return words([c * MONT % Q for v in p for c in F.words(v)]).reshape(-1)


def exact(case, seed):
    unmont = pow(MONT, -1, R)
    if case["kind"] == "ntt":
        n = 1 << case["log_n"]
        if n * case["batch"] > 1 << 18:
            return None
        inv, coset = "inverse" in case["op"], case["op"].startswith("coset")
        w = pow(5, (R - 1) >> case["log_n"], R)
        a, out = ints(ntt_inputs(case, seed)), []
        for b in range(case["batch"]):
            x = a[b * n:(b + 1) * n]
            if coset and not inv:
                t = 1
                for i in range(n):
                    x[i], t = x[i] * t % R, t * COSET % R
            x = _fft(x, pow(w, -1, R) if inv else w)
            if inv:
                t, g = pow(n, -1, R), pow(COSET, -1, R) if coset else 1
                for i in range(n):
                    x[i], t = x[i] * t % R, t * g % R
            out += x
        return words(out).view(np.int64)
    if case["kind"] == "msm":
        k, s = msm_inputs(case, seed)
        t = sum(a * b for a, b in zip(ints(k), ints(s))) * unmont * unmont % R
        F, g = (_Fq2, G2_GEN) if case["g2"] else (_Fq, G1_GEN)
        return _affine_words(F, _times(F, g, t), case["g2"])
    if case["kind"] == "kzg":
        tau, f, z = kzg_inputs(case, seed)
        f, z = ints(f), ints(z)[0] * unmont % R
        ft = fz = 0
        for c in reversed(f):  # Montgomery words: a common factor 2^256
            ft, fz = (ft * tau + c) % R, (fz * z + c) % R
        q = (ft - fz) * pow(tau - z, -1, R) * unmont % R
        return _affine_words(_Fq, _times(_Fq, G1_GEN, q)), words([fz])[0]
    return None
