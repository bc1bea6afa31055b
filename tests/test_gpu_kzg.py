"""GPU tests of the KZG commitment and opening (cuda-zkml_amd/csrc/kzg.hip;
zk_kzg_commit / zk_kzg_open, reference KZGCommitment, src/prover/groth16.cu:
393-438).

Pins (closed forms over an SRS built from a known tau, [tau^i]_1 = tau^i G1):
  commit  = f(tau) G1;
  open    = q(tau) G1 with q(tau) = (f(tau) - f(z)) / (tau - z), and the
            returned f(z) equals Horner's f(z) in Python;
  the pairing equation e(C - f(z) G1, G2) = e(proof, [tau]_2 - z G2) holds
  (host pairing), and fails for a wrong f(z);
  degrees 0 and 1 give the identity proof (the reference's rule); the sizes
  cross the edges of the blocked scan's threads (4 values), blocks (1024) and
  levels (2^20).
The expected points come from the oracle's CPU fixed-base multiply.
"""
import random

import numpy as np
import pytest

import zkml_amd
from bindings import oracle, ptr
from zkpy import G1, G2, MONT, P as Q, R, g1, g2

pytestmark = pytest.mark.gpu


def mont_words(vals):
    return np.array([[(v * MONT % R) >> (64 * k) & ((1 << 64) - 1) for k in range(4)] for v in vals],
                    dtype=np.uint64).reshape(-1, 4)


def gen_points(scalars):
    """k G1 for each k (oracle, CPU), (n, 8) Montgomery affine words."""
    k = mont_words(scalars)
    out = np.zeros((len(scalars), 8), dtype=np.uint64)
    oracle().orc_g1_gen_batch(ptr(k), len(scalars), ptr(out), 8)
    return out


def horner(coeffs, x):
    acc = 0
    for c in reversed(coeffs):
        acc = (acc * x + c) % R
    return acc


@pytest.fixture(scope="module")
def ctx():
    return zkml_amd.Context(0)


SIZES = [0, 1, 2, 3, 31, 32, 33, 1024, 1025, 1057, 40000]


@pytest.fixture(scope="module")
def srs():
    rng = random.Random(77)
    tau = rng.randrange(2, R)
    n = max(SIZES)
    return tau, gen_points([pow(tau, i, R) for i in range(n)])


@pytest.mark.parametrize("degree", SIZES)
def test_commit_and_open_closed_forms(ctx, srs, degree):
    tau, pts = srs
    rng = random.Random(degree)
    f = [rng.randrange(R) for _ in range(degree)]
    z = rng.randrange(R)
    print(f"[kzg] degree {degree}", flush=True)
    d_srs = ctx.upload(pts[:max(degree, 1)])
    d_f = ctx.upload(mont_words(f) if degree else np.zeros((1, 4), dtype=np.uint64))
    com = ctx.kzg_commit(d_srs, d_f, degree)
    proof, fz = ctx.kzg_open(d_srs, d_f, degree, mont_words([z])[0])
    ft, fzv = horner(f, tau), horner(f, z)
    assert zkml_amd.words_int(fz) * pow(MONT, -1, R) % R == fzv
    expect_c = gen_points([ft])[0] if ft else np.zeros(8, dtype=np.uint64)
    assert np.array_equal(com, expect_c)
    if degree <= 1:
        assert not proof.any()
        return
    qt = (ft - fzv) * pow((tau - z) % R, -1, R) % R
    expect_p = gen_points([qt])[0] if qt else np.zeros(8, dtype=np.uint64)
    assert np.array_equal(proof, expect_p)


def _std_point_g1(pt):
    return np.array([v for c in pt for v in zkml_amd.std_words(c)], dtype=np.uint64)


def _std_point_g2(pt):
    return np.array([v for c2 in pt for c in c2 for v in zkml_amd.std_words(c)], dtype=np.uint64)


def test_pairing_equation(ctx, srs):
    tau, pts = srs
    rng = random.Random(5)
    degree = 200
    f = [rng.randrange(R) for _ in range(degree)]
    z = rng.randrange(R)
    d_srs = ctx.upload(pts[:degree])
    d_f = ctx.upload(mont_words(f))
    com = ctx.kzg_commit(d_srs, d_f, degree)
    proof, fz = ctx.kzg_open(d_srs, d_f, degree, mont_words([z])[0])
    fzv = zkml_amd.words_int(fz) * pow(MONT, -1, R) % R

    def affine(w):  # Montgomery Fq words -> Python ints
        x = zkml_amd.words_int(w[:4]) * pow(MONT, -1, Q) % Q
        y = zkml_amd.words_int(w[4:]) * pow(MONT, -1, Q) % Q
        return (x, y)

    C, Pi = affine(com), affine(proof)
    lhs_pt = g1.padd(C, g1.pneg(g1.pmul(G1, fzv)))
    rhs_q = g2.padd(g2.pmul(G2, tau), g2.pneg(g2.pmul(G2, z)))
    lhs = zkml_amd.pairing(_std_point_g1(lhs_pt), _std_point_g2(G2))
    rhs = zkml_amd.pairing(_std_point_g1(Pi), _std_point_g2(rhs_q))
    assert np.array_equal(lhs, rhs)
    wrong = g1.padd(C, g1.pneg(g1.pmul(G1, (fzv + 1) % R)))
    assert not np.array_equal(zkml_amd.pairing(_std_point_g1(wrong), _std_point_g2(G2)), rhs)


@pytest.mark.parametrize("degree", [4, 5, 6, 1023, 1026, 2049, 4098, 1048577, 1049603])
def test_open_division_blocks(ctx, degree):
    """The division scans blocks of 1024 quotient coefficients, four per thread,
    and the blocks' values the same way: ragged ends of a thread, of a block and
    of the second level (from 2^20 + 1 coefficients on a third one)."""
    rng = np.random.default_rng(degree)
    tau, z = (int(rng.integers(1 << 62)) ** 4 % R for _ in range(2))
    powers, p = [], MONT % R
    for _ in range(degree):
        powers.append(p.to_bytes(32, "little"))
        p = p * tau % R
    d_srs = ctx.alloc(degree * 64)
    ctx.g1_generator_mul(ctx.upload(np.frombuffer(b"".join(powers), dtype=np.uint64).reshape(-1, 4)), degree, d_srs)
    words = zkml_amd.random_fr(degree, rng)  # Montgomery words
    raw = [int.from_bytes(w.tobytes(), "little") for w in words]
    print(f"[kzg division] degree {degree}", flush=True)
    proof, fz = ctx.kzg_open(d_srs, ctx.upload(words), degree, mont_words([z])[0])
    ft, fzv = horner(raw, tau), horner(raw, z)
    assert zkml_amd.words_int(fz) == fzv
    qt = (ft - fzv) * pow((tau - z) * MONT % R, -1, R) % R
    assert np.array_equal(proof, gen_points([qt])[0])


def _open_raw(ctx, d_srs, coeffs_ptr, degree, z):
    """zk_kzg_open through the C ABI, the coefficients at any address."""
    import ctypes
    out, fz = np.zeros(8, dtype=np.uint64), np.zeros(4, dtype=np.uint64)
    zw = mont_words([z])[0].copy()
    rc = zkml_amd.lib().zk_kzg_open(ctx.h, ctypes.c_void_p(d_srs.ptr), ctypes.c_void_p(coeffs_ptr), degree, ptr(zw),
                                    ptr(out), ptr(fz), None)
    return rc, out, fz


@pytest.mark.parametrize("degree", [2, 33, 1500])
def test_open_takes_coefficients_where_the_copy_did(ctx, srs, degree):
    """Coefficients that the division does not read in place go through the
    runtime's copy: at an address that is a multiple of 8 only, and in host
    memory.  Same proof and value as from a device buffer."""
    _, pts = srs
    rng = random.Random(degree)
    f, z = [rng.randrange(R) for _ in range(degree)], rng.randrange(R)
    d_srs = ctx.upload(pts[:degree])
    words = mont_words(f)
    want, fz = ctx.kzg_open(d_srs, ctx.upload(words), degree, mont_words([z])[0])
    assert zkml_amd.words_int(fz) * pow(MONT, -1, R) % R == horner(f, z)
    shifted = ctx.upload(np.concatenate([np.zeros(1, dtype=np.uint64), words.reshape(-1)]))
    for name, at in (("shifted", shifted.ptr + 8), ("host", words.ctypes.data)):
        print(f"[kzg coefficients] degree {degree} {name}", flush=True)
        rc, out, got_fz = _open_raw(ctx, d_srs, at, degree, z)
        assert rc == 0, name
        assert np.array_equal(out, want) and np.array_equal(got_fz, fz), name


def test_open_refuses_a_coefficient_buffer_shorter_than_the_degree(ctx, srs):
    """A degree beyond the buffer's end is refused (the runtime checks the copy's
    range), not read.  The buffer ends inside a page, so that even an unchecked
    read of one coefficient more would stay in mapped memory."""
    _, pts = srs
    d_srs, d_f = ctx.upload(pts[:128]), ctx.upload(mont_words(list(range(1, 101))))
    rc, _, _ = _open_raw(ctx, d_srs, d_f.ptr, 101, 5)
    assert rc != 0
    rc, _, _ = _open_raw(ctx, d_srs, d_f.ptr, 100, 5)
    assert rc == 0


def test_open_with_z_in_the_result_buffers(ctx, srs):
    """z may share its words with the proof or with f(z): it is read before
    they are written."""
    import ctypes
    _, pts = srs
    rng = random.Random(9)
    degree = 300
    f, z = [rng.randrange(R) for _ in range(degree)], rng.randrange(R)
    d_srs, d_f = ctx.upload(pts[:degree]), ctx.upload(mont_words(f))
    want, fz = ctx.kzg_open(d_srs, d_f, degree, mont_words([z])[0])
    for shared in ("proof", "value"):
        out, got = np.zeros(8, dtype=np.uint64), np.zeros(4, dtype=np.uint64)
        zw = out[2:6] if shared == "proof" else got
        zw[:] = mont_words([z])[0]
        rc = zkml_amd.lib().zk_kzg_open(ctx.h, ctypes.c_void_p(d_srs.ptr), ctypes.c_void_p(d_f.ptr), degree, ptr(zw),
                                        ptr(out), ptr(got), None)
        assert rc == 0
        assert np.array_equal(out, want) and np.array_equal(got, fz), shared
