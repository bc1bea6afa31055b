"""Error paths of the NTT's cached tables: a device allocation that fails
while a transform builds its plan or its coset tables returns ZK_ERR_OOM,
caches nothing half-built, and the same context's next transforms (same size,
same coset) are bit-exact against the CPU oracle.  The failures are injected
with the library's zk_debug_fail_device_alloc hook; no device memory is
exhausted.  (The reference has no such path: it exits on any CUDA error,
src/common.cuh:11-19.)"""
import numpy as np
import pytest

from test_gpu_ntt import oracle_coset, oracle_ntt, rand_words

pytestmark = pytest.mark.gpu


def _fail_at(nth):
    import zkml_amd
    assert zkml_amd.lib().zk_debug_fail_device_alloc(nth) == 0


@pytest.mark.parametrize("log_n", [11, 17])
def test_table_allocation_failure_then_recovery(log_n):
    import zkml_amd
    ctx = zkml_amd.Context(0)  # fresh: no plan, coset table or pass buffer yet
    try:
        a = rand_words(1 << log_n, 100 + log_n)
        d_in = ctx.upload(a)
        d_out = ctx.alloc(a.nbytes)
        # A first coset transform allocates the plan's tables, then the coset
        # tables, then the pass-to-pass buffer.  Fail each in turn: the plan
        # (1st), the coset tables (2nd, after the plan is cached), the pass
        # buffer (2nd again, after the coset tables are cached).
        for nth in (1, 2, 2):
            _fail_at(nth)
            with pytest.raises(zkml_amd.ZkError, match="ZK_ERR_OOM|out of memory|allocation"):
                ctx.coset_ntt(d_out, d_in, log_n, 7, False)
            _fail_at(0)
        ctx.coset_ntt(d_out, d_in, log_n, 7, False)
        assert np.array_equal(ctx.d2h(d_out, a.shape), oracle_coset(a, log_n, 7, False))
        # plan cached, a new coset generator needs new tables: fail them once
        _fail_at(1)
        with pytest.raises(zkml_amd.ZkError):
            ctx.coset_ntt(d_out, d_in, log_n, 5, True)
        _fail_at(0)
        ctx.coset_ntt(d_out, d_in, log_n, 5, True)
        assert np.array_equal(ctx.d2h(d_out, a.shape), oracle_coset(a, log_n, 5, True))
        ctx.ntt(d_out, d_in, log_n, False)
        assert np.array_equal(ctx.d2h(d_out, a.shape), oracle_ntt(a, log_n, False))
    finally:
        _fail_at(0)
        ctx.close()


def _free_bytes():
    import ctypes
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_pk_window_table_allocation_failure_falls_back(tmp_path):
    """zk_pk_load of a key with 2^15 variables builds window tables for its
    queries (each table, then its temporary, in the order A, B1, L, B2, H).
    A failed allocation of a table or of its temporary drops every table: the
    load still succeeds, leaves no error behind and holds a fraction of the
    tables' memory, and the next proof is byte-identical to a table-backed
    proof and to the oracle's prove on the same key and seed."""
    import zkml_amd
    from test_gpu_groth16 import PROVE_SEED, SETUP_SEED, _oracle_of
    ctx = zkml_amd.Context(0)
    try:
        nc, npub = (1 << 15) - 64, 4
        A, B, C, w = zkml_amd.synthetic_r1cs(nc, npub, 16, 15)
        r = ctx.r1cs(nc, w.shape[0], npub, A, B, C)
        pk_path, vk_path = str(tmp_path / "pk.bin"), str(tmp_path / "vk.bin")
        ctx.setup(r, SETUP_SEED, pk_path, vk_path)
        ctx.sync()
        before = _free_bytes()
        pk = ctx.load_pk(pk_path)
        with_tables = before - _free_bytes()
        proof, _ = ctx.prove(pk, r, w, npub, PROVE_SEED)
        pk.close()
        # 1: A's table, 2: A's temporary, 7: B2's table, 10: H's temporary
        for nth in (1, 2, 7, 10):
            print(f"[pk tables] allocation {nth} fails", flush=True)
            ctx.sync()
            before = _free_bytes()
            _fail_at(nth)
            try:
                pk = ctx.load_pk(pk_path)
            finally:
                _fail_at(0)
            used = before - _free_bytes()
            assert used < with_tables // 2, (nth, used, with_tables)
            assert zkml_amd.lib().zk_last_error(ctx.h) in (None, b"")
            again, _ = ctx.prove(pk, r, w, npub, PROVE_SEED)
            assert again == proof, nth
            pk.close()
        oc = _oracle_of(A, B, C, nc, w.shape[0], npub)
        rc, proof_o, _ = oc.prove(pk_path, w, PROVE_SEED, threads=16)
        assert rc == 0 and proof_o == proof
        r.close()
    finally:
        _fail_at(0)
        ctx.close()


@pytest.mark.parametrize("g2,n", [(False, 1000), (False, 40000), (False, 300007), (True, 9000), (True, 70001)])
def test_msm_allocates_only_on_the_first_call_of_a_size(g2, n):
    """After one MSM of a size, other scalars of that size need no device
    memory: the workspaces follow the size, not the scalars' digit counts.  No
    entries at all first, then a few, then witness-like, uniform and equal
    scalars (one hot bucket in every window), each with the next allocation
    armed to fail, against the closed form."""
    import zkml_amd
    import zkpy as Z
    from test_gpu_msm import closed_form_scalar, gpu_points, rand_std, to_mont, witness_like
    ctx = zkml_amd.Context(0)
    try:
        rng = np.random.default_rng(n + g2)
        kstd = rand_std(n, rng)
        dp = gpu_points(ctx, to_mont(kstd), g2=g2)
        run = ctx.msm_g2 if g2 else ctx.msm_g1
        G, gen, from_words = (Z.g2, Z.G2, Z.g2_from_words) if g2 else (Z.g1, Z.G1, Z.g1_from_words)
        none = np.zeros((n, 4), dtype=np.uint64)
        few = none.copy()
        few[:: max(1, n // 50)] = rand_std(len(few[:: max(1, n // 50)]), rng)
        equal = np.repeat(rand_std(1, rng), n, axis=0)
        assert not run(dp, ctx.upload(to_mont(none)), n).any()
        for name, s in (("few", few), ("witness", witness_like(n, rng)), ("uniform", rand_std(n, rng)),
                        ("equal", equal)):
            print(f"[msm allocations {'g2' if g2 else 'g1'} {n}] {name}", flush=True)
            ds = ctx.upload(to_mont(s))
            _fail_at(1)
            got = run(dp, ds, n)
            _fail_at(0)
            assert from_words(got) == G.pmul(gen, closed_form_scalar(kstd, s)), name
    finally:
        _fail_at(0)
        ctx.close()


@pytest.mark.parametrize("rows", [5000, 20000])
def test_proofs_of_one_circuit_allocate_only_once(rows, tmp_path):
    """Proofs of one circuit (x_i^2 = y_i) with other witnesses than the first
    proof's (few entries, small values, uniform values) need no device memory
    of their own, plain MSMs (5000 rows) and window tables (20,000): each with
    the next allocation armed to fail gives the proof of a fresh context."""
    import zkml_amd
    import zkpy as Z
    from r1cs_gen import Circuit
    from test_gpu_groth16 import PROVE_SEED, SETUP_SEED
    rng = np.random.default_rng(rows)
    nv = 1 + 2 * rows  # 1, then x_i, then y_i
    xs = [(i, 1 + i, 1) for i in range(rows)]
    circ = Circuit(rows, nv, 1, nv - 2, xs, xs, [(i, 1 + rows + i, 1) for i in range(rows)], None)
    mats = circ.mats()

    def witness(kind):
        x = [0] * rows
        for i in range(0, rows, 100 if kind == "few" else 1):
            x[i] = int(rng.integers(1, 1 << 15)) if kind == "small" else int(rng.integers(1, 1 << 62)) ** 5 % Z.R
        circ.w = [1] + x + [v * v % Z.R for v in x]
        return circ.witness_words()

    pk_path, vk_path = str(tmp_path / "pk.bin"), str(tmp_path / "vk.bin")
    proofs, ws = {}, {k: witness(k) for k in ("few", "small", "uniform")}
    for fresh in (False, True):
        for kind in (("few", "small", "uniform") if not fresh else ("small", "uniform")):
            if fresh or kind == "few":
                ctx = zkml_amd.Context(0)
                r = ctx.r1cs(rows, nv, 1, *mats)
                if not proofs:
                    ctx.setup(r, SETUP_SEED, pk_path, vk_path)
                pk = ctx.load_pk(pk_path)
            print(f"[proof allocations] {rows} rows, {kind}, {'fresh context' if fresh else 'kept context'}",
                  flush=True)
            try:
                _fail_at(0 if fresh or kind == "few" else 1)
                proof, _ = ctx.prove(pk, r, ws[kind], 1, PROVE_SEED)
            finally:
                _fail_at(0)
            if not fresh:
                proofs[kind] = proof
            else:
                assert proof == proofs[kind], kind
            if fresh or kind == "uniform":
                pk.close()
                r.close()
                ctx.close()
    assert len(set(proofs.values())) == 3
