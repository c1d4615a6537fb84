"""What a full device does: the library's buffers are bounded from the host with
SAP_AMD_DEVICE_LIMIT (bytes), past which an allocation fails through the
runtime as the device's own memory would.

  * The sweeps' tables are optional (they only make the sweeps faster): a
    setup without room for them succeeds, with the plain sweeps, and gives the
    same preconditioner.
  * They give way to what cannot be done without: the SaP-C buffers and work
    space of the same setup, a solve's vectors, the next setup's larger band.
  * They take at most a quarter of the memory that is free (what that is taken
    to be is set with SAP_AMD_DEVICE_FREE), so that what another solver or the
    program allocates next fits as it does beside a solver without tables.

Tolerances: both sweep variants carry the operator's own rounding, as in the
staged sweeps' and the application tests: 1e-13 (block-diagonal) and 1e-10
(truncated SPIKE, block cyclic reduction) of max |z| in FP64, 3e-5 in FP32.
"""
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

MIB = 1 << 20


@pytest.fixture(scope="module")
def sap():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import saplibrary_amd
    saplibrary_amd.lib()
    return saplibrary_amd


@pytest.fixture
def limit(monkeypatch):
    """limit(bytes) bounds the library's buffers, limit(None) lifts the bound."""
    gc.collect()

    def set_to(b):
        if b is None:
            monkeypatch.delenv("SAP_AMD_DEVICE_LIMIT", raising=False)
        else:
            monkeypatch.setenv("SAP_AMD_DEVICE_LIMIT", str(int(b)))
    return set_to


def apply(g, v):
    z = torch.empty_like(v)
    g.precond_apply(v, z)
    torch.cuda.synchronize()
    return z.cpu().numpy()


# A row's tables take 264 (FP32) or 272 (FP64) bytes a direction.
@pytest.mark.parametrize("prec_double", [False, True])
@pytest.mark.parametrize("kind", ["block", "spike", "bcr"])
def test_without_room_for_the_tables(sap, oracle, limit, kind, prec_double):
    n, k, P = 60000, 20, 8
    print(f"[memory] {kind} fp64={prec_double}", flush=True)
    band, v = oracle.gen_banded(n, k, 1.2, 81), torch.from_numpy(oracle.gen_vector(n, 82)).cuda()
    A = sap.BandedMatrix(torch.from_numpy(band).cuda())
    opts = sap.Options(precondType=sap.Spike if kind == "spike" else sap.Block, factMethod=sap.LU_UL,
                       useBCR=1 if kind == "bcr" else 0, trackReordering=1,
                       precValueType=sap.PREC_DOUBLE if prec_double else sap.PREC_FLOAT)
    sz = 8 if prec_double else 4
    bands = (3 if kind == "spike" else 1) * n * (2 * k + 1) * sz
    blocks = 4 * (n // (2 * k) + P) * k * k * sz if kind == "bcr" else 0
    cap = bands + blocks + 40 * n + (30 if kind == "bcr" else 20) * MIB   # (the tables: 31 MB, bcr 45 MB and more)
    limit(cap)
    g = sap.Solver(P, opts)
    g.setup(A)
    z = apply(g, v)
    g.update(A.band)   # again without tables
    assert np.array_equal(apply(g, v), z)
    limit(None)
    g.setup(A)         # with tables
    zt = apply(g, v)
    assert not np.array_equal(zt, z)
    cpu = oracle.Solver(P, fact="LU_UL" if kind == "spike" else "LU_only", precond="Spike" if kind == "spike" else "Block",
                        prec_double=prec_double)
    assert cpu.setup(band) == 0
    ref = cpu.apply(v.cpu().numpy())
    tol = 3e-5 if not prec_double else 1e-13 if kind == "block" else 1e-10
    for got in (z, zt):
        np.testing.assert_allclose(got, ref, rtol=0, atol=tol * np.abs(ref).max())


# The tables of n rows (one band, FP32): both directions of 264 bytes a row and
# one padded block per partition.
def tables_bytes(n, P):
    return 2 * (n // 32 + P) * 8448


def spike_options(sap, **kw):
    return sap.Options(precondType=sap.Spike, factMethod=sap.LU_only, trackReordering=1, relTol=1e-10, refine=8, **kw)


# LU_only: the spike tips' work space (n x 32 values) is needed after the tables
def test_tables_give_way_to_the_setup(sap, oracle, limit):
    n, k, P = 60000, 20, 8
    band, v = oracle.gen_banded(n, k, 1.2, 83), torch.from_numpy(oracle.gen_vector(n, 84)).cuda()
    A = sap.BandedMatrix(torch.from_numpy(band).cuda())
    cpu = oracle.Solver(P, fact="LU_only", precond="Spike", prec_double=False)
    assert cpu.setup(band) == 0
    ref = cpu.apply(v.cpu().numpy())
    limit((2 * k + 1) * 4 * n + tables_bytes(n, P) + 40 * n)
    g = sap.Solver(P, spike_options(sap))
    g.setup(A)
    np.testing.assert_allclose(apply(g, v), ref, rtol=0, atol=3e-5 * np.abs(ref).max())
    g.update(A.band)
    np.testing.assert_allclose(apply(g, v), ref, rtol=0, atol=3e-5 * np.abs(ref).max())


def test_tables_give_way_to_the_solve_and_the_next_setup(sap, oracle, limit):
    n, k, P = 60000, 20, 8
    A = sap.BandedMatrix(torch.from_numpy(oracle.gen_banded(n, k, 1.2, 85)).cuda())
    big = sap.BandedMatrix(torch.from_numpy(oracle.gen_banded(3 * n // 2, k, 1.2, 86)).cuda())
    # the band, its vectors and the tables; a solve takes 32 FP64 vectors more
    limit((2 * k + 1) * 4 * n + tables_bytes(n, P) + 40 * n)
    g = sap.Solver(P, sap.Options(precondType=sap.Block, relTol=1e-10, refine=8))
    g.setup(A)
    for M in (A, big):
        if M is big:
            limit((2 * k + 1) * 4 * M.num_rows + (40 + 256) * M.num_rows + MIB)
            g.setup(M)
        x0 = torch.rand(M.num_rows, dtype=torch.float64, device="cuda")
        b = sap.band_spmv(M, x0, torch.empty_like(x0))
        x = torch.zeros_like(b)
        assert g.solve(None, b, x), g.getMonitorMessage()
        r = b - sap.band_spmv(M, x, torch.empty_like(x))
        assert float(r.norm() / b.norm()) <= 1e-10


def test_tables_give_way_to_a_batch(sap, oracle, limit):
    n, k, P, nr = 30000, 20, 8, 1
    mats = [sap.BandedMatrix(torch.from_numpy(oracle.gen_banded(n, k, 1.2, 87 + s)).cuda()) for s in range(3)]
    B = [torch.rand(n, nr, dtype=torch.float64, device="cuda") for _ in mats]

    def run():
        b = sap.SystemBatch([P] * len(mats), sap.Options(precondType=sap.Block, relTol=1e-10, refine=8))
        b.setup(mats)
        X = [torch.zeros_like(c) for c in B]
        assert b.solve(B, X)
        return X
    ref = run()
    gc.collect()
    one = (2 * k + 1) * 4 * n + 40 * n + tables_bytes(n, P)
    for cap in (2 * one + one // 2,                              # the third system's tables do not fit
                3 * one + MIB,                                   # the solve's vectors do not
                3 * (one - tables_bytes(n, P)) + 3 * n * 8 * 24):  # nor does the third system
        limit(cap)
        try:
            X = run()
        finally:
            limit(None)
        gc.collect()
        for x, y in zip(X, ref):
            assert float((x - y).norm() / y.norm()) <= 1e-9


# Variable bandwidth: with less and less memory the setup is truncated SPIKE with
# the tables, then without, and only then anything else.
def test_tables_give_way_to_the_spike_buffers(sap, oracle, limit):
    from tests.csr_cases import sparse_band
    n, P = 6000, 3
    rp, ci, val = sparse_band(n, 90, 8, 57)
    A = sap.CsrMatrix.from_host(rp, ci, val)
    v = torch.from_numpy(oracle.gen_vector(n, 404)).cuda()
    opts = sap.Options(precValueType=sap.PREC_DOUBLE)
    g = sap.Solver(P, opts)
    g.setup(A)
    full = apply(g, v)
    tol = 1e-10 * np.abs(full).max()
    del g
    gc.collect()
    seen = []
    for cap in range(32 * MIB, 0, -MIB // 4):
        limit(cap)
        g = None
        try:
            g = sap.Solver(P, opts)
            g.setup(A)
            z = apply(g, v)
            seen.append("tables" if np.array_equal(z, full) else "spike" if np.abs(z - full).max() <= tol else "other")
        except sap.SapError as e:
            assert "Out_of_memory" in str(e) or g is None, str(e)
            seen.append("oom")
        finally:
            limit(None)
            del g
            gc.collect()
        if seen[-1] == "oom" and len(seen) > 4 and seen[-4:] == ["oom"] * 4:
            break
    print("[memory] " + " ".join(seen), flush=True)
    order = ["tables", "spike"]
    good = [s for s in seen if s in order]
    assert seen[:len(good)] == sorted(good, key=order.index) and "tables" in good and "spike" in good


def test_tables_take_a_quarter_of_the_free_memory(sap, oracle, limit, monkeypatch):
    n, k, P = 60000, 20, 8
    A = sap.BandedMatrix(torch.from_numpy(oracle.gen_banded(n, k, 1.2, 91)).cuda())
    v = torch.from_numpy(oracle.gen_vector(n, 92)).cuda()
    size = 2 * (n // 32 + P) * 2112 * 4   # of the tables: (n / 32 + P) blocks of 2112 values, two directions

    def z_with(free):
        if free:
            monkeypatch.setenv("SAP_AMD_DEVICE_FREE", str(free))
        g = sap.Solver(P, sap.Options(precondType=sap.Block))
        g.setup(A)
        monkeypatch.delenv("SAP_AMD_DEVICE_FREE", raising=False)
        return apply(g, v)
    full = z_with(0)
    limit((2 * k + 1) * 4 * n + 40 * n + 20 * MIB)
    plain = z_with(0)
    limit(None)
    assert not np.array_equal(plain, full)
    assert np.array_equal(z_with(4 * size), full)
    assert np.array_equal(z_with(4 * size - 4), plain)
