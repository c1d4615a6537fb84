"""What a full device does: the library's buffers are bounded from the host with
SAP_AMD_DEVICE_LIMIT (bytes), past which an allocation fails through the
runtime as the device's own memory would.

  * The sweeps' tables are optional (they only make the sweeps faster): a
    setup without room for them succeeds, with the plain sweeps, and gives the
    same preconditioner.

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
