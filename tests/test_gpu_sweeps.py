"""The staged triangular sweeps (block-diagonal application, one sweep pass)
at the sizes where they can go wrong, against the CPU oracle's Block
preconditioner: widths around the blocks of 32 (FP32) / 16 (FP64) columns,
around the first far row (k = BS + 1), each wavefront's last far row (64 rows
a group), two rows per lane (k > 192 + BS) and the widest staged band;
partitions whose last block is partial, full, a single row, and shorter than
the pipeline is deep.

Tolerances: the operator's own error, n eps |M^-1| |L| |D| |U'| |z|, is below
100 eps for these rows (diagonal 1.2 times the off-diagonal abs-sum), and both
sides carry it: 1e-13 (FP64) and 3e-5 (FP32) of max |z|.

Factors with growth: the sweeps multiply with the inverse of each diagonal
block only while no entry of it passes 16 and substitute otherwise.  On bands
with a diagonal far below the off-diagonal sums (no pivoting, so the factors
grow) the application is compared through its normwise backward error
|A z - v| / (|A| |z|), which an LU solve without pivoting keeps within about
n eps times the growth of the factors; 1e-10 leaves 4 decades of growth.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def sap():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import saplibrary_amd
    saplibrary_amd.lib()
    return saplibrary_amd


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).cuda()


def apply(sap, band, v, P, **opts):
    g = sap.Solver(P, sap.Options(**opts))
    g.setup(sap.BandedMatrix(dev(band)))
    z = torch.empty(len(v), dtype=torch.float64, device="cuda")
    g.precond_apply(dev(v), z)
    torch.cuda.synchronize()
    return z.cpu().numpy()


SIZES = [
    # n, k, P
    (997, 1, 3), (1024, 2, 4), (500, 15, 3), (640, 16, 5), (771, 17, 2), (999, 31, 3), (1024, 32, 4), (1111, 33, 3),
    (1300, 47, 3), (1500, 48, 3), (1601, 63, 3), (1602, 64, 3), (1603, 65, 2), (1700, 80, 4), (2000, 95, 3),
    (2001, 96, 3), (1930, 97, 3), (1923, 128, 3), (2100, 129, 3), (3000, 160, 3), (2500, 207, 2), (2700, 208, 2),
    (2701, 209, 2), (2900, 223, 2), (3000, 224, 2), (3001, 225, 2), (2050, 256, 2), (3300, 300, 2), (2600, 384, 2),
    (2001, 400, 1), (1700, 416, 1), (33, 5, 1), (65, 8, 1), (31, 3, 1),
]


@pytest.mark.parametrize("n,k,P", SIZES)
@pytest.mark.parametrize("prec_double", [True, False])
def test_staged_sweeps_match_oracle(sap, oracle, n, k, P, prec_double):
    print(f"[sweeps] n={n} k={k} P={P} fp64={prec_double}", flush=True)
    band = oracle.gen_banded(n, k, 1.2, 700 + k)
    v = oracle.gen_vector(n, 701)
    z = apply(sap, band, v, P, precondType=sap.Block,
              precValueType=sap.PREC_DOUBLE if prec_double else sap.PREC_FLOAT)
    cpu = oracle.Solver(P, fact="LU_only", precond="Block", prec_double=prec_double)
    assert cpu.setup(band) == 0
    ref = cpu.apply(v)
    np.testing.assert_allclose(z, ref, rtol=0, atol=(1e-13 if prec_double else 3e-5) * np.abs(ref).max())


@pytest.mark.parametrize("n,k,d", [(3000, 20, 0.2), (3000, 20, 0.1), (2500, 50, 0.1), (2600, 90, 0.05)])
def test_blocks_that_grow_are_substituted(sap, oracle, n, k, d):
    print(f"[sweeps] growth n={n} k={k} d={d}", flush=True)
    band = oracle.gen_banded(n, k, d, 720 + k)
    v = oracle.gen_vector(n, 721)
    z = apply(sap, band, v, 1, precondType=sap.Block, precValueType=sap.PREC_DOUBLE, safeFactorization=1)
    res = oracle.band_spmv(band, z) - v
    norm = np.abs(band).sum(axis=1).max()
    assert np.isfinite(z).all()
    assert np.abs(res).max() <= 1e-10 * norm * np.abs(z).max()
