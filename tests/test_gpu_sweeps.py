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
block only while no entry of it passes 8 and substitute otherwise.  On bands
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


def host_apply(F, v):
    """M^{-1} v of one partition in FP64 from its factor band (row c: column c,
    entry (r, c) at k + r - c): L, D, U'."""
    n, k = len(F), F.shape[1] // 2
    x = v.astype(np.float64)
    for c in range(n):
        m = min(k, n - 1 - c)
        x[c + 1:c + 1 + m] -= F[c, k + 1:k + 1 + m] * x[c]
    x /= F[:, k]
    for c in range(n - 1, -1, -1):
        m = min(k, c)
        x[c - m:c] -= F[c, k - m:k] * x[c]
    return x


def host_inverse_max(F, bs):
    """Largest entry of the inverse of each unit-lower diagonal block of bs rows."""
    k = F.shape[1] // 2
    out = []
    for c0 in range(0, len(F) - bs + 1, bs):
        L = np.eye(bs)
        for j in range(bs):
            m = min(k, bs - 1 - j)
            L[j + 1:j + 1 + m, j] = F[c0 + j, k + 1:k + 1 + m]
        out.append(np.abs(np.linalg.inv(L)).max())
    return np.array(out)


@pytest.mark.parametrize("n,k,d", [(1200, 20, 0.1), (1203, 33, 0.1), (1500, 50, 0.1), (1600, 90, 0.05),
                                   (1601, 150, 0.05), (1500, 300, 0.02)])
@pytest.mark.parametrize("prec_double", [True, False])
def test_substitution_against_the_factors(sap, oracle, n, k, d, prec_double):
    """The substituting blocks in both precisions, against the same factors
    applied in FP64 on the host: the sweeps' own error alone.  Substitution
    keeps |L D U' z - v| within about 2 k eps of |L| |D| |U'| |z| (a sum of k
    products a row in either solve); the blocks that are multiplied may add
    what their inverses' entries (up to 8) allow, so 8 k eps."""
    print(f"[sweeps] factors n={n} k={k} d={d} fp64={prec_double}", flush=True)
    band = oracle.gen_banded(n, k, d, 740 + k)
    v = oracle.gen_vector(n, 741)
    g = sap.Solver(1, sap.Options(precondType=sap.Block, factMethod=sap.LU_only, safeFactorization=1,
                                  precValueType=sap.PREC_DOUBLE if prec_double else sap.PREC_FLOAT))
    g.setup(sap.BandedMatrix(dev(band)))
    z = torch.empty(n, dtype=torch.float64, device="cuda")
    g.precond_apply(dev(v), z)
    z = z.cpu().numpy()
    F = g.factors()
    grown = host_inverse_max(F, 16 if prec_double else 32)
    assert (grown > 16).sum() >= 2, grown          # the branch is reached
    # w = L D U' z through the factors, row sums of |L| |D| |U'| |z| beside it
    def times(F, x, ab=lambda t: t):
        y = ab(x).copy()
        for c in range(n):                         # U' (unit upper)
            m = min(k, c)
            y[c - m:c] += ab(F[c, k - m:k]) * ab(x)[c]
        y = y * ab(F[:, k])
        w = y.copy()
        for c in range(n):                         # L (unit lower)
            m = min(k, n - 1 - c)
            w[c + 1:c + 1 + m] += ab(F[c, k + 1:k + 1 + m]) * y[c]
        return w
    vt = v if prec_double else v.astype(np.float32).astype(np.float64)
    eps = 2.0 ** -53 if prec_double else 2.0 ** -24
    res = np.abs(times(F, z) - vt).max()
    bound = times(F, z, np.abs).max()
    print(f"[sweeps] backward error {res / bound / eps:.1f} eps, blocks grown {int((grown > 16).sum())}", flush=True)
    assert res <= 8 * k * eps * bound
    # and the value itself: n eps by the four decades these factors amplify
    ref = host_apply(F, vt)
    assert np.isfinite(z).all() and np.linalg.norm(z - ref) <= 1e-2 * np.linalg.norm(ref)


@pytest.mark.parametrize("k", [70, 96, 200])
def test_substitution_in_the_spike_passes(sap, oracle, k):
    """LU and UL factors of every partition, full sweeps in halves and interface
    sweeps (k >= 70: every pivot boosted) with blocks that grow: the same
    operator as with the plain sweeps (no memory for the tables).  FP64: 1e-8,
    n eps by four to five decades that these factors amplify.  FP32: what FP64
    shows, scaled by the two eps, by 16 for the difference between the two
    precisions' factors."""
    import os
    n, P, d = 8 * k + 37, 3, 0.03
    print(f"[sweeps] spike k={k}", flush=True)
    band, v = oracle.gen_banded(n, k, d, 760 + k), oracle.gen_vector(n, 761)

    def difference(prec):
        opts = dict(precondType=sap.Spike, factMethod=sap.LU_UL, safeFactorization=1, precValueType=prec)
        z = apply(sap, band, v, P, **opts)
        os.environ["SAP_AMD_DEVICE_FREE"] = "4"
        try:
            plain = apply(sap, band, v, P, **opts)
        finally:
            del os.environ["SAP_AMD_DEVICE_FREE"]
        assert np.isfinite(z).all()
        return np.linalg.norm(z - plain) / np.linalg.norm(plain)
    d64, d32 = difference(sap.PREC_DOUBLE), difference(sap.PREC_FLOAT)
    print(f"[sweeps] staged against plain {d64:.2e} {d32:.2e}", flush=True)
    assert 0 < d64 <= 1e-8 and 0 < d32 <= 16 * 2.0 ** 29 * d64


def test_substitution_costs_little_more(sap):
    """A band whose blocks mostly grow may not sweep several times slower than
    one of the same size without growth (the chain of substitutions is 31 steps
    of a register broadcast and a multiply-add)."""
    def us(d):
        n, k, P = 100000, 20, 16
        g = sap.Solver(P, sap.Options(precondType=sap.Block, safeFactorization=1))
        g.setup(sap.BandedMatrix.generate(n, k, d, 7))
        v = torch.ones(n, dtype=torch.float64, device="cuda")
        z = torch.empty_like(v)
        best = 1e9
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                g.precond_apply(v, z)
            b.record()
            torch.cuda.synchronize()
            best = min(best, a.elapsed_time(b) / 5 * 1e3)
        return best
    grown, plain = us(0.1), us(1.2)
    print(f"[sweeps] {grown:.0f} us with growth, {plain:.0f} without", flush=True)
    assert grown <= 3 * plain


@pytest.mark.parametrize("prec_double,a", [(False, 1.078125), (False, 1.0859375), (True, 1.15625 + 2 ** -20), (True, 1.1875 + 2 ** -20)])
def test_inverses_above_the_limit_are_not_multiplied(sap, prec_double, a):
    """A lower bidiagonal matrix (1 and a) is its own L, and the inverse of a
    block holds the powers of a: 10.3 and 12.9 at most in FP32's blocks of 32
    rows, 8.8 and 13.2 in FP64's of 16.  With x = 1 in every block's first two
    rows and 0 elsewhere, substitution gives x back exactly (each step is exact
    or 0 - 0); the product with the inverse rounds a^i - (a + 1) a^(i - 1) +
    a a^(i - 2)."""
    bs = 16 if prec_double else 32
    n = 8 * bs + 5
    band = np.zeros((n, 3))
    band[:, 1] = 1.0
    band[1:, 0] = a
    x = np.zeros(n)
    x[::bs] = x[1::bs] = 1.0
    v = x.copy()
    v[1:] += a * x[:-1]
    z = apply(sap, band, v, 1, precondType=sap.Block, factMethod=sap.LU_only,
              precValueType=sap.PREC_DOUBLE if prec_double else sap.PREC_FLOAT)
    assert np.array_equal(z, x)
