"""The blocked factorization with its window in global memory, at the edges of
its range and of its 16-row tiles, 32-row panels and 64-row loads: factors of
both directions against the oracle's.  The tolerance is that of the other wide
bands (rounding of the update chains, relative to the largest factor entry)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# n, k, P: FP64 takes 113 .. 224 here, FP32 225 .. 480.  Partition lengths end
# in panels of 1, 15, 17 and 32 rows; one is shorter than the window.
FP64 = [(1539, 113, 3), (1185, 128, 3), (1230, 129, 3), (2000, 160, 4), (1373, 209, 3), (929, 224, 2), (1030, 150, 1)]
FP32 = [(1539, 225, 3), (1185, 272, 2), (1313, 273, 2), (2001, 401, 2), (1473, 480, 2), (600, 300, 1)]


@pytest.mark.parametrize("case,double", [(c, True) for c in FP64] + [(c, False) for c in FP32])
@pytest.mark.parametrize("fact", ["LU_UL", "LU_only"])
def test_factors_match_oracle(case, double, fact):
    import saplibrary_amd as sap
    from oracle import pyoracle as oracle
    n, k, P = case
    band = oracle.gen_banded(n, k, 0.8, 25)
    cpu = oracle.Solver(P, fact=fact, precond="Block", prec_double=double)
    assert cpu.setup(band) == 0
    g = sap.Solver(P, sap.Options(factMethod=sap.LU_UL if fact == "LU_UL" else sap.LU_only, precondType=sap.Block,
                                  precValueType=sap.PREC_DOUBLE if double else sap.PREC_FLOAT))
    g.setup(sap.BandedMatrix(torch.from_numpy(band).cuda()))
    assert g.numPartitions == cpu.num_partitions
    Fg, Fc = g.factors(), cpu.factors()
    np.testing.assert_allclose(Fg, Fc, rtol=0, atol=(1e-10 if double else 2e-4) * np.abs(Fc).max())


def test_two_threads_factor_different_widths():
    """Setups of two widths at the same time: the kernel's LDS limit, one per
    process, must never fall below what the other thread's launch needs."""
    import threading
    import saplibrary_amd as sap
    from oracle import pyoracle as oracle
    opts = dict(factMethod=sap.LU_only, precondType=sap.Block, precValueType=sap.PREC_DOUBLE)
    bands = [oracle.gen_banded(700, k, 0.8, 26) for k in (113, 224)]
    one = []
    for b in bands:
        g = sap.Solver(1, sap.Options(**opts))
        g.setup(sap.BandedMatrix(torch.from_numpy(b).cuda()))
        one.append(g.factors())
    errors = []

    def work(b, ref):
        try:
            st = torch.cuda.Stream()
            with torch.cuda.stream(st):
                A = sap.BandedMatrix(torch.from_numpy(b).cuda())
                g = sap.Solver(1, sap.Options(**opts))
                for _ in range(150):
                    g.setup(A)
                assert np.array_equal(g.factors(), ref)
        except Exception as e:   # (reported by the main thread)
            errors.append(e)
    threads = [threading.Thread(target=work, args=x) for x in zip(bands, one)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
