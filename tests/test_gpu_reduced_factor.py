"""The reduced blocks' LU and inverse at the widths where the kernels change
(matrix in registers, in LDS, in global memory; inverse by blocked sweeps or
column by column): one truncated-SPIKE application against the oracle's, at
the tolerance of the other application tests."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,double", [(142, True), (143, True), (160, True), (161, True), (256, True), (300, True),
                                      (201, False), (202, False), (224, False), (225, False), (416, False),
                                      (417, False)])
def test_spike_apply_matches_oracle(k, double):
    import saplibrary_amd as sap
    from oracle import pyoracle as oracle
    n, P = 6 * k + 11, 3
    band, v = oracle.gen_banded(n, k, 0.8, 31), oracle.gen_vector(n, 32)
    cpu = oracle.Solver(P, fact="LU_UL", precond="Spike", prec_double=double)
    assert cpu.setup(band) == 0
    g = sap.Solver(P, sap.Options(precondType=sap.Spike,
                                  precValueType=sap.PREC_DOUBLE if double else sap.PREC_FLOAT))
    g.setup(sap.BandedMatrix(torch.from_numpy(band).cuda()))
    assert g.numPartitions == cpu.num_partitions
    z = torch.empty(n, dtype=torch.float64, device="cuda")
    g.precond_apply(torch.from_numpy(v).cuda(), z)
    ref = cpu.apply(v)
    np.testing.assert_allclose(z.cpu().numpy(), ref, rtol=0, atol=(1e-10 if double else 3e-5) * np.abs(ref).max())
