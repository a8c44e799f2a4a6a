"""V-cycles whose Q_1 levels smooth with the assembled operator, against the FP64
oracle: every parity of the smoother degree (which buffer holds the
iterate, steps sharing a launch), Gauss and Gauss-Lobatto entries, metric
terms stored and on the fly, Q_1 as the fine level and below others, cell counts
that differ per direction, the separate smoothing operator, and transfers of 2
and 3 entries per row.

Tolerance: a V-cycle is a few dozen FP32 applies of operators whose rows cancel to
about 1e-2 of their entries: 6e-8 * 1e2 * a few tens = 1e-4."""
import numpy as np
import pytest

from oracle import mg_oracle as M
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degree", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("p,nq,quad,n,cmax,geometry,sq",
                         [(1, 2, O.GLL, (8, 12, 4), 20, 1, 0), (1, 3, O.GAUSS, (12, 4, 8), 20, 0, 0),
                          (2, 3, O.GAUSS, (8, 4, 12), 20, 1, 0), (3, 4, O.GLL, (4, 8, 4), 20, 0, 0),
                          (1, 3, O.GAUSS, (16, 8, 8), 20, 1, 2)])
def test_vcycle_matches_oracle(gpu, degree, p, nq, quad, n, cmax, geometry, sq):
    import torch
    from benchmarks_amd.laplace import PreconditionMG
    mg = PreconditionMG(p, nq, quad, n, deform=0.05, geometry=geometry, coarse_max_dofs=cmax,
                        smoother_degree=degree, fine_smoother_n_q_points_1d=sq)
    om = M.Multigrid(p, nq, quad, n, deform=0.05, coarse_max_dofs=cmax, smoother_degree=degree,
                     fine_smoother_nq=sq or None)
    A = mg.operator()
    for seed in (8, 9):  # the second cycle starts from the first one's buffers
        r = O.splitmix64_uniform(seed, A.m())
        z = A.initialize_dof_vector()
        mg.vmult(z, torch.from_numpy(r).cuda())
        zo, zg = om.vmult(r), z.cpu().numpy()
        assert np.linalg.norm(zg - zo) <= 1e-4 * np.linalg.norm(zo)
        cons = om.levels[0]["problem"].constrained.astype(bool)
        assert np.array_equal(zg[cons], r[cons])
