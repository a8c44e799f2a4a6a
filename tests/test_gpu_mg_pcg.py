"""The multigrid CG's fused vector passes: p.Ap from the apply's partials (plane,
patch and Gauss kernels) and, with more partials than one workgroup sums, from a
dot product of its own; a right-hand side that is not zero on the constrained
rows; a second solve from the first one's buffers.

The solution satisfies the oracle's operator to the tolerance of the solve (1e-10)
plus FP64 rounding of the residual recurrence, a few 1e-13: 2e-10."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p,q,quad,n,geometry", [(4, 5, O.GLL, (8, 8, 4), 1),
                                                 (2, 3, O.GAUSS, (24, 24, 24), 1),
                                                 (1, 2, O.GAUSS, (96, 64, 96), 0),
                                                 (2, 4, O.GAUSS, (56, 56, 48), 0)])
def test_solution_satisfies_the_oracles_operator(gpu, p, q, quad, n, geometry):
    import torch
    from benchmarks_amd.laplace import PreconditionMG, ReductionControl, SolverCG
    mg = PreconditionMG(p, q, quad, n, deform=0.05, geometry=geometry)
    A = mg.operator()
    P = O.make_problem(p, q, quad, n, deform=0.05)
    for seed, masked in ((3, True), (4, False)):
        b = O.splitmix64_uniform(seed, P.N)
        if masked:
            b[P.constrained.astype(bool)] = 0
        x = A.initialize_dof_vector()
        ctl = ReductionControl(60, 1e-300, 1e-10)
        SolverCG(ctl).solve(A, x, torch.from_numpy(b).cuda(), mg)
        r = b - P.vmult(x.cpu().numpy())
        assert np.linalg.norm(r) <= 2e-10 * np.linalg.norm(b), ctl.last_step()
