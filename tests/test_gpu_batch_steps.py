"""The batched CG's step in three launches (small batches whose variants were
not chosen) against the oracle: iterates after step limits on both sides of a
round of eight steps, on meshes whose tiles wrap over mesh rows, end ragged or hold
one cell, and a batch that mixes instances done at once with others.

Tolerance: rounding (1e-16) times the steps (17) times the condition of the
Jacobi-preconditioned operators (below 1e4 on these meshes) is 2e-11; 1e-10."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

INST = [(2, (5, 4, 3)), (3, (1, 6, 4)), (4, (11, 1, 3)), (5, (2, 3, 2)), (6, (1, 1, 5)),
        (2, (29, 2, 2)), (6, (4, 3, 2)), (3, (17, 2, 1)), (5, (8, 1, 1)), (4, (3, 3, 3)),
        (2, (40, 3, 5))]


@pytest.mark.parametrize("use_graph", [True, False])
@pytest.mark.parametrize("steps", [1, 7, 8, 9, 17])
def test_iterate_after_steps_matches_oracle(gpu, steps, use_graph):
    import torch
    from benchmarks_amd.laplace import BatchedLaplace, NoConvergence
    B = BatchedLaplace(INST, autotune=False, deform=0.05)
    b = torch.from_numpy(O.splitmix64_uniform(9, B.m())).cuda()
    B.zero_constrained(b)
    done = 3  # an instance without a right-hand side
    b[B.offsets[done]:B.offsets[done + 1]] = 0
    inv = B.compute_inverse_diagonal()
    for _ in range(2):  # the second solve starts from the first one's state
        x = B.initialize_dof_vector()
        with pytest.raises(NoConvergence):
            B.solve(x, b, inv, max_steps=steps, abs_tol=1e-300, rel_tol=1e-14,
                    use_graph=use_graph)
    bh, xh = b.cpu().numpy(), x.cpu().numpy()
    for i, (p, n) in enumerate(INST):
        a, e = B.offsets[i], B.offsets[i + 1]
        if i == done:
            assert not xh[a:e].any()
            continue
        P = O.make_problem(p, p + 1, O.GLL, n, deform=0.05)
        xo, r, _ = P.cg(bh[a:e], inv_diag=P.inverse_diagonal(), max_steps=steps, abs_tol=1e-300,
                        rel_tol=1e-14)
        assert r.steps == steps and not r.converged
        assert np.linalg.norm(xh[a:e] - xo) <= 1e-10 * np.linalg.norm(xo), (i, p, n)
