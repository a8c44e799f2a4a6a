"""The two forms of the batched CG's steps on both sides of the line between them
(batch.cpp small_batch: 4096 tiles and segments in one instance): iterates after
step limits against the oracle, with metric terms stored and from the vertices;
and that the small form does not depend on the variants in use.

Tolerance: rounding (1e-16) times the steps (9) times the condition of the
Jacobi-preconditioned operators (2e4 at degree 2 on 46 cells per direction) is
2e-11; 1e-10."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

SMALL = (45, 45, 46)  # 3326 tiles of 28 cells + 752 segments of 1024 rows
LARGE = (46, 46, 45)  # 3400 + 768
OTHERS = [(6, (2, 3, 2)), (3, (17, 2, 1)), (4, (9, 10, 11)), (5, (8, 1, 1))]


def _kernels(f):
    """Names of the kernels that f launches."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        f()
        torch.cuda.synchronize()
    return {e.key for e in p.key_averages()}


def _batch(n, form):
    import torch
    from benchmarks_amd.laplace import BatchedLaplace
    B = BatchedLaplace([(2, n)] + OTHERS, autotune=False, deform=0.05)
    for p in range(2, 7):
        B.set_variant(p, B.tuning(p)["geometry"].index(form))
    b = torch.from_numpy(O.splitmix64_uniform(9, B.m())).cuda()
    B.zero_constrained(b)
    return B, b, B.compute_inverse_diagonal()


def _solve(B, b, inv, steps, use_graph):
    from benchmarks_amd.laplace import NoConvergence
    x = B.initialize_dof_vector()
    with pytest.raises(NoConvergence):
        B.solve(x, b, inv, max_steps=steps, abs_tol=1e-300, rel_tol=1e-14, use_graph=use_graph)
    return x


@pytest.mark.parametrize("form", ["stored", "on_the_fly"])
@pytest.mark.parametrize("n", [SMALL, LARGE])
def test_iterate_on_both_sides_of_the_line(gpu, n, form):
    B, b, inv = _batch(n, form)
    bh = b.cpu().numpy()
    inst = [(2, n)] + OTHERS
    for steps, use_graph in ((1, True), (9, False), (9, True)):
        xh = _solve(B, b, inv, steps, use_graph).cpu().numpy()
        for i, (p, m) in enumerate(inst):
            a, e = B.offsets[i], B.offsets[i + 1]
            P = O.make_problem(p, p + 1, O.GLL, m, deform=0.05)
            xo, r, _ = P.cg(bh[a:e], inv_diag=P.inverse_diagonal(), max_steps=steps,
                            abs_tol=1e-300, rel_tol=1e-14)
            assert r.steps == steps
            assert np.linalg.norm(xh[a:e] - xo) <= 1e-10 * np.linalg.norm(xo), (i, steps)


def test_variants_are_a_large_batch_s(gpu):
    """A small batch keeps its one-launch apply when a variant is set; a large one
    runs the variants."""
    for n, own in ((SMALL, True), (LARGE, False)):
        B, b, inv = _batch(n, "on_the_fly")
        B.set_variant(2, B.tuning(2)["default_variant"])
        _solve(B, b, inv, 2, False)
        names = _kernels(lambda: _solve(B, b, inv, 2, False))
        assert any("k_b_apply" in k for k in names) == own, names
        assert any("k_b_direction_small" in k for k in names) == own, names
