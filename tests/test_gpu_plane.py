"""The plane-per-lane kernel of box meshes with the metric from the vertices,
on meshes large enough for its rule, against the oracle: every instance,
undeformed and deformed, groups of cells that wrap over mesh rows, ragged
last groups, chunks of layers of different depth, single-cell rows.

FP64: sums of a few hundred products per row, 1e-12 relative.  FP32: the
metric is formed from coordinates rounded to FP32, whose differences (the cell
sizes, 1/n of the box) lose n 2^-24, twice in the metric: with n <= 64 cells
per direction 8e-6, and the products of the apply add about 1e-6."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

GLL, GAUSS = O.GLL, O.GAUSS
FORMS = ([(p, p + 1, GLL) for p in range(1, 8)] + [(p, p + 1, GAUSS) for p in range(1, 8)] +
         [(p, p + 2, GAUSS) for p in range(1, 7)])


def _need(p, q, quad, deform, fp32):
    """Waves from which the kernel is taken, at least (0: never)."""
    if quad == GLL:
        return 2048 if fp32 else 8192
    if deform == 0.0:
        return 4096 if fp32 else 5120
    if fp32:
        return 0 if (p, q) == (4, 5) else 6144 if q <= 4 else 12288 if q == 5 else 8192
    return 6144 if q <= 5 else 16384


def _check(op, P, dtype, tol):
    import torch
    x = O.splitmix64_uniform(5, P.N).astype(dtype)
    ref = P.vmult(x.astype(np.float64))
    y = torch.full((P.N,), float("nan"), dtype=getattr(torch, np.dtype(dtype).name),
                   device="cuda")
    xd = torch.from_numpy(x).cuda()
    for _ in range(2):
        op.vmult(y, xd)
    got = y.cpu().numpy().astype(np.float64)
    assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref)
    c = P.constrained.astype(bool)
    assert np.array_equal(got[c], x.astype(np.float64)[c])
    return xd, y, ref


@pytest.mark.parametrize("deform", [0.0, 0.05])
@pytest.mark.parametrize("p,q,quad", [f for f in FORMS if f[1] <= 7])
def test_fp64_forms_match_oracle(gpu, p, q, quad, deform):
    """Two groups per layer, the first of which wraps over rows."""
    from benchmarks_amd.laplace import LaplaceOperator
    C = 64 // q
    nx = 2 if q >= 6 and deform else 5
    ny = 1 if q >= 6 and deform else -(-(C + 2) // nx)
    groups = -(-nx * ny // C)
    nz = -(-_need(p, q, quad, deform, False) // groups) + 3
    op = LaplaceOperator(p, q, quad, n_cells=(nx, ny, nz), deform=deform, geometry=1)
    P = O.make_problem(p, q, quad, (nx, ny, nz), deform=deform)
    xd, y, ref = _check(op, P, np.float64, 1e-12)
    # accumulation onto a vector that is not zero
    y.fill_(0.5)
    op.vmult_add(y, xd)
    free = ~P.constrained.astype(bool)
    got = y.cpu().numpy()
    assert np.linalg.norm(got[free] - 0.5 - ref[free]) <= 1e-12 * np.linalg.norm(ref)
    assert np.all(got[~free] == 0.5)


@pytest.mark.parametrize("deform", [0.0, 0.05])
@pytest.mark.parametrize("p,q,quad", [f for f in FORMS if f[1] <= 8])
def test_fp32_forms_match_oracle(gpu, p, q, quad, deform):
    from benchmarks_amd.laplace import LaplaceOperator
    C = 64 // q
    need = _need(p, q, quad, deform, True)
    if not need:
        pytest.skip("the Gauss kernel runs this form at every size")
    n = [17, 13, 65]
    while n[2] > 64:
        n[0] += 2
        n[1] += 2
        n[2] = -(-need // -(-n[0] * n[1] // C))
    op = LaplaceOperator(p, q, quad, n_cells=n, deform=deform, geometry=1, with_fp32=True)
    P = O.make_problem(p, q, quad, n, deform=deform)
    _check(op, P, np.float32, 1e-5)


# rows of one cell, one row, more cells in a row than a group, exact groups
@pytest.mark.parametrize("n", [(1, 1, 2100), (1, 40, 800), (40, 1, 900), (24, 1, 1100),
                               (12, 12, 200), (13, 12, 170)])
def test_group_shapes(gpu, n):
    from benchmarks_amd.laplace import LaplaceOperator
    for deform in (0.0, 0.05):
        op = LaplaceOperator(2, 3, GAUSS, n_cells=n, deform=deform, geometry=1)
        P = O.make_problem(2, 3, GAUSS, n, deform=deform)
        _check(op, P, np.float64, 1e-12)


def test_dot_partials_drive_cg(gpu):
    """p.Ap from the kernel: Jacobi-CG takes the oracle's steps."""
    import torch
    from benchmarks_amd.laplace import (DiagonalMatrix, LaplaceOperator, ReductionControl,
                                        SolverCG)
    for p, q, quad, n, deform in ((2, 3, GLL, (21, 20, 120), 0.05), (3, 5, GAUSS, (12, 25, 90), 0.0)):
        op = LaplaceOperator(p, q, quad, n_cells=n, deform=deform, geometry=1)
        P = O.make_problem(p, q, quad, n, deform=deform)
        b = np.where(P.constrained.astype(bool), 0.0, O.splitmix64_uniform(3, P.N))
        x = op.initialize_dof_vector()
        ctl = ReductionControl(500, 1e-300, 1e-4)
        SolverCG(ctl).solve(op, x, torch.from_numpy(b).cuda(),
                            DiagonalMatrix(op.compute_inverse_diagonal()))
        _, r, _ = P.cg(b, inv_diag=P.inverse_diagonal(), rel_tol=1e-4, abs_tol=1e-300)
        assert abs(ctl.last_step() - r.steps) <= 1, (ctl.last_step(), r.steps)
