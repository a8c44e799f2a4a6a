"""The start value of vmult (zero, identity rows) in one pass or two, and its
form where a caller's map gathers constrained DoFs, against the oracle's
element operator.  vmult sums at most 8 cells' contributions per DoF in FP64,
each from products of a few hundred terms: 1e-12 relative is far above that
rounding and far below any wrong row."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


# DoF counts around one wavefront, one workgroup and several
@pytest.mark.parametrize("p,n", [(1, (1, 1, 1)), (1, (3, 3, 3)), (2, (2, 2, 1)), (3, (7, 2, 3)),
                                 (2, (16, 15, 17))])
@pytest.mark.parametrize("det", [False, True])
def test_vmult_start_and_identity_rows(gpu, p, n, det):
    import torch
    from benchmarks_amd.laplace import LaplaceOperator
    op = LaplaceOperator(p, p + 1, O.GLL, n_cells=n, deform=0.05, with_fp32=True, geometry=1)
    op.set_deterministic(det)
    P = O.make_problem(p, p + 1, O.GLL, n, deform=0.05)
    x = O.splitmix64_uniform(7, P.N)
    ref = P.vmult(x)
    y = torch.full((P.N,), float("nan"), dtype=torch.float64, device="cuda")
    op.vmult(y, torch.from_numpy(x).cuda())
    assert _rel(y.cpu().numpy(), ref) <= 1e-12
    c = P.constrained.astype(bool)
    assert np.array_equal(y.cpu().numpy()[c], x[c])
    y32 = torch.full((P.N,), float("nan"), dtype=torch.float32, device="cuda")
    x32 = x.astype(np.float32)
    op.vmult(y32, torch.from_numpy(x32).cuda())
    assert _rel(y32.cpu().numpy().astype(np.float64), P.vmult(x32.astype(np.float64))) <= 1e-5
    assert np.array_equal(y32.cpu().numpy()[c], x32[c])


def test_map_that_gathers_constrained_dofs(gpu):
    """Constrained rows stay the identity when the map holds their DoFs."""
    import torch
    from benchmarks_amd.laplace import LaplaceOperator
    p, n = 2, (3, 2, 2)
    P = O.make_problem(p, p + 1, O.GAUSS, n, deform=0.05)
    E = P.E
    Nx, Ny = n[0] * p + 1, n[1] * p + 1
    e = np.arange(E)
    a = np.arange(p + 1)
    gx = (e % n[0] * p)[:, None] + a
    gy = (e // n[0] % n[1] * p)[:, None] + a
    gz = (e // (n[0] * n[1]) * p)[:, None] + a
    full = gx[:, None, None, :] + Nx * (gy[:, None, :, None] + Ny * gz[:, :, None, None])
    cons = np.flatnonzero(P.constrained).astype(np.uint32)
    op = LaplaceOperator.from_arrays(p, p + 1, O.GAUSS, full.astype(np.uint32), P.cellX, cons, P.N)
    x = O.splitmix64_uniform(9, P.N)
    x[cons] = 0.0  # gathered as zero either way: the free rows equal the masked map's
    y = torch.full((P.N,), float("nan"), dtype=torch.float64, device="cuda")
    op.vmult(y, torch.from_numpy(x).cuda())
    assert _rel(y.cpu().numpy(), P.vmult(x)) <= 1e-12
    assert np.array_equal(y.cpu().numpy()[cons], x[cons])
