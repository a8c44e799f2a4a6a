"""Applies through a DoF map on meshes large enough that faces are joined where the
kernel can: more than 256 workgroups of the Gauss kernel at q = 6..8, in orders of the
DoFs in which they are joined and in ones in which it depends on the form; more
than 16 (FP64) and 512 (FP32) workgroups of the collocation kernel at q = 9; and metric
terms larger than the memory-side cache at q = 5.

FP64: sums of a few hundred products per row, 1e-12.  FP32: 1e-5 (6e-8 times the
products of a row, of either sign)."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_face_join import NONE, _maps

pytestmark = pytest.mark.gpu

# workgroups of 7, 5 and 4 cells (q = 6, 7, 8), of 3 (q = 9)
CASES = [(4, 6, O.GAUSS, (13, 12, 12)), (5, 6, O.GAUSS, (13, 12, 12)),
         (5, 7, O.GAUSS, (11, 11, 11)), (6, 7, O.GAUSS, (11, 11, 11)),
         (6, 8, O.GAUSS, (11, 10, 10)), (7, 8, O.GAUSS, (11, 10, 10)),
         (5, 7, O.GAUSS, (18, 17, 17)), (8, 9, O.GLL, (5, 4, 3)),
         (8, 9, O.GLL, (12, 12, 11))]


def _reference(P, q, m, X, N, x):
    base = {np.asarray(P.cellX).reshape(P.E, 24)[e].tobytes(): e for e in range(P.E)}
    src = np.array([base[X[e].tobytes()] for e in range(P.E)])
    G = np.ascontiguousarray(np.asarray(P.G).reshape(P.E, -1)[src]).ravel()
    u = np.where(m == NONE, 0.0, x[np.where(m == NONE, 0, m)])
    u = np.ascontiguousarray(u).ravel()
    w = (O.bk5_evec(q, P.E, P.D, G, u) if P.collocation else
         O.bk3_evec(P.p + 1, q, P.E, P.B, P.D, G, u)).reshape(m.shape)
    y = np.zeros(N)
    np.add.at(y, m[m != NONE], w[m != NONE])
    return y


@pytest.mark.parametrize("p,q,quad,n", CASES)
def test_large_meshes_in_any_order(gpu, p, q, quad, n):
    import torch
    from benchmarks_amd.laplace import LaplaceOperator
    P = O.make_problem(p, q, quad, n, deform=0.05)
    for name, m, X, N in _maps(P, p, n, np.random.RandomState(p)):
        m = np.ascontiguousarray(m, dtype=np.uint32).reshape(P.E, -1)
        x = O.splitmix64_uniform(4, N)
        ref = _reference(P, q, m, X, N, x)
        ref32 = _reference(P, q, m, X, N, x.astype(np.float32).astype(np.float64))
        cons = np.setdiff1d(np.arange(N, dtype=np.uint32), m[m != NONE])
        for geometry in (0, 1) if quad == O.GAUSS else (0,):
            op = LaplaceOperator.from_arrays(p, q, quad, m, X, cons, N, with_fp32=True,
                                             geometry=geometry)
            for dt, tol, r in ((np.float64, 1e-12, ref), (np.float32, 1e-5, ref32)):
                xd = x.astype(dt)
                want = r.copy()
                want[cons] = xd[cons]
                y = torch.full((N,), float("nan"), dtype=torch.from_numpy(xd).dtype, device="cuda")
                op.vmult(y, torch.from_numpy(xd).cuda())
                got = y.cpu().numpy().astype(np.float64)
                err = np.linalg.norm(got - want) / np.linalg.norm(want)
                assert err <= tol, (name, geometry, dt, err)


def test_metric_larger_than_the_cache(gpu):
    """36 x 36 x 35 cells x 6 x 125 terms are 272 MB."""
    import torch
    from benchmarks_amd.laplace import LaplaceOperator
    p, q, n = 4, 5, (36, 36, 35)
    P = O.make_problem(p, q, O.GLL, n, deform=0.05)
    op = LaplaceOperator.from_arrays(p, q, O.GLL, P.map, P.cellX,
                                     np.flatnonzero(P.constrained).astype(np.uint32), P.N)
    x = O.splitmix64_uniform(4, P.N)
    ref = P.vmult(x)
    y = torch.empty(P.N, dtype=torch.float64, device="cuda")
    op.vmult(y, torch.from_numpy(x).cuda())
    assert np.linalg.norm(y.cpu().numpy() - ref) <= 1e-12 * np.linalg.norm(ref)


def _joins(op, N):
    """Whether the apply's kernel joins faces (its last template argument)."""
    import torch
    from torch.profiler import ProfilerActivity, profile
    x = torch.zeros(N, dtype=torch.float64, device="cuda")
    y = torch.empty_like(x)
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        op.vmult(y, x)
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages() if "k_apply_interp<" in e.key]
    assert len(names) == 1, names
    args = names[0].split("k_apply_interp<")[1].split(">")[0].split(",")
    return args[8].strip() == "true"


@pytest.mark.parametrize("p,q,n,ordered,shuffled", [
    (4, 6, (3, 3, 3), False, False), (4, 6, (13, 12, 12), True, True),
    (6, 8, (11, 10, 10), False, True), (7, 8, (11, 10, 10), False, True),
    (5, 7, (11, 11, 11), True, True), (5, 7, (18, 17, 17), False, True)])
def test_which_form_runs(gpu, p, q, n, ordered, shuffled):
    from benchmarks_amd.laplace import LaplaceOperator
    P = O.make_problem(p, q, O.GAUSS, n)
    cons = np.flatnonzero(P.constrained).astype(np.uint32)
    m = np.asarray(P.map, dtype=np.uint32)
    perm = np.random.RandomState(1).permutation(P.N).astype(np.uint32)
    t = np.where(m == NONE, NONE, perm[np.where(m == NONE, 0, m)]).astype(np.uint32)
    for mm, cc, want in ((m, cons, ordered), (t, perm[cons], shuffled)):
        op = LaplaceOperator.from_arrays(p, q, O.GAUSS, mm, P.cellX, cc, P.N)
        assert _joins(op, P.N) == want
