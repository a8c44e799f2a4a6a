"""Transfers and smoothing on small, ragged and non-nested-looking grids: the
axis passes against dense interpolation matrices, and the Chebyshev smoother
against its recurrence in FP64.

Transfers are sums of at most (p+1)^3 products in FP64: 1e-13 relative.  The
FP32 smoother of k steps rounds each of its few operations per row and the
apply's sums of ~100 products: k x 100 x 2^-24 = 4e-5 bounds it for k = 6."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _gll(n):
    return O.basis_tables(n - 1, n, O.GLL)[2]


def _dense_1d(nc, pc, nf, pf):
    """Interpolation of the coarse degree-pc line at the fine nodes."""
    sc, sf = _gll(pc + 1), _gll(pf + 1)
    r = nf // nc
    P = np.zeros((nf * pf + 1, nc * pc + 1))
    for j in range(P.shape[0]):
        ef = min(j // pf, nf - 1)
        xi = ((ef % r) + sf[j - ef * pf]) / r
        for m in range(pc + 1):
            w = 1.0
            for k in range(pc + 1):
                if k != m:
                    w *= (xi - sc[k]) / (sc[m] - sc[k])
            P[j, ef // r * pc + m] = w
    return P


@pytest.mark.parametrize("pf,pc,nf,nc", [(2, 1, (1, 1, 1), (1, 1, 1)), (4, 2, (3, 1, 2), (3, 1, 2)),
                                         (1, 1, (2, 4, 6), (1, 2, 3)), (8, 4, (1, 2, 1), (1, 2, 1)),
                                         (3, 3, (4, 2, 2), (2, 1, 1)), (4, 1, (6, 2, 4), (3, 1, 2))])
def test_transfers_match_dense_interpolation(gpu, pf, pc, nf, nc):
    import torch
    from benchmarks_amd.laplace import LaplaceOperator, transfer_prolongate, transfer_restrict
    fine = LaplaceOperator(pf, pf + 1, O.GLL, n_cells=nf, geometry=1)
    coarse = LaplaceOperator(pc, pc + 1, O.GLL, n_cells=nc, geometry=1)
    P = [_dense_1d(nc[d], pc, nf[d], pf) for d in range(3)]
    K = np.kron(P[2], np.kron(P[1], P[0]))
    c = O.splitmix64_uniform(1, coarse.m())
    f = O.splitmix64_uniform(2, fine.m())
    got_f = transfer_prolongate(fine, coarse, torch.from_numpy(c).cuda()).cpu().numpy()
    got_c = transfer_restrict(fine, coarse, torch.from_numpy(f).cuda()).cpu().numpy()
    assert np.linalg.norm(got_f - K @ c) <= 1e-13 * np.linalg.norm(K @ c)
    assert np.linalg.norm(got_c - K.T @ f) <= 1e-13 * np.linalg.norm(K.T @ f)


@pytest.mark.parametrize("quad,dq,det", [(O.GLL, 1, False), (O.GLL, 1, True), (O.GAUSS, 2, False)])
@pytest.mark.parametrize("zero", [True, False])
@pytest.mark.parametrize("degree", [1, 2, 6])
def test_smoother_keeps_identity_rows(gpu, quad, dq, det, zero, degree):
    """Start vectors with nonzero constrained rows, whose operator is 1."""
    import torch
    from benchmarks_amd.laplace import LaplaceOperator, chebyshev_f32
    p, n = 3, (4, 3, 2)
    op = LaplaceOperator(p, p + dq, quad, n_cells=n, deform=0.05, with_fp32=True, geometry=1)
    if det:
        op.set_deterministic(True)
    Pb = O.make_problem(p, p + dq, quad, n, deform=0.05)
    inv = Pb.inverse_diagonal()
    b, x = O.splitmix64_uniform(3, Pb.N), O.splitmix64_uniform(4, Pb.N)
    lmin, lmax = 0.2, 3.0
    f = lambda a: torch.from_numpy(a.astype(np.float32)).cuda()  # noqa: E731
    b32, x32, inv32 = (a.astype(np.float32).astype(np.float64) for a in (b, x, inv))
    theta, delta = 0.5 * (lmax + lmin), 0.5 * (lmax - lmin)
    ref = np.zeros(Pb.N) if zero else x32
    d = inv32 * (b32 - Pb.vmult(ref)) / theta
    ref = ref + d
    rho = delta / theta
    for _ in range(1, degree):
        new = 1.0 / (2.0 * theta / delta - rho)
        d = new * rho * d + 2.0 * new / delta * inv32 * (b32 - Pb.vmult(ref))
        ref = ref + d
        rho = new
    got = f(x)
    for _ in range(2):  # the second call reuses the handle's scratch
        got = f(x)
        chebyshev_f32(op, f(inv), got, f(b), degree, lmin, lmax, zero)
    assert np.linalg.norm(got.cpu().numpy() - ref) <= 4e-5 * np.linalg.norm(ref)
