"""Entries of a caller's DoF map that lie outside the vector are refused, wherever they
stand, with the first one's position; the marker of constrained nodes is accepted."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu
NONE = 0xFFFFFFFF


@pytest.mark.parametrize("n", [(1, 1, 1), (3, 2, 2)])
def test_entries_out_of_range(gpu, n):
    from benchmarks_amd._lib import MfxError
    from benchmarks_amd.laplace import LaplaceOperator
    p, q = 2, 3
    P = O.make_problem(p, q, O.GAUSS, n)
    cons = np.flatnonzero(P.constrained).astype(np.uint32)

    def make(m):
        return LaplaceOperator.from_arrays(p, q, O.GAUSS, m, P.cellX, cons, P.N)

    base = np.asarray(P.map, dtype=np.uint32).copy()
    for at in (0, 1, base.size // 2, base.size - 1):
        for value, ok in ((P.N - 1, True), (P.N, False), (0x7FFFFFFF, False), (NONE - 1, False),
                          (NONE, True)):
            m = base.copy()
            m[at] = value
            if ok:
                make(m)
                continue
            m[base.size - 1] = value  # a later one is not the one named
            with pytest.raises(MfxError, match="map entry out of range at %d$" % at):
                make(m)
