"""The batched collocation variants' default against the tile that launch_apply
uses (host arithmetic only): the cells per workgroup are those whose count is one
workgroup, and one cell more two."""
import ctypes

import pytest


class RowMesh(ctypes.Structure):
    _fields_ = [("n", ctypes.c_uint32 * 3)]


@pytest.mark.parametrize("p", range(2, 7))
def test_default_variant_is_the_default_tile(p):
    from benchmarks_amd import _lib
    L = ctypes.CDLL(_lib.LIB_PATH)
    blocks = L._ZN3mfx14apply_n_blocksEiibjNS_7RowMeshE
    blocks.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_bool, ctypes.c_uint32, RowMesh]
    blocks.restype = ctypes.c_uint32
    describe = L._ZN3mfx21launch_colloc_variantEiiPKdS1_S1_PdPKjjPKtPKiP12ihipStream_tPiSB_
    describe.argtypes = [ctypes.c_int] * 2 + [ctypes.c_void_p] * 5 + [ctypes.c_uint32] + \
        [ctypes.c_void_p] * 5
    cells, prefetch = ctypes.c_int(), ctypes.c_int()
    describe(p, L._ZN3mfx22colloc_default_variantEi(p), None, None, None, None, None, 0, None, None,
             None, ctypes.addressof(cells), ctypes.addressof(prefetch))
    n = cells.value
    assert blocks(p, p + 1, True, n, RowMesh()) == 1
    assert blocks(p, p + 1, True, n + 1, RowMesh()) == 2
