"""Rounding of the weight gradients' FP32 sums on a large grid.

The weights make every activation of channel 0 equal to 1 and the output gradient
of layer 6 equal to dy, so the gradient of that layer's middle weight is the sum
of dy, whose values are exact in bfloat16.  Every 32768th node holds 2^30: an FP32 sum
that holds it loses each later chunk of 32 nodes of 243/128 (60.75, less than half
of the 128 between neighbouring values), so the error shows how many chunks one chain adds.

Bound: a weight's sum goes through at most 32 products of a chunk, the chunks of a
block (16), the blocks of a unit (66: 4.28M nodes in 128 units are 1045 chunks), 32 units
per stride of the reduction and 4 strides: 150 roundings of 2^-24 each on positive
terms, 9e-6 relative.  One chain over a unit's chunks loses half of them, 3e-5."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAYERS = [(1, 16), (16, 32), (32, 64), (64, 64), (64, 64), (64, 32), (32, 16), (16, 1)]


def test_sum_over_a_large_grid(gpu):
    import torch
    from benchmarks_amd.laplace import LearnedPreconditioner
    w = [np.zeros((o, 27, i), np.float32) for i, o in LAYERS]
    for layer in (0, 1, 7):
        w[layer][0, 13, 0] = 1.0
    net = LearnedPreconditioner(0)
    net.set_params(np.concatenate([a.reshape(-1) for a in w]))
    dims = (257, 129, 129)
    n = dims[0] * dims[1] * dims[2]
    dy = torch.full((n,), 243.0 / 128.0, dtype=torch.float32, device="cuda")
    dy[::32768] = 2.0 ** 30
    g = net.gradient(dims, torch.ones(n, dtype=torch.float32, device="cuda"), dy)
    at = sum(a.size for a in w[:6]) + 13 * LAYERS[6][0]
    exact = dy.double().sum().item()
    assert abs(g[at].item() - exact) <= 9e-6 * exact
