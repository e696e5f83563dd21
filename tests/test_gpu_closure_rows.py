"""Closure gradients at the edges of the row split over workgroups.

The gradient kernels give each of at most 256 workgroups every 256th row and
load the next row while one is worked on, so 1 row, a workgroup count that is
not full, one row more than workgroups and a ragged third pass take different
paths.  Bars: those of the other gradient tests (BF16 flips of activations at
rounding boundaries, 5e-3 of each block's norm; loss 1e-4).
"""

import numpy as np
import pytest

from oracle import closure_oracle as C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 3, 255, 256, 257, 515])
def test_gradients_over_row_counts(rows):
    import torch
    from vlapy_amd.closure import Closure, init_params

    rng = np.random.default_rng(rows)
    p = init_params(rows, out_gain=1.0)
    p += (0.05 * rng.standard_normal(p.size)).astype(np.float32)
    f = rng.standard_normal((rows, 256)).astype(np.float32)
    t = rng.standard_normal((rows, 256)).astype(np.float32)
    net = Closure(p, in_scale=0.7, max_rows=rows + 2)
    print("closure gradients rows", rows, flush=True)
    dev = torch.device("cuda:0")
    g, loss = net.gradients(torch.as_tensor(f, device=dev), torch.as_tensor(t, device=dev))
    g = g.cpu().numpy().astype(np.float64)
    l_ref, g_ref = C.loss_and_grad(p, f, t, 0.7, bf16=True)
    assert abs(loss.item() / l_ref - 1) <= 1e-4
    for name in ("W1", "b1", "W2", "b2", "W3", "b3", "W4", "b4"):
        lo, hi = C.OFF[name]
        e = np.linalg.norm(g[lo:hi] - g_ref[lo:hi]) / np.linalg.norm(g_ref[lo:hi])
        print(name, "grad rel err", e, flush=True)
        assert e <= 5e-3, name
