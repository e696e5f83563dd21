"""A run of no steps: leaves f and E alone, and refuses a tuning that no run of
this plan can take, as a run of steps does."""

import numpy as np
import pytest

from oracle import vpfp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,refused", [(128, False), (256, True)])
def test_no_steps(nx, refused):
    import torch
    from vlapy_amd import ops
    from vlapy_amd._lib import Plan

    print("no steps", nx, flush=True)
    nv, k = 64, 0.35
    g = O.Grid.make(nx, nv, 2 * np.pi / k, 6.0)
    p = Plan(nx, nv, "fp64", g.kx, g.one_over_kx, g.v, g.kv, g.dv, 0.0, 0.1, "dg")
    dev = torch.device("cuda:0")
    f0 = torch.as_tensor(O.perturbed_maxwellian(g.x, g.v, k, 0.2), device=dev)
    e0 = torch.linspace(-1.0, 1.0, nx, dtype=torch.float64, device=dev)
    f, e = f0.clone(), e0.clone()
    ops.step_n(p, f, e, 0)
    p.set_tuning(fuse_field=2)
    for n in (0, 1):
        if refused:
            with pytest.raises(NotImplementedError):
                ops.step_n(p, f, e, n)
        elif n == 0:
            ops.step_n(p, f, e, n)
    torch.cuda.synchronize()
    assert torch.equal(f, f0) and torch.equal(e, e0)
