"""PEFRL steps without a collision, moments or f store end with their field, in a
launch of its own: E, its history, the series and f against the oracle where the
other fields are formed from the partial densities directly and where they are
summed first, and the launches that a step takes.  Bars: those of one-step parity
(1e-12 in f, 1e-11 in E)."""

import numpy as np
import pytest

from oracle import vpfp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,nv,summed", [(4, 64, False), (64, 1024, False), (256, 1024, True), (512, 64, True)])
@pytest.mark.parametrize("series", [True, False])
def test_step_ends_with_its_field(nx, nv, summed, series):
    import torch
    from vlapy_amd import ops
    from vlapy_amd._lib import Plan

    print("pefrl end", nx, nv, series, flush=True)
    n, dt, k = 3, 0.1, 0.35
    g = O.Grid.make(nx, nv, 2 * np.pi / k, 6.0)
    f0 = O.perturbed_maxwellian(g.x, g.v, k, 0.2)
    drv = 0.01 * np.random.default_rng(nx + nv).standard_normal((n, 5, nx))
    dev = torch.device("cuda:0")
    p = Plan(nx, nv, "fp64", g.kx, g.one_over_kx, g.v, g.kv, g.dv, 0.0, dt, "dg")
    p.set_profiling(True)
    f, e = torch.as_tensor(f0, device=dev).clone(), torch.zeros(nx, dtype=torch.float64, device=dev)
    eh = torch.zeros(n, nx, dtype=torch.float64, device=dev)
    se = torch.zeros(n, 2, dtype=torch.float64, device=dev)
    ops.step_n_scheme(p, "pefrl", f, e, n, torch.as_tensor(drv, device=dev), eh, None, se if series else None)
    launches = {kind: c for kind, (_, c) in p.kernel_times().items()}
    assert launches == {"row": 4 * n, "drift": 5 * n, "field": (5 if summed else 1) * n, "other": 0}
    er, fr = np.zeros(nx), f0.copy()
    for i in range(n):
        calls = iter(drv[i])
        er, fr = O.pefrl_step(g, er, fr, i * dt, dt, lambda t: next(calls))
        assert np.abs(eh[i].cpu().numpy() - er).max() < 1e-11 * np.abs(er).max(), i
        if series:
            ref = np.array([np.mean(er ** 2), np.mean(drv[i, -1] ** 2)])
            assert np.abs(se[i].cpu().numpy() / ref - 1.0).max() < 1e-11, i
    assert np.array_equal(e.cpu().numpy(), eh[-1].cpu().numpy())
    assert np.abs(f.cpu().numpy() - fr).max() < 1e-12 * np.abs(fr).max()
