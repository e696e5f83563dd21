"""The fused step's field, formed by the row kernel from the drift's partial
densities: few of them (read by every row workgroup) and many (summed first),
at the smallest grids and on both sides of the rule, with a driver, the series
and the x-modes that ride on the next row launch; and the plan's own field
solves at sizes around a wavefront and off powers of two.

Tolerances: the FP64 bars of one-step parity, 1e-12 of max |f| and 1e-11 of
max |E| (E is the solve of 1 - n, a difference of numbers of order 1), over
three steps."""

import numpy as np
import pytest

from oracle import vpfp_oracle as O

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.abs(np.asarray(a) - np.asarray(b)).max() / np.abs(np.asarray(b)).max())


@pytest.mark.parametrize("nx,nv", [(4, 64), (16, 8192), (128, 1024), (128, 2048), (256, 64), (256, 512), (256, 1024),
                                   (512, 16), (1024, 64)])
@pytest.mark.parametrize("scheme", ["leapfrog", "pefrl"])
def test_step_field_and_riders(nx, nv, scheme):
    import torch

    from vlapy_amd import ops
    from vlapy_amd._lib import Plan

    print("field rows", nx, nv, scheme, flush=True)
    n, dt, nu, k = 3, 0.1, 1e-2, 0.35
    g = O.Grid.make(nx, nv, 2 * np.pi / k, 6.0)
    f0 = O.perturbed_maxwellian(g.x, g.v, k, 0.2)
    rng = np.random.default_rng(nx + nv)
    nf = 1 if scheme == "leapfrog" else 5
    drv = 0.01 * rng.standard_normal((n, nf, nx))
    p = Plan(nx, nv, "fp64", g.kx, g.one_over_kx, g.v, g.kv, g.dv, nu, dt, "dg")
    dev = torch.device("cuda:0")
    f, e = torch.as_tensor(f0, device=dev).clone(), torch.zeros(nx, dtype=torch.float64, device=dev)
    eh = torch.zeros(n, nx, dtype=torch.float64, device=dev)
    se = torch.zeros(n, 2, dtype=torch.float64, device=dev)
    nm = 2
    st = torch.zeros(n, nm, nv, dtype=torch.complex128, device=dev)
    d = torch.as_tensor(drv if nf > 1 else drv[:, 0], device=dev).contiguous()
    if scheme == "leapfrog":
        ops.step_n_store(p, f, e, n, st, nm, d, eh, None, se)
    else:
        ops.step_n_scheme(p, scheme, f, e, n, d, eh, None, se, st, nm)
    er, fr = np.zeros(nx), f0.copy()
    for i in range(n):
        calls = iter(drv[i])
        step = O.leapfrog_step if scheme == "leapfrog" else O.pefrl_step
        er, fr = step(g, er, fr, i * dt, dt, lambda t: next(calls))
        fr = O.collide(fr, g.v, nu, dt, g.dv, "dg")
        assert rel(eh[i].cpu().numpy(), er) < 1e-11, i
        ref = np.array([np.mean(er ** 2), np.mean(drv[i, -1] ** 2)])
        assert np.abs(se[i].cpu().numpy() / ref - 1.0).max() < 1e-11, i
        modes = np.fft.fft(fr, axis=0)[:nm]
        assert np.abs(st[i].cpu().numpy() - modes).max() < 1e-12 * np.abs(modes).max(), i
    assert rel(e.cpu().numpy(), er) < 1e-11
    assert rel(f.cpu().numpy(), fr) < 1e-12


@pytest.mark.parametrize("nx", [2, 3, 5, 63, 64, 65, 100, 1000, 4096])
@pytest.mark.parametrize("nv", [8, 511, 512, 3000])
def test_plan_field_solves_any_size(nx, nv):
    import torch

    from vlapy_amd import ops
    from vlapy_amd._lib import Plan

    print("plan field", nx, nv, flush=True)
    rng = np.random.default_rng(nx * nv)
    dx, dv = 0.3, 0.02
    kx = np.fft.fftfreq(nx, d=dx) * 2 * np.pi
    okx = np.zeros(nx)
    okx[1:] = 1.0 / kx[1:]
    f0 = rng.uniform(0.5, 1.5, (nx, nv)) / (nv * dv)
    drv = rng.standard_normal(nx)
    p = Plan(nx, nv, "fp64", one_over_kx=okx, dv=dv)
    dev = torch.device("cuda:0")
    f, d = torch.as_tensor(f0, device=dev), torch.as_tensor(drv, device=dev)
    out, ch = (torch.zeros(nx, dtype=torch.float64, device=dev) for _ in range(2))
    ops.compute_charges(p, f, ch)
    n_ref = O.compute_charges(f0, dv)
    assert rel(ch.cpu().numpy(), n_ref) < 1e-13
    ops.field(p, f, d, out)
    ref = drv + O.solve_for_field(n_ref, okx)
    assert rel(out.cpu().numpy(), ref) < 1e-11
    ops.solve_for_field(p, ch, out)
    assert np.abs(out.cpu().numpy() - (ref - drv)).max() < 1e-11 * np.abs(ref).max()
