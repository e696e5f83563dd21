"""Large grids: one column tile per drift workgroup or several, rows of 8192.

A drift launch whose workgroups take one tile each runs a kernel of its own,
kept to the registers that let two workgroups share a CU, and FP32 rows of
nv = 8192 change their split with the number of rows.  The sizes are the
smallest and largest x columns that this concerns, the row counts lie on both
sides of the number of CUs, and the tiles per workgroup include counts that do
not divide the tiles.

Bars: FP64 those of the other steps (1e-12 in f, 1e-11 in E).  FP32: each of
the three steps applies two kicks and a drift, about 2 log2(N) = 26 roundings
of 2^-24 each to a value, in quadrature: 3 * 3 * sqrt(26) * 2^-24 = 2.7e-6,
doubled for the largest of ~1e6 values: 6e-6 in f.  E is the integral of the
density's error, whose roundings average over the 8192 columns but are common
to a row where f is large; it is held to 6e-6 max |f| L / 2 absolute.
"""

import numpy as np
import pytest

from oracle import vpfp_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nx,nv,tile", [(4, 64, 4), (512, 64, 16), (1024, 32, 8), (2048, 32, 8), (256, 8192, 8),
                                        (512, 8192, 16)])
@pytest.mark.parametrize("per", [1, 3])
def test_step_over_tiles_per_workgroup(nx, nv, tile, per, precision):
    import torch
    from vlapy_amd import ops
    from vlapy_amd._lib import Plan

    k, nu, dt, n = 0.35, 1e-3, 0.1, 3
    L = 2 * np.pi / k
    g = O.Grid.make(nx, nv, L, 6.0)
    f0 = O.perturbed_maxwellian(g.x, g.v, k, 0.2)
    e0 = 0.01 * np.random.default_rng(nx + nv).standard_normal(nx)
    p = Plan(nx, nv, precision, g.kx, g.one_over_kx, g.v, g.kv, g.dv, nu, dt, "dg")
    p.set_tuning(drift_tile=tile, drift_tiles=per)
    print("large tiles", nx, nv, tile, per, precision, flush=True)
    dev = torch.device("cuda:0")
    f = torch.as_tensor(f0, dtype=ops.f_dtype(p), device=dev).clone().contiguous()
    e = torch.as_tensor(e0, device=dev).clone()
    ops.step_n(p, f, e, n)
    torch.cuda.synchronize()
    er, fr = e0.copy(), f0.copy()
    for i in range(n):
        er, fr = O.leapfrog_step(g, er, fr, i * dt, dt)
        fr = O.collide(fr, g.v, nu, dt, g.dv, "dg")
    df = np.abs(f.double().cpu().numpy() - fr).max() / np.abs(fr).max()
    de = np.abs(e.cpu().numpy() - er).max()
    print("f", df, "E", de, "max E", np.abs(er).max(), flush=True)
    if precision == "fp64":
        assert df < 1e-12 and de < 1e-11 * np.abs(er).max()
    else:
        assert df < 6e-6 and de < 6e-6 * np.abs(fr).max() * L / 2


@pytest.mark.parametrize("nx,nv,precision,delta", [(256, 8192, "fp32", True), (512, 8192, "fp32", True),
                                                   (512, 4096, "fp32", False), (1024, 4096, "fp32", False),
                                                   (512, 8192, "fp64", False), (1024, 8192, "fp64", False)])
@pytest.mark.parametrize("nu", [0.0, 1e-3])
def test_row_split_by_rule_equals_the_eight_value_split(nx, nv, precision, delta, nu):
    """The split the rule takes against 8 values per thread, which every row
    length has: the same transforms in another order of sums, so twice the bars
    above (each side's own rounding); delta-f stores values a tenth as large."""
    import torch
    from vlapy_amd import ops
    from vlapy_amd._lib import Plan

    k, dt, n = 0.35, 0.1, 3
    g = O.Grid.make(nx, nv, 2 * np.pi / k, 6.0)
    f0 = O.perturbed_maxwellian(g.x, g.v, k, 0.1)
    if delta:
        f0 = f0 - np.exp(-g.v ** 2 / 2)[None, :] / np.sqrt(2 * np.pi)
    e0 = 0.01 * np.random.default_rng(nx + nv).standard_normal(nx)
    dev = torch.device("cuda:0")
    out = []
    for q in (0, 8):
        p = Plan(nx, nv, precision, g.kx, g.one_over_kx, g.v, g.kv, g.dv, nu, dt, "dg")
        if delta:
            p.set_delta(True)
        p.set_tuning(row_q=q)
        print("row split", nx, nv, precision, delta, nu, q, flush=True)
        f = torch.as_tensor(f0, dtype=ops.f_dtype(p), device=dev).clone().contiguous()
        e = torch.as_tensor(e0, device=dev).clone()
        ops.step_n(p, f, e, n)
        torch.cuda.synchronize()
        out.append((f.double().cpu().numpy(), e.cpu().numpy()))
    (fa, ea), (fb, eb) = out
    df = np.abs(fa - fb).max() / np.abs(fb).max()
    de = np.abs(ea - eb).max()
    print("f", df, "E", de, flush=True)
    if precision == "fp64":
        assert df < 2e-12 and de < 2e-11 * np.abs(eb).max()
    else:
        assert df < 1.2e-5 and de < 1.2e-5 * np.abs(fb).max() * np.pi / k
