"""vpfp_solve_for_field: the transform is staged before E is written, so the
output may be the charge density's own buffer; and a density of one wavenumber,
which it concentrates in one bin, gives E without the noise of other bins.

Bars: in place equals out of place to the bit.  A density of period 4 with
amplitudes a multiple of 2^-20 is exact in 1 - n, and every butterfly of its
transform adds equal values or cancels exactly: what is left are the roundings
along the way of its bin, at most two per level and direction,
4 log2(nx) 2^-53 relative.  Other sizes: 1e-11 of max |E| as elsewhere."""

import numpy as np
import pytest

from oracle import vpfp_oracle as O

pytestmark = pytest.mark.gpu


def _plan(nx):
    from vlapy_amd._lib import Plan

    dx = 0.3
    kx = np.fft.fftfreq(nx, d=dx) * 2 * np.pi
    okx = np.zeros(nx)
    okx[1:] = 1.0 / kx[1:]
    return Plan(nx, 4, "fp64", one_over_kx=okx), okx


@pytest.mark.parametrize("nx", [2, 4, 63, 64, 128, 500, 1024, 4096])
def test_field_in_place_of_the_density(nx):
    import torch
    from vlapy_amd import ops

    print("field in place", nx, flush=True)
    p, okx = _plan(nx)
    n = np.random.default_rng(nx).uniform(0.5, 1.5, nx)
    d = torch.as_tensor(n, device=torch.device("cuda:0"))
    out = torch.zeros_like(d)
    ops.solve_for_field(p, d, out)
    ops.solve_for_field(p, d, d)
    torch.cuda.synchronize()
    assert torch.equal(d, out)
    ref = O.solve_for_field(n, okx)
    assert np.abs(out.cpu().numpy() - ref).max() <= 1e-11 * max(np.abs(ref).max(), 1e-300)


@pytest.mark.parametrize("nx", [16, 256, 1024, 2048, 4096])
def test_one_wavenumber(nx):
    import torch
    from vlapy_amd import ops

    print("field of one wavenumber", nx, flush=True)
    p, okx = _plan(nx)
    a, b = 0.3 // 2.0 ** -20 * 2.0 ** -20, 0.4 // 2.0 ** -20 * 2.0 ** -20
    rho = np.tile([a, b, -a, -b], nx // 4)
    d = torch.as_tensor(1.0 - rho, device=torch.device("cuda:0"))
    out = torch.zeros_like(d)
    ops.solve_for_field(p, d, out)
    # rho = a cos + b sin of k x at the quarter periods, E = (b cos - a sin) / k
    ref = np.tile([b, -a, -b, a], nx // 4) * okx[nx // 4]
    err = np.abs(out.cpu().numpy() - ref).max() / np.abs(ref).max()
    print("relative error", err, flush=True)
    assert err <= 4 * np.log2(nx) * 2.0 ** -53
