"""The plan autotuner on a grid whose default sums the partial densities before
the row kernel forms the field from them: that form is one of its candidates, and
the tuned plan keeps the step's bars (1e-12 in f, 1e-11 in E)."""

import os
import re

import numpy as np
import pytest

from oracle import vpfp_oracle as O

HERE = os.path.dirname(os.path.abspath(__file__))


def test_summed_field_is_a_candidate_wherever_the_rule_takes_it():
    src = open(os.path.join(HERE, "..", "vlapy_amd", "csrc", "vpfp.hip")).read()
    body = src[src.index("int autotune_plan("):]
    body = body[:body.index("tune_search(")]
    skips = re.findall(r"if \(fuse == -1([^;]*?)\)\s*continue;", body)
    # -1 is left out only where the candidate's own shape makes it mode 2
    assert len(skips) == 1 and "rule_mode(p->nx, drift_wgs(p->nv, C, dt, false)) == kFieldRows" in skips[0]


@pytest.mark.gpu
@pytest.mark.parametrize("nx,nv", [(128, 2048), (256, 64)])
def test_autotuned_plan_keeps_parity(nx, nv):
    import torch
    from vlapy_amd import ops
    from vlapy_amd._lib import Plan

    print("autotune", nx, nv, flush=True)
    k, nu, dt, n = 0.35, 1e-2, 0.1, 2
    g = O.Grid.make(nx, nv, 2 * np.pi / k, 6.0)
    f0 = O.perturbed_maxwellian(g.x, g.v, k, 0.2)
    p = Plan(nx, nv, "fp64", g.kx, g.one_over_kx, g.v, g.kv, g.dv, nu, dt, "dg")
    t = p.autotune(n_steps=4)
    print("tuning", t, flush=True)
    assert t["fuse_field"] in (-1, 0, 1, 2)
    p.set_tuning(**{key: t[key] for key in ("row_q", "drift_tile", "fuse_field", "drift_order", "drift_tiles")})
    dev = torch.device("cuda:0")
    f, e = torch.as_tensor(f0, device=dev).clone(), torch.zeros(nx, dtype=torch.float64, device=dev)
    ops.step_n(p, f, e, n)
    er, fr = np.zeros(nx), f0.copy()
    for i in range(n):
        er, fr = O.leapfrog_step(g, er, fr, i * dt, dt)
        fr = O.collide(fr, g.v, nu, dt, g.dv, "dg")
    assert np.abs(f.cpu().numpy() - fr).max() < 1e-12 * np.abs(fr).max()
    assert np.abs(e.cpu().numpy() - er).max() < 1e-11 * np.abs(er).max()
