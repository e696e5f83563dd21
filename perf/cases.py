"""Workloads of the VPFP framework on one GPU, each through a public entry point.

Every case is a dict with a "kind":

  closures  one leapfrog + collision step composed from the vlapy.core-style
            closures on device tensors, the driver evaluated on the host
  relax     the collision operator and the field solve alone, on any number
            of x cells (no pushers)
  step      ops.step_n: a batch of fused leapfrog + collision steps
  scheme    ops.step_n_scheme: the same with a 4th- or 6th-order splitting
  inner     the inner loop of a run with host arrays in and out: per-step
            fields, series and the stored f
  scan      scan.Scan.run: many independent runs of uneven sizes together
  apply     Closure.apply: the learned correction on coarse velocity rows
  train     Closure.gradients: forward and backward of the same network

FP64 cases return every array in FP64; FP32 ones return fields and histories
in FP32 too, the precision a program with FP32 state keeps them in.  FP32
plans keep no moments here: f log f is NaN in them wherever the tails of f
round below zero.
"""

import math
import os

import numpy as np
import torch

import vlapy_amd

VMAX = 6.4
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(vlapy_amd.__file__)))
NETWORK = os.path.join(ROOT, "vlapy_amd", "data", "closure_c5.npz")


def listed():
    return [
        # a script that composes its own step from the closures, on the
        # default grid: small kernels, one call each
        {"name": "closures 32x512 fp64", "kind": "closures", "nx": 32, "nv": 512, "op": "lb"},
        # relaxation studies of the collision operator: rows that are not a
        # power of two, so the field solve is the direct transform
        {"name": "relax 100x1024 fp64", "kind": "relax", "nx": 100, "nv": 1024, "op": "dg", "precision": "fp64"},
        # collisionless Landau damping, the first run of any user
        {"name": "landau 64x512 fp64", "kind": "step", "nx": 64, "nv": 512, "precision": "fp64", "op": "lb",
         "nu": 0.0, "delta": False, "moments": False, "steps": 20},
        # collisional plasma wave with all stored moments
        {"name": "epw 64x1024 fp64", "kind": "step", "nx": 64, "nv": 1024, "precision": "fp64", "op": "dg",
         "nu": 1e-3, "delta": False, "moments": True, "steps": 20},
        # the same wave driven by a pulse through the inner loop that a run of
        # the reference calls, two x-modes of f stored per step
        {"name": "inner 64x1024 fp64", "kind": "inner", "nx": 64, "nv": 1024, "op": "dg", "steps": 100,
         "store": "modes"},
        # higher-order splitting: many more drifts and field solves per step
        {"name": "pefrl 64x1024 fp64", "kind": "scheme", "nx": 64, "nv": 1024, "scheme": "pefrl", "op": "dg",
         "nu": 1e-3, "steps": 5},
        # one high-resolution grid (filamentation), both storage types
        {"name": "fine 1024x8192 fp64", "kind": "step", "nx": 1024, "nv": 8192, "precision": "fp64", "op": "dg",
         "nu": 1e-4, "delta": False, "moments": False, "steps": 4},
        {"name": "fine 1024x8192 fp32", "kind": "step", "nx": 1024, "nv": 8192, "precision": "fp32", "op": "dg",
         "nu": 1e-4, "delta": False, "moments": False, "steps": 4},
        # a large parameter scan in the storage that keeps FP32 damping rates
        # exact, and a smaller one in FP64
        {"name": "scan 4096 fp32 delta", "kind": "scan", "n": 4096, "mix": 20261202, "precision": "fp32",
         "delta": True, "grouped": True, "op": "dg", "steps": 4},
        {"name": "scan 512 fp64", "kind": "scan", "n": 512, "mix": 7, "precision": "fp64", "delta": False,
         "grouped": True, "op": "dg", "steps": 4},
        # the learned correction of 512 coarse runs at nx = 64
        {"name": "apply 32768 rows", "kind": "apply", "rows": 32768},
        # one training batch of that network
        {"name": "train 4096 rows", "kind": "train", "rows": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closures", "relax", "step", "step", "step", "scheme", "inner", "scan", "scan", "apply",
                       "train"])
    op = rng.choice(["lb", "dg"])
    nx, nv = 2 ** rng.randint(4, 10), 2 ** rng.randint(7, 13)
    if kind == "closures":
        return {"kind": kind, "nx": min(nx, 256), "nv": min(nv, 2048), "op": op}
    if kind == "relax":
        return {"kind": kind, "nx": _log_int(rng, 2, 900), "nv": nv, "op": op,
                "precision": rng.choice(["fp64", "fp32"])}
    if kind == "step":
        precision = rng.choice(["fp64", "fp32"])
        return {"kind": kind, "nx": nx, "nv": nv, "precision": precision, "op": op,
                "nu": rng.choice([0.0, 10.0 ** rng.uniform(-5, -2)]), "delta": rng.random() < 0.3,
                "moments": precision == "fp64" and rng.random() < 0.5, "steps": rng.randint(1, 12)}
    if kind == "scheme":
        return {"kind": kind, "nx": min(nx, 256), "nv": min(nv, 2048), "scheme": rng.choice(["pefrl", "h-sixth"]),
                "op": op, "nu": rng.choice([0.0, 10.0 ** rng.uniform(-5, -2)]), "steps": rng.randint(1, 5)}
    if kind == "inner":
        return {"kind": kind, "nx": min(nx, 128), "nv": min(nv, 2048), "op": op, "steps": rng.randint(5, 100),
                "store": rng.choice(["modes", "all"])}
    if kind == "scan":
        precision = rng.choice(["fp64", "fp32"])
        return {"kind": kind, "n": _log_int(rng, 16, 2000), "mix": rng.randint(1, 10 ** 6), "precision": precision,
                "delta": rng.random() < 0.5, "grouped": rng.random() < 0.75, "op": op, "steps": rng.randint(1, 4)}
    if kind == "apply":
        return {"kind": kind, "rows": _log_int(rng, 64, 32768)}
    return {"kind": kind, "rows": _log_int(rng, 16, 4096)}


# --------------------------------------------------------------------------- inputs


def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _grid(nx, nv, k=0.3, vmax=VMAX):
    xmax = 2.0 * np.pi / k
    dx = xmax / nx
    x = np.linspace(dx / 2.0, xmax - dx / 2.0, nx)
    kx = np.fft.fftfreq(nx, d=dx) * 2.0 * np.pi
    okx = np.zeros(nx)
    okx[1:] = 1.0 / kx[1:]
    dv = 2.0 * vmax / nv
    v = np.linspace(-vmax + dv / 2.0, vmax - dv / 2.0, nv)
    kv = np.fft.fftfreq(nv, d=dv) * 2.0 * np.pi
    return {"x": x, "kx": kx, "one_over_kx": okx, "v": v, "kv": kv, "dv": dv, "k": k, "nx": nx, "nv": nv}


def _maxwellian(v):
    return np.exp(-v ** 2 / 2.0) / np.sqrt(2.0 * np.pi)


def _f0(g, seed):
    """Density perturbations of the box's first harmonics on a Maxwellian, with
    a slow drift and a temperature of each run's own."""
    rng = np.random.default_rng(seed)
    n, u = np.ones(g["nx"]), np.zeros(g["nx"])
    for m in (1, 2, 3):
        n += 0.05 / m * rng.uniform(0.5, 1.0) * np.cos(m * g["k"] * g["x"] + rng.uniform(0, 2 * np.pi))
        u += 0.02 / m * rng.uniform(-1.0, 1.0) * np.cos(m * g["k"] * g["x"] + rng.uniform(0, 2 * np.pi))
    w = g["v"][None, :] - u[:, None]
    return n[:, None] * np.exp(-w ** 2 / 2.0) / np.sqrt(2.0 * np.pi)


def _pulse(g, seed):
    rng = np.random.default_rng(seed + 1)
    return {"first": {"k0": g["k"], "w0": 1.16 * rng.uniform(0.98, 1.02), "t_L": 0.0, "t_R": 40.0, "t_wL": 5.0,
                      "t_wR": 5.0, "a0": 0.01 * rng.uniform(0.5, 1.0)}}


def _driver(g, pulses, t):
    out = np.zeros(g["nx"])
    for p in pulses.values():
        env = 0.5 * (np.tanh((t - p["t_L"]) / p["t_wL"]) - np.tanh((t - p["t_R"]) / p["t_wR"]))
        out = out + env * p["k0"] * p["a0"] * np.sin(p["k0"] * g["x"] - p["w0"] * t)
    return out


DT = 0.05
CLOSURES_NU, RELAX_NU, INNER_NU = 1e-2, 1e-2, 1e-3


def _scan_parameters(case, seed):
    """Wavenumbers, amplitudes and collision frequencies from the seed; the mix
    of grid sizes belongs to the case."""
    from vlapy_amd.scan import draw_parameters

    p, sizes = draw_parameters(case["n"], seed), draw_parameters(case["n"], case["mix"])
    p["nx"], p["nv"] = sizes["nx"], sizes["nv"]
    return p


def _rows(rows, seed):
    """Coarse velocity rows as a scan holds them: perturbed Maxwellians."""
    gen = torch.Generator(device=_dev()).manual_seed(seed)
    r = lambda: torch.rand(rows, 1, generator=gen, device=_dev(), dtype=torch.float64)  # noqa: E731
    v = torch.as_tensor(_grid(4, 256)["v"], device=_dev())[None, :]
    amp = 10.0 ** (-4.0 + 3.0 * r())
    return ((1.0 + amp * torch.cos(6.2831853 * r())) * torch.exp(-(v - 0.2 * amp) ** 2 / 2.0)
            / math.sqrt(2.0 * math.pi) * (1.0 + 0.2 * amp * torch.cos(3.0 * v + 6.2831853 * r())))


def _train_inputs(case, seed):
    x = _rows(case["rows"], seed)
    gen = torch.Generator(device=_dev()).manual_seed(seed + 1)
    v = torch.as_tensor(_grid(4, 256)["v"], device=_dev())[None, :]
    a = torch.randn(case["rows"], 3, generator=gen, device=_dev(), dtype=torch.float64)
    t = sum(a[:, j:j + 1] * v ** j for j in range(3)) * torch.exp(-v ** 2 / 2.0)
    return x.float().contiguous(), t.float().contiguous()


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("apply", "train"):
        from vlapy_amd import closure

        if kind == "apply":
            return {"case": case, "net": closure.Closure.load(NETWORK, max_rows=1),
                    "f": _rows(case["rows"], seed).float().contiguous()}
        x, t = _train_inputs(case, seed)
        return {"case": case, "net": closure.Closure(in_scale=2.5, out_scale=1e-5, max_rows=case["rows"], seed=3),
                "x": x, "target": t}
    if kind == "scan":
        from vlapy_amd.scan import Scan

        return {"case": case, "scan": Scan(_scan_parameters(case, seed), vmax=VMAX, dt=0.1, op=case["op"],
                                           precision=case["precision"], delta=case["delta"],
                                           grouped=case["grouped"])}
    g = _grid(case["nx"], case["nv"])
    s = {"case": case, "grid": g}
    f0 = _f0(g, seed)
    if kind in ("closures", "relax", "inner"):
        from vlapy_amd import field_driver

        pulses = _pulse(g, seed)
        nu = {"closures": CLOSURES_NU, "relax": RELAX_NU, "inner": INNER_NU}[kind]
        params = {"nu": nu, "nx": g["nx"], "nv": g["nv"],
                  "fokker-planck": {"type": case["op"], "solver": "batched_tridiagonal"},
                  "vlasov-poisson": {"time": "leapfrog", "vdfdx": "exponential", "edfdv": "exponential",
                                     "poisson": "spectral"},
                  "backend": {"core": "hip", "precision": case.get("precision", "fp64")}}
        rules = {"space": ["k0", "k1"] if case.get("store") == "modes" else "all"}
        stuff = dict(g, nu=nu, dt=DT, f=f0, e=np.zeros(g["nx"]), rules_to_store_f=rules,
                     precision=params["backend"]["precision"],
                     driver_function=field_driver.get_driver_function(g["x"], pulses))
        if kind == "inner":
            from vlapy_amd import outer_loop

            t = DT * np.arange(case["steps"])
            s["storage"], s["loop"] = outer_loop.get_sim_config_and_inner_loop_step(params, stuff, case["steps"],
                                                                                    rules)
            s["t"], s["driver"] = t, np.stack([stuff["driver_function"](ti) for ti in t])
            return s
        from vlapy_amd.core import field, step

        s["fp"] = step.get_collision_step(stuff, params)
        s["f"] = torch.as_tensor(f0, device=_dev()).to(
            torch.float64 if stuff["precision"] == "fp64" else torch.float32).contiguous()
        if kind == "closures":
            s["vp"] = step.get_vlasov_poisson_step(params, stuff)
            s["e"] = torch.as_tensor(_driver(g, pulses, 0.0), device=_dev())
        else:
            s["solve"] = field.get_field_solver(stuff, "spectral")
            s["driver"] = torch.as_tensor(_driver(g, pulses, 0.0), device=_dev())
        return s
    from vlapy_amd._lib import Plan

    precision = case.get("precision", "fp64")
    plan = Plan(g["nx"], g["nv"], precision, g["kx"], g["one_over_kx"], g["v"], g["kv"], g["dv"], case["nu"], DT,
                case["op"])
    if case.get("delta"):
        plan.set_delta(True)
        f0 = f0 - _maxwellian(g["v"])[None, :]
    n, dev = case["steps"], _dev()
    s["plan"] = plan
    s["f"] = torch.as_tensor(f0, device=dev).to(torch.float64 if precision == "fp64" else torch.float32).contiguous()
    s["e"] = torch.zeros(g["nx"], dtype=torch.float64, device=dev)
    s["e_hist"] = torch.empty(n, g["nx"], dtype=torch.float64, device=dev)
    s["series"] = torch.empty(n, 2, dtype=torch.float64, device=dev)
    s["moments"] = (torch.empty(n, 8, g["nx"], dtype=torch.float64, device=dev)
                    if case.get("moments") or kind == "scheme" else None)
    if kind == "scheme":
        pulses = _pulse(g, seed)
        s["driver"] = torch.as_tensor(np.stack([[_driver(g, pulses, DT * (i + 0.2 * j)) for j in range(5)]
                                                for i in range(n)]), device=dev)
    return s


# --------------------------------------------------------------------------- the calls


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "closures":
        e, f = s["vp"](e=s["e"], f=s["f"], t=1.0)
        return {"e": e, "f": s["fp"](f)}
    if kind == "relax":
        f = s["fp"](s["f"])
        e = s["solve"](s["driver"], f)
        return {"f": f, "e": e if case["precision"] == "fp64" else e.float()}
    if kind == "step":
        from vlapy_amd import ops

        ops.step_n(s["plan"], s["f"], s["e"], case["steps"], None, s["e_hist"], s["moments"], s["series"])
        out = {"e": s["e"], "e_hist": s["e_hist"], "series": s["series"]}
        if case["precision"] == "fp32":
            out = {k: t.float() for k, t in out.items()}
        return dict(out, f=s["f"], moments=s["moments"])
    if kind == "scheme":
        from vlapy_amd import ops

        ops.step_n_scheme(s["plan"], case["scheme"], s["f"], s["e"], case["steps"], s["driver"], s["e_hist"],
                          s["moments"], s["series"])
        return {k: s[k] for k in ("f", "e", "e_hist", "moments", "series")}
    if kind == "inner":
        st = s["storage"] = s["loop"](s["t"], s["driver"], s["storage"])
        return {"f": st["f"], "e": st["e"], "stored_f": st["stored_f"], "fields": st["fields"],
                "series": {k: v for k, v in st["series"].items() if not k.startswith("mean_t_plus")}}
    if kind == "scan":
        sc = s["scan"]
        e2 = sc.run(case["steps"])
        lo = case["precision"] == "fp32"
        return {"e2": e2.astype(np.float32) if lo else e2, "f": [c.f for c in sc.classes],
                "e": [c.e.float() if lo else c.e for c in sc.classes]}
    if kind == "apply":
        return s["net"].apply(s["f"])
    grad, loss = s["net"].gradients(s["x"], s["target"])
    return {"grad": grad, "loss": loss}


# --------------------------------------------------------------------------- work


def _step_flops(nx, nv, kicks, drifts, collide):
    """Per cell: a real transform pair is 5 log2 N, the phases 6; the
    tridiagonal step with its moments about 20."""
    cell = kicks * (5 * math.log2(nv) + 6) + drifts * (5 * math.log2(nx) + 8) + (20 if collide else 0)
    return cell * nx * nv


def work(case):
    kind = case["kind"]
    if kind == "apply":
        return {"bytes": 2 * case["rows"] * 1024 + 4 * 41793, "flops": case["rows"] * 21.3e6}
    if kind == "train":
        return {"bytes": 2 * case["rows"] * 1024 + 8 * 41793, "flops": case["rows"] * 3 * 21.3e6}
    if kind == "scan":
        p = _scan_parameters(case, 0)
        size = 4 if case["precision"] == "fp32" else 8
        cells = int(np.sum(p["nx"] * p["nv"]))
        flops = sum(_step_flops(int(nx), int(nv), 2, 1, True) for nx, nv in zip(p["nx"], p["nv"]))
        return {"bytes": 2 * size * cells, "flops": case["steps"] * flops}
    nx, nv, n = case["nx"], case["nv"], case.get("steps", 1)
    size = 4 if case.get("precision") == "fp32" else 8
    if kind == "relax":
        return {"bytes": 2 * size * nx * nv + 16 * nx, "flops": 22 * nx * nv}
    collide = case.get("nu", 1.0) > 0.0
    kicks, drifts = {"closures": (2, 1), "inner": (2, 1), "step": (2 if collide else 1, 1),
                     "scheme": (6 if case.get("scheme") == "h-sixth" else 4, 5)}[kind]
    b = 2 * size * nx * nv
    if kind in ("step", "scheme"):
        b += n * nx * 8 * (1 + (8 if case.get("moments") or kind == "scheme" else 0))
    if kind == "inner":
        b += n * (nx * 8 * 9 + (2 * nv * 8 if case["store"] == "modes" else nx * nv * 8))
    return {"bytes": b, "flops": n * _step_flops(nx, nv, kicks, drifts, collide)}


# --------------------------------------------------------------------------- 64-bit results


def _shift(f, phi, dim):
    """Re ifft(exp(-i m phi) fft(f)) along dim; phi holds the phase of the
    first harmonic of every line."""
    n = f.shape[dim]
    m = torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64, device=f.device)
    th = m * phi.unsqueeze(-1) if dim == f.dim() - 1 else m.unsqueeze(-1) * phi.unsqueeze(-2)
    return torch.fft.ifft(torch.polar(torch.ones_like(th), -th) * torch.fft.fft(f, dim=dim), dim=dim).real


def _trapz(f, dv):
    return dv * (f.sum(-1) - 0.5 * (f[..., 0] + f[..., -1]))


def _field(f, dv, okx):
    return torch.fft.ifft(1j * okx * torch.fft.fft(1.0 - _trapz(f, dv), dim=-1), dim=-1).real


def _collide(f, v, dv, ndt, op):
    """Implicit Lenard-Bernstein / Dougherty step by Gaussian elimination along
    v; ndt (nu dt) broadcasts over the rows of f."""
    vbar = _trapz(f * v, dv) if op == "dg" else torch.zeros_like(f[..., 0])
    temp = _trapz(f * (v - vbar.unsqueeze(-1)) ** 2, dv)
    a0, h = -temp / dv ** 2, 0.5 / dv
    shape, nv = f.shape, f.shape[-1]
    vb, a0, ndt = (t.reshape(-1) for t in torch.broadcast_tensors(vbar, a0, ndt))
    lo = (ndt * (a0 + (v[:, None] - vb) * h))        # row m + 1, column m
    up = (ndt * (a0 - (v[:, None] - vb) * h))        # row m - 1, column m
    b = 1.0 - 2.0 * ndt * a0
    x = f.reshape(-1, nv).t().contiguous()
    back = x.is_cuda and x.shape[1] <= 512           # few rows: numpy on the host is quicker
    if back:
        lo, up, b, x = (t.cpu().numpy() for t in (lo, up, b, x))
    c = [None] * nv
    c[0] = up[1] / b
    x[0] = x[0] / b
    for m in range(1, nv):
        den = 1.0 / (b - lo[m - 1] * c[m - 1])
        c[m] = up[m + 1] * den if m + 1 < nv else None
        x[m] = (x[m] - lo[m - 1] * x[m - 1]) * den
    for m in range(nv - 2, -1, -1):
        x[m] -= c[m] * x[m + 1]
    x = torch.as_tensor(x, device=f.device)
    return x.t().contiguous().reshape(shape)


def _moments(f, v, dv):
    return torch.stack([_trapz(f * v ** p, dv) for p in range(6)] + [_trapz(f ** 2, dv), _trapz(f * torch.log(f), dv)])


_XSI, _LAM, _CHI = 0.1786178958448091, -0.2123418310626054, -0.6626458266981849e-1
_SIXTH = (0.168735950563437422448196, 0.377851589220928303880766, -0.093175079568731452657924,
          0.049086460976116245491441, 0.264177609888976700200146, 0.186735929134907054308413,
          -0.000069728715055305084099, -0.000625704827430047189169, -0.002213085124045325561636,
          -2.916600457689847816445691e-6, 3.048480261700038788680723e-5, 4.985549387875068121593988e-7)


def _stages(kind, scheme=None):
    """(kick weight before each drift, drift weights, last kick weight)"""
    if kind != "scheme":
        return [0.5], [1.0], 0.5
    if scheme == "pefrl":
        k0 = 0.5 * (1.0 - 2.0 * _LAM)
        return [0.0, k0, _LAM, _LAM, k0], [_XSI, _CHI, 1.0 - 2.0 * (_CHI + _XSI), _CHI, _XSI], 0.0
    a1, a2, a3, b1, b2, b3, c1, c2, c3, d2, d3, e3 = _SIXTH
    k1 = b1 + 2.0 * c1 * DT ** 2
    k2 = b2 + 2.0 * c2 * DT ** 2 + 4.0 * d2 * DT ** 4
    k3 = b3 + 2.0 * c3 * DT ** 2 + 4.0 * d3 * DT ** 4 - 8.0 * e3 * DT ** 6
    return [k1, k2, k3, k3, k2], [a1, a2, a3, a2, a1], k1


def _exact_grid(case, seed):
    kind = case["kind"]
    g = _grid(case["nx"], case["nv"])
    dev = _dev()
    put = lambda a: torch.as_tensor(a, device=dev)  # noqa: E731
    f = put(_f0(g, seed))
    v, okx, dv = put(g["v"]), put(g["one_over_kx"]), g["dv"]
    dk_x, dk_v = g["kx"][1] if g["nx"] > 1 else 0.0, g["kv"][1]
    pulses = _pulse(g, seed)
    fp32, delta = case.get("precision") == "fp32", case.get("delta")
    back = put(_maxwellian(g["v"]))
    if fp32:  # the state a program hands over is FP32
        f = (f - back).float().double() + back if delta else f.float().double()
    nu = torch.tensor(case.get("nu", {"closures": CLOSURES_NU, "relax": RELAX_NU, "inner": INNER_NU}.get(kind)),
                      dtype=torch.float64, device=dev)
    if kind == "relax":
        f = _collide(f, v, dv, nu * DT, case["op"])
        return {"f": f, "e": put(_driver(g, pulses, 0.0)) + _field(f, dv, okx)}
    n = case.get("steps", 1)
    e = put(_driver(g, pulses, 0.0)) if kind == "closures" else torch.zeros(g["nx"], dtype=torch.float64, device=dev)
    kicks, drifts, last = _stages(kind, case.get("scheme"))
    eh, mo, se, st = [], [], [], []
    for i in range(n):
        for j, (kw, dw) in enumerate(zip(kicks, drifts)):
            if kw:
                f = _shift(f, dk_v * kw * DT * e, 1)
            f = _shift(f, dk_x * dw * DT * v, 0)
            t = {"closures": 1.0 + DT, "inner": DT * i + DT, "scheme": DT * (i + 0.2 * j)}.get(kind)
            d = put(_driver(g, pulses, t)) if t is not None else torch.zeros_like(e)
            e = d + _field(f, dv, okx)
        if last:
            f = _shift(f, dk_v * last * DT * e, 1)
        if nu > 0.0:
            f = _collide(f, v, dv, nu * DT, case["op"])
        eh.append(e)
        se.append(torch.stack([(e ** 2).mean(), (d ** 2).mean()]))
        if case.get("moments") or kind in ("scheme", "inner"):
            mo.append(_moments(f, v, dv))
        if kind == "inner":
            st.append(torch.fft.fft(f, dim=0)[:2] if case["store"] == "modes" else f)
    if kind == "closures":
        return {"e": e, "f": f}
    eh, se = torch.stack(eh), torch.stack(se)
    mo = torch.stack(mo) if mo else None
    if kind == "inner":
        de = np.stack([_driver(g, pulses, DT * i) for i in range(n)])
        de2 = np.mean(de ** 2, axis=1)
        fields = {key: mo[:, row] for row, key in enumerate(("n", "j", "T", "q", "fv4", "vN"))}
        series = {"mean_n": mo[:, 0].mean(-1), "mean_j": mo[:, 1].mean(-1), "mean_T": mo[:, 2].mean(-1),
                  "mean_e2": se[:, 0], "mean_de2": de2, "mean_cum_de2": np.cumsum(de2),
                  "mean_f2": mo[:, 6].mean(-1), "mean_flogf": mo[:, 7].mean(-1)}
        return {"f": f, "e": e, "stored_f": torch.stack(st), "fields": dict(fields, e=eh, driver=de),
                "series": series}
    if delta:
        f = f - back
    return {"f": f, "e": e, "e_hist": eh, "series": se, "moments": mo}


def _exact_scan(case, seed):
    p = _scan_parameters(case, seed)
    dev, dt, n = _dev(), 0.1, case["steps"]
    e2, fs, es = torch.zeros(n, case["n"], dtype=torch.float64, device=dev), [], []
    for nx, nv in sorted(set(zip(p["nx"].tolist(), p["nv"].tolist()))):
        idx = np.nonzero((p["nx"] == nx) & (p["nv"] == nv))[0]
        g = _grid(nx, nv)
        k = torch.as_tensor(p["k"][idx], device=dev)[:, None]
        amp = torch.as_tensor(p["amp"][idx], device=dev)[:, None]
        nu = torch.as_tensor(p["nu"][idx], device=dev)[:, None]
        v = torch.as_tensor(g["v"], device=dev)
        x = (torch.arange(nx, dtype=torch.float64, device=dev) + 0.5) * (2.0 * math.pi / nx) / k
        okx = torch.as_tensor(_grid(nx, 4, 1.0)["one_over_kx"], device=dev) / k
        back = torch.exp(-v ** 2 / 2.0) / math.sqrt(2.0 * math.pi)
        f = (1.0 + amp * torch.cos(k * x)).unsqueeze(-1) * back
        if case["precision"] == "fp32":
            f = (f - back).float().double() + back if case["delta"] else f.float().double()
        e = torch.zeros(idx.size, nx, dtype=torch.float64, device=dev)
        at = torch.as_tensor(idx, device=dev)
        for i in range(n):
            f = _shift(f, g["kv"][1] * 0.5 * dt * e, 2)
            f = _shift(f, k * dt * v, 1)
            e = _field(f, g["dv"], okx)
            f = _shift(f, g["kv"][1] * 0.5 * dt * e, 2)
            f = _collide(f, v, g["dv"], nu * dt, case["op"])
            e2[i, at] = (e ** 2).mean(-1)
        fs.append(f - back if case["delta"] else f)
        es.append(e)
    return {"e2": e2, "f": fs, "e": es}


def _network(p, x):
    """The convolution network of include/vpfc.h on rows x, in 64 bits."""
    at = 0

    def take(n):
        nonlocal at
        at += n
        return p[at - n:at]

    def taps(a):  # [rows, c, 256] -> [rows, 5 c, 256], tap-major
        a = torch.nn.functional.pad(a, (2, 2))
        return torch.cat([a[:, :, j:j + 256] for j in range(5)], dim=1)

    a = x.unsqueeze(1)
    for width in (5, 320, 320):
        w, b = take(64 * width).reshape(64, width), take(64)
        a = torch.tanh(torch.matmul(w, taps(a)) + b[:, None])
    w, b = take(320).reshape(1, 320), take(1)
    return (torch.matmul(w, taps(a)) + b[:, None])[:, 0]


def exact(case, seed):
    kind = case["kind"]
    if kind == "scan":
        return _exact_scan(case, seed)
    if kind == "apply":
        f = _rows(case["rows"], seed).float().double()
        with np.load(NETWORK, allow_pickle=False) as z:
            net = {key: torch.as_tensor(z[key], device=f.device).double()
                   for key in ("params", "in_scale", "out_scale", "cons_v", "cons_bg")}
        v, bg = net["cons_v"], net["cons_bg"]
        w = torch.ones_like(v)
        w[0] = w[-1] = 0.5
        powers = torch.stack([v ** j for j in range(3)])
        gram = (powers * w * bg) @ powers.t()
        out = []
        for part in f.split(2048):
            y = _network(net["params"], net["in_scale"] * part)
            c = torch.linalg.solve(gram.cpu(), ((y * w) @ powers.t()).t().cpu()).to(f.device).t()
            out.append(part + net["out_scale"] * (y - bg * (c @ powers)))
        return torch.cat(out)
    if kind == "train":
        from vlapy_amd import closure

        x, t = _train_inputs(case, seed)
        p = torch.as_tensor(closure.init_params(3), device=x.device).double().requires_grad_()
        loss, n = torch.zeros((), dtype=torch.float64, device=x.device), case["rows"] * 256
        for a, b in zip(x.split(1024), t.split(1024)):
            part = ((_network(p, 2.5 * a.double()) - b.double()) ** 2).sum() / n
            part.backward()
            loss += part.detach()
        return {"grad": p.grad, "loss": loss.reshape(1)}
    return _exact_grid(case, seed)
