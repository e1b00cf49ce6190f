"""The work that users of this framework have it do, as cases to measure.

A case is a dict of plain values.  `listed()` names the standing ones, `draw`
gives more of the same ranges, `prepare` makes what a program holds before the
call, `run` is one pass through the public entry points, `work` the bytes and
operations that a pass cannot do without and `exact` the same outputs in plain
64-bit torch.

Paths:
  host     one closure of a batch in host memory (GpuClosure.solve_host)
  closure  one closure of a batch on the device from the plain start
  loop     time steps of a whole flow on the device (run_steps), from its
           initial state: closure, uQ, reconstruction, dt, flux and update
  sweeps   the step's sweeps called one by one, and the mean and variance
  predict  the warm-start network's duals for a batch of cells
  grad     loss and gradient of the warm-start network for one batch
"""
import math

import numpy as np
import torch

from uqcreator_amd import mesh as meshes
from uqcreator_amd import native, workloads

KIND = {"burgers": native.BOUNDED_BARRIER, "euler1d": native.EULER1D, "euler2d": native.EULER2D,
        "sw2d": native.SHALLOW_WATER2D, "sw2d_barrier": native.SHALLOW_WATER2D_BARRIER}
PRECISION = {"fp64": native.FP64, "mixed": native.MIXED}
GAMMA, GRAVITY = 1.4, 9.81


def listed():
    return [
        # a program that keeps its cells in host memory and closes a few of them at a time: the smallest call
        {"name": "host_small", "path": "host", "closure": "euler2d", "d": 2, "degree": 3, "q1": 5, "cells": 96,
         "precision": "fp64"},
        # input/burgers1d_step.toml: 2000 cells, six moments; launches count more than work
        {"name": "burgers_loop", "path": "loop", "flow": "burgers", "cells": 2000, "degree": 5, "q1": 12,
         "steps": 128, "orders": "uniform", "precision": "fp64"},
        # input/euler2d_naca.toml and its mixed variant, the benchmark's flow
        {"name": "naca_loop_fp64", "path": "loop", "flow": "naca", "ni": 512, "nj": 128, "degree": 3, "q1": 5,
         "steps": 40, "orders": "uniform", "precision": "fp64"},
        {"name": "naca_loop_mixed", "path": "loop", "flow": "naca", "ni": 512, "nj": 128, "degree": 3, "q1": 5,
         "steps": 40, "orders": "uniform", "precision": "mixed"},
        # input/euler2d_naca_adaptive.toml: every cell on its own refinement level
        {"name": "naca_levels", "path": "loop", "flow": "naca", "ni": 512, "nj": 128, "degree": 3, "q1": 5,
         "steps": 40, "orders": "levels", "precision": "fp64"},
        # per-cell orders 1..6 on 7 x 7 points (up to 112 duals in a cell)
        {"name": "naca_orders_mixed", "path": "loop", "flow": "naca", "ni": 256, "nj": 64, "degree": 6, "q1": 7,
         "steps": 12, "orders": "mixed", "precision": "mixed"},
        # input/shallowwater2d_dambreak.toml on a coarser grid: 105 duals, 125 points, friction
        {"name": "dambreak_mixed", "path": "loop", "flow": "dambreak", "nx": 256, "degree": 4, "q1": 5, "steps": 12,
         "orders": "uniform", "precision": "mixed"},
        # the batched closure of the benchmark, plain and mixed, ragged batches
        {"name": "closure_fp64", "path": "closure", "closure": "euler1d", "d": 2, "degree": 4, "q1": 7,
         "cells": 100003, "precision": "fp64"},
        {"name": "closure_mixed", "path": "closure", "closure": "euler1d", "d": 2, "degree": 4, "q1": 7,
         "cells": 100003, "precision": "mixed"},
        # a program with a time loop of its own calls the sweeps one by one
        {"name": "sweeps_euler2d", "path": "sweeps", "flow": "naca", "ni": 512, "nj": 128, "degree": 3, "q1": 5},
        # the learned warm start: inference over the benchmark's cells, and its training step
        {"name": "warm_predict", "path": "predict", "closure": "euler2d", "d": 2, "degree": 3, "q1": 5,
         "cells": 65536, "hidden": 256},
        {"name": "warm_grad", "path": "grad", "closure": "euler2d", "d": 2, "degree": 3, "q1": 5, "rows": 1024,
         "hidden": 256},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["host", "closure", "closure", "loop", "loop", "loop", "loop", "sweeps", "predict", "grad"])
    precision = rng.choice(["fp64", "mixed"])
    if path == "host":
        return {"path": path, "closure": rng.choice(["euler1d", "euler2d", "sw2d_barrier"]), "d": 2,
                "degree": rng.randint(1, 3), "q1": rng.randint(4, 6), "cells": _log(rng, 1, 1024),
                "precision": precision}
    if path == "closure":
        if rng.random() < 0.5:
            return {"path": path, "closure": "euler1d", "d": 2, "degree": 4, "q1": 7, "cells": _log(rng, 256, 100000),
                    "precision": precision}
        return {"path": path, "closure": rng.choice(["euler1d", "euler2d", "sw2d_barrier"]), "d": 2,
                "degree": rng.randint(1, 3), "q1": rng.randint(4, 6), "cells": _log(rng, 256, 30000),
                "precision": precision}
    if path == "loop":
        flow = rng.choice(["burgers", "naca", "naca", "dambreak"])
        if flow == "burgers":
            deg = rng.choice([5, 5, rng.randint(2, 7)])
            q1 = 12 if deg == 5 else deg + rng.randint(3, 6)
            return {"path": path, "flow": flow, "cells": _log(rng, 100, 5000), "degree": deg, "q1": q1,
                    "steps": _log(rng, 16, 128), "orders": "uniform", "precision": precision}
        if flow == "naca":
            orders = rng.choice(["uniform", "uniform", "levels", "mixed"])
            deg, q1 = (3, 5) if orders != "mixed" else (rng.randint(4, 6), 7)
            if orders == "uniform" and rng.random() < 0.3:
                deg, q1 = 2, 4
            most = 512 if orders != "mixed" else 192
            return {"path": path, "flow": flow, "ni": 2 * _log(rng, 24, most // 2), "nj": _log(rng, 12, most // 4),
                    "degree": deg, "q1": q1, "steps": _log(rng, 4, 24 if orders != "mixed" else 10),
                    "orders": orders, "precision": precision}
        deg = rng.choice([2, 3, 4])
        return {"path": path, "flow": flow, "nx": _log(rng, 24, 180), "degree": deg, "q1": deg + 1,
                "steps": _log(rng, 4, 12), "orders": "uniform", "precision": precision}
    if path == "sweeps":
        if rng.random() < 0.6:
            return {"path": path, "flow": "naca", "ni": 2 * _log(rng, 24, 256), "nj": _log(rng, 12, 128),
                    "degree": rng.randint(1, 4), "q1": rng.randint(5, 7)}
        return {"path": path, "flow": "dambreak", "nx": _log(rng, 24, 180), "degree": rng.randint(2, 4), "q1": 5}
    if path == "predict":
        return {"path": path, "closure": rng.choice(["euler1d", "euler2d", "sw2d_barrier"]), "d": 2,
                "degree": rng.randint(2, 4), "q1": 5, "cells": _log(rng, 200, 65000), "hidden": rng.choice([128, 256])}
    return {"path": path, "closure": rng.choice(["euler1d", "euler2d"]), "d": 2, "degree": rng.randint(2, 4), "q1": 5,
            "rows": 32 * _log(rng, 2, 128), "hidden": rng.choice([128, 256])}


# ---------------------------------------------------------------------------
# shapes
# ---------------------------------------------------------------------------
def _basis(case):
    flow = case.get("flow")
    d = case["d"] if "d" in case else {"burgers": 1, "naca": 2, "dambreak": 3}[flow]
    deg = case["degree"]
    degrees = list(range(1, deg + 1)) if case.get("orders") in ("levels", "mixed") else [deg]
    return native.Basis(d, degrees, case["q1"])


def _closure_name(case):
    return case["closure"] if "closure" in case else {"burgers": "burgers", "naca": "euler2d",
                                                      "dambreak": "sw2d_barrier"}[case["flow"]]


def _mesh(case):
    if case["flow"] == "burgers":
        return meshes.mesh1d(case["cells"], 0.0, 3.0)
    if case["flow"] == "naca":
        return meshes.naca_ogrid(case["ni"], case["nj"])
    return meshes.quad_grid(case["nx"], case["nx"], -1.0, 1.0, -1.0, 1.0, native.BC_DIRICHLET)


def _n_cells(case):
    if "cells" in case:
        return case["cells"]
    return case["ni"] * case["nj"] if case["flow"] == "naca" else case["nx"] ** 2


def _problem(case):
    if case["flow"] == "burgers":
        return native.problem(native.BURGERS, flux=native.FLUX_LAX_FRIEDRICHS, cfl=0.5)
    if case["flow"] == "naca":
        return native.problem(native.EULER2D_PROBLEM, flux=native.FLUX_LAX_FRIEDRICHS, cfl=0.4)
    return native.problem(native.SHALLOW_WATER2D_PROBLEM, flux=native.FLUX_REFERENCE, cfl=0.45, friction=0.01,
                          friction_dim=2)


def _parameters(case):
    """Closure parameters, as the configurations of these flows have them."""
    name = _closure_name(case)
    p = {"epsilon": 1e-10}
    if name == "burgers":
        p.update(u_minus=2.9, u_plus=12.1)
    elif name == "euler1d":
        p.update(du_exact=1, safe_line_search=1)
    elif name == "euler2d":
        p.update(**({"epsilon": 1e-6} if "flow" in case else {"epsilon": 1e-9, "safe_line_search": 1}))
    else:
        p.update(epsilon=1e-8, barrier=0.01)
    return p


def _handle(case, basis):
    return native.GpuClosure(KIND[_closure_name(case)], basis,
                             precision=PRECISION[case.get("precision", "fp64")], **_parameters(case))


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


# ---------------------------------------------------------------------------
# plain 64-bit forms: closures, fluxes, Newton
# ---------------------------------------------------------------------------
def _u_of(name, L, want_du=False):
    """U(Lambda) for Lambda (..., S); with want_du also DU (..., S, S)."""
    S = L.shape[-1]
    if name == "burgers":
        lo, hi = 2.9, 12.1
        s = torch.sigmoid(L)
        U = lo + (hi - lo) * s
        return (U, ((hi - lo) * s * torch.sigmoid(-L))[..., None]) if want_du else U
    if name.startswith("euler"):
        v0, v, w = L[..., 0], L[..., 1:S - 1], L[..., S - 1]
        q = (v * v).sum(-1)
        g1 = 1.0 - GAMMA
        e = torch.exp((q / (2 * w) - v0 + GAMMA + torch.log(-w)) / g1)
        f = torch.cat([torch.ones_like(e)[..., None], -v / w[..., None],
                       ((q - 2 * w) / (2 * w * w))[..., None]], -1)  # U = e f
        U = e[..., None] * f
        if not want_du:
            return U
        de = torch.cat([-torch.ones_like(e)[..., None], v / w[..., None],
                        (-q / (2 * w * w) + 1 / w)[..., None]], -1) * (e / g1)[..., None]
        D = f[..., :, None] * de[..., None, :]
        for s in range(1, S - 1):
            D[..., s, s] -= e / w
            D[..., s, S - 1] += e * L[..., s] / (w * w)
            D[..., S - 1, s] += e * L[..., s] / (w * w)
        D[..., S - 1, S - 1] += e * (-q / w ** 3 + 1 / (w * w))
        return U, D
    b = 0.01 if name == "sw2d_barrier" else 0.0
    c = L[..., 0] + 0.5 * (L[..., 1] ** 2 + L[..., 2] ** 2)
    r = torch.sqrt(c * c + 4 * GRAVITY * b)
    h = torch.where(c > 0, (c + r) / (2 * GRAVITY), 2 * b / (r - torch.where(c > 0, -r, c)))
    a = torch.stack([torch.ones_like(c), L[..., 1], L[..., 2]], -1)
    U = h[..., None] * a
    if not want_du:
        return U
    D = (h / r)[..., None, None] * a[..., :, None] * a[..., None, :]
    D[..., 1, 1] += h
    D[..., 2, 2] += h
    return U, D


def _ds_of(name, u):
    """Plain start of the mean states u (..., S)."""
    if name == "burgers":
        return torch.zeros_like(u)
    if name.startswith("euler"):
        S = u.shape[-1]
        rho, m, E = u[..., 0], u[..., 1:S - 1], u[..., S - 1]
        ei = E - (m * m).sum(-1) / (2 * rho)
        q = (m * m).sum(-1)
        return torch.cat([(GAMMA - q / (2 * rho * ei) - torch.log(ei) + GAMMA * torch.log(rho))[..., None],
                          m / ei[..., None], (-rho / ei)[..., None]], -1)
    b = 0.01 if name == "sw2d_barrier" else 0.0
    h, v = u[..., :1], u[..., 1:] / u[..., :1]
    return torch.cat([GRAVITY * h - b / h - 0.5 * (v * v).sum(-1, keepdim=True), v], -1)


def _plain_start(name, u):
    lam = torch.zeros_like(u)
    lam[:, 0] = _ds_of(name, u[:, 0])
    return lam


def _project(vals, phiw):
    """(n, Q, S) -> moments (n, M, S)."""
    n, Q, S = vals.shape
    return (vals.transpose(1, 2).reshape(n * S, Q) @ phiw).reshape(n, S, -1).transpose(1, 2).contiguous()


def _at_points(lam, phi):
    n, M, S = lam.shape
    return (lam.transpose(1, 2).reshape(n * S, M) @ phi.T).reshape(n, S, -1).transpose(1, 2).contiguous()


def _solve(H, g):
    """H x = g for a batch of symmetric positive definite H (overwritten), scaled to a unit diagonal."""
    n = H.shape[-1]
    d = H.diagonal(dim1=1, dim2=2).rsqrt()
    H = H.mul_(d[:, :, None]).mul_(d[:, None, :])
    y = g * d
    for j in range(n - 1):
        col = H[:, j + 1:, j] / H[:, j, j, None]
        H[:, j + 1:, j + 1:] -= col[:, :, None] * H[:, j, None, j + 1:]
        y[:, j + 1:] -= col * y[:, j, None]
    for j in range(n - 1, -1, -1):
        y[:, j] /= H[:, j, j]
        y[:, :j] -= H[:, :j, j] * y[:, j, None]
    return y * d


def _newton(name, phi, phiw, u, lam, mask=None, chunk=8192):
    """Duals whose closure reproduces u, in place in lam; mask (n, M) of the moments a cell has."""
    Q, M = phi.shape
    S = u.shape[-1]
    pair = (phi[:, :, None] * phiw[:, None, :]).reshape(Q, M * M)
    eye = torch.eye(S * M, dtype=torch.float64, device=u.device)

    def points(l, c):  # (moments past a cell's order may hold what an earlier level left)
        return _at_points(l if mask is None else l * mask[c][..., None], phi)

    def gradient(l, c):
        g = _project(_u_of(name, points(l, c)), phiw) - u[c]
        return g if mask is None else g * mask[c][..., None]

    for c0 in range(0, u.shape[0], chunk):
        todo = torch.arange(c0, min(c0 + chunk, u.shape[0]), device=u.device)
        scale = u[todo].flatten(1).norm(dim=1)
        g = gradient(lam[todo], todo)
        last = torch.zeros(len(todo), dtype=torch.bool, device=u.device)  # its last step is still to come
        for _ in range(60):
            norm = g.flatten(1).norm(dim=1)
            near = norm < 1e-9 * scale
            keep = ~(near & last)
            if not bool(keep.any()):
                break
            todo, scale, g, norm, last = todo[keep], scale[keep], g[keep], norm[keep], near[keep]
            l = lam[todo]
            _, D = _u_of(name, points(l, todo), True)
            n = len(todo)
            H = (D.permute(0, 2, 3, 1).reshape(n * S * S, Q) @ pair).reshape(n, S, S, M, M)
            H = H.permute(0, 3, 1, 4, 2).reshape(n, M * S, M * S)
            H = 0.5 * (H + H.transpose(1, 2))
            if mask is not None:
                on = mask[todo].repeat_interleave(S, 1)
                H = H * on[:, :, None] * on[:, None, :] + eye * (1 - on)[:, :, None]
            step = _solve(H, g.reshape(n, -1)).reshape(n, M, S)
            size = torch.ones(n, 1, 1, dtype=torch.float64, device=u.device)
            for _ in range(40):
                new = gradient(l - size * step, todo)
                worse = ~(new.flatten(1).norm(dim=1) <= norm) & ~near[keep]
                if not bool(worse.any()):
                    break
                size = torch.where(worse[:, None, None], 0.5 * size, size)
            lam[todo] = l - size * step
            g = new
    return lam


def _wave_speed_and_flux(flow, U, n):
    """Per point: normal velocity scaled pieces of the 2D fluxes (unit-normal velocity left to the caller)."""
    if flow == "naca":
        rho, mx, my, E = U.unbind(-1)
        vx, vy = mx / rho, my / rho
        p = (GAMMA - 1) * (E - 0.5 * rho * (vx * vx + vy * vy))
        a = torch.sqrt(GAMMA * p / rho)
        F = torch.stack([mx * n[0] + my * n[1], (mx * vx + p) * n[0] + my * vx * n[1],
                         mx * vy * n[0] + (my * vy + p) * n[1], (E + p) * (vx * n[0] + vy * n[1])], -1)
    else:
        h, mx, my = U.unbind(-1)
        vx, vy = mx / h, my / h
        a = torch.sqrt(GRAVITY * h)
        p = 0.5 * GRAVITY * h * h
        F = torch.stack([mx * n[0] + my * n[1], (mx * vx + p) * n[0] + mx * vy * n[1],
                         mx * vy * n[0] + (my * vy + p) * n[1]], -1)
    return F, vx, vy, a


def _rates(flow, m, uq, xi):
    """Sum of the point fluxes of every cell's edges (and the friction), (n, Q, S); zero in Dirichlet cells."""
    n, Q, S = uq.shape
    total = torch.zeros_like(uq)
    padded = torch.cat([uq, torch.ones(1, Q, S, dtype=uq.dtype, device=uq.device)])
    if flow == "burgers":
        for e in range(2):
            nx = m["normal"][:, e, 0][:, None]
            a, b = uq[..., 0], padded[m["nbr"][:, e].long()][..., 0]
            beta = torch.maximum(a.abs(), b.abs())
            total[..., 0] += 0.25 * (a * a + b * b) * nx - 0.5 * beta * (b - a) * nx.abs()
    else:
        wall = m["bc"] == native.BC_NOSLIP
        bx, by = m["bnormal"][:, 0][:, None], m["bnormal"][:, 1][:, None]
        for e in range(m["nbr"].shape[1]):
            nb = m["nbr"][:, e].long()
            left, right = uq, padded[nb]
            if bool(wall.any()):
                ghost = (wall & (nb == n))[:, None, None]
                rho, vx, vy = uq[..., 0], uq[..., 1] / uq[..., 0], uq[..., 2] / uq[..., 0]
                vn = bx * vx + by * vy
                tx, ty = vx - vn * bx, vy - vn * by
                G = uq.clone()
                G[..., 1], G[..., 2] = rho * tx, rho * ty
                if S == 4:
                    G[..., 3] += 0.5 * rho * (tx * tx + ty * ty - vx * vx - vy * vy)
                left, right = torch.where(ghost, G, left), torch.where(ghost, G, right)
            nv = m["normal"][:, e]
            nu = m["unit_normal"][:, e]
            length = nv.norm(dim=1)[:, None]
            nrm = (nv[:, 0][:, None], nv[:, 1][:, None])
            ux, uy = nu[:, 0][:, None], nu[:, 1][:, None]
            Fl, vxl, vyl, al = _wave_speed_and_flux(flow, left, nrm)
            Fr, vxr, vyr, ar = _wave_speed_and_flux(flow, right, nrm)
            ul, ur = ux * vxl + uy * vyl, ux * vxr + uy * vyr
            if flow == "naca":
                sm = torch.maximum(ul.abs() + al, ur.abs() + ar)
                total += 0.5 * (Fl + Fr) - (0.5 * sm * length)[..., None] * (right - left)
            else:
                lo, hi = (ul - al)[..., None], (ur + ar)[..., None]
                mid = ((hi * Fl - lo * Fr) + hi * lo * (right - left) * length[..., None]) / (hi - lo)
                total += torch.where(lo >= 0, Fl, torch.where(hi <= 0, Fr, mid))
        if flow == "dambreak":
            sp = torch.sqrt(uq[..., 1] ** 2 + uq[..., 2] ** 2) / uq[..., 0]
            cf = 0.01 * (1.0 + xi[:, 2])[None, :]
            total[..., 1:] += (m["area"][:, None] * cf * sp / uq[..., 0])[..., None] * uq[..., 1:]
    return torch.where((m["bc"] == native.BC_DIRICHLET)[:, None, None], torch.zeros_like(total), total)


def _time_step(flow, cfl, m, uq):
    dx = m["dx_param"][:, None]
    if flow == "burgers":
        return float((cfl * dx / uq[..., 0].abs()).min())
    _, vx, vy, a = _wave_speed_and_flux(flow, uq, (0.0, 0.0))
    s = torch.maximum(torch.maximum((vy - a).abs(), (vy + a).abs()), torch.maximum((vx - a).abs(), (vx + a).abs()))
    return float((cfl / dx / s).min())


def _mesh_tensors(mesh):
    return {k: _dev(getattr(mesh, k)) for k in ("nbr", "unit_normal", "normal", "area", "dx_param", "bc", "bnormal")}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _waves(rng, x, y, count=6, most=6):
    """A smooth random field of (x, y), of size about one."""
    f = torch.zeros_like(x)
    for _ in range(count):
        kx, ky = rng.integers(1, most + 1), rng.integers(0, most + 1)
        f = f + rng.normal() / math.sqrt(count) * torch.cos(2 * math.pi * (kx * x + ky * y) + 2 * math.pi * rng.random())
    return f


def _flow_moments(case, seed, basis, mesh):
    """The moments a run starts from (or stands at): the flow of the configuration with a disturbance by the seed."""
    rng = np.random.default_rng(seed)
    phiw, xi = _dev(basis.phiw), _dev(basis.xi)
    if case["flow"] == "burgers":
        x0, sigma = 0.5 + 0.8 * rng.random(), 0.15 + 0.1 * rng.random()
        ic = workloads.burgers_step_ic(x0=x0, sigma=sigma)
        return _project(_dev(ic(mesh.center, basis.xi)), phiw)
    if case["flow"] == "naca":
        # free stream with uncertain angle and Mach number; the disturbance, and its own uncertainty, fall off from
        # the profile, so that the outer half of the cells is at rest in the stream as in a run
        ni, nj = case["ni"], case["nj"]
        fs = _dev(workloads.euler2d_freestream_ic()(mesh.center[:1], basis.xi)[0])
        j, i = torch.meshgrid(torch.arange(nj, device="cuda", dtype=torch.float64) / nj,
                              torch.arange(ni, device="cuda", dtype=torch.float64) / ni, indexing="ij")
        i, j = i.reshape(-1), j.reshape(-1)
        size = 0.05 * torch.exp(-(j / 0.12) ** 2)
        d = [size[:, None] * (_waves(rng, i, j)[:, None] + 0.4 * _waves(rng, i, j)[:, None] * xi[:, 0] +
                              0.4 * _waves(rng, i, j)[:, None] * xi[:, 1]) for _ in range(4)]
        rho, vx, vy = fs[:, 0], fs[:, 1] / fs[:, 0], fs[:, 2] / fs[:, 0]
        p = (GAMMA - 1) * (fs[:, 3] - 0.5 * rho * (vx * vx + vy * vy))
        a = torch.sqrt(GAMMA * p / rho)
        rho, p = rho * (1 + d[0]), p * (1 + d[3])
        vx, vy = vx + a * d[1], vy + a * d[2]
        return _project(torch.stack([rho, rho * vx, rho * vy, p / (GAMMA - 1) + 0.5 * rho * (vx * vx + vy * vy)], -1),
                        phiw)
    # dam break with a swell on a part of the water
    ic = workloads.sw2d_dambreak_ic(ratio=1.8 + 0.4 * rng.random(), dpos=0.08 + 0.04 * rng.random())
    vals = _dev(ic(mesh.center, basis.xi))
    x, y = _dev(mesh.center[:, 0]), _dev(mesh.center[:, 1])
    cx, cy = rng.uniform(-0.5, 0.5, 2)
    size = 0.05 * torch.exp(-((x - cx) ** 2 + (y - cy) ** 2) / 0.15 ** 2)
    h = vals[..., 0] * (1 + size[:, None] * (_waves(rng, x, y)[:, None] + 0.2 * xi[:, 2]))
    v = [torch.sqrt(GRAVITY * vals[..., 0]) * (size * _waves(rng, x, y))[:, None] for _ in range(2)]
    return _project(torch.stack([h, h * v[0], h * v[1]], -1), phiw)


def _cells_of_duals(name, seed, basis, n):
    """Cells of known duals: random states with a random higher part, damped where it would leave the realisable
    range; returns (duals, moments, plain start)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    S = native.STATES[KIND[name]]

    def uniform(lo, hi):
        return lo + (hi - lo) * torch.rand(n, device="cuda", dtype=torch.float64, generator=gen)

    if name == "euler1d":
        rho, v, p = uniform(0.5, 2), uniform(-1, 1), uniform(0.5, 2)
        cons = torch.stack([rho, rho * v, p / (GAMMA - 1) + 0.5 * rho * v * v], -1)
    elif name == "euler2d":
        rho, vx, vy, p = uniform(0.5, 2), uniform(-1, 1), uniform(-1, 1), uniform(0.5, 2)
        cons = torch.stack([rho, rho * vx, rho * vy, p / (GAMMA - 1) + 0.5 * rho * (vx * vx + vy * vy)], -1)
    else:
        h, vx, vy = uniform(1, 3), uniform(-1, 1), uniform(-1, 1)
        cons = torch.stack([h, h * vx, h * vy], -1)
    lam = torch.empty(n, basis.M, S, device="cuda", dtype=torch.float64).normal_(generator=gen)
    lam *= 0.05 if name == "euler1d" else 0.01
    lam[:, 0] = _ds_of(name, cons)
    phi, phiw = _dev(basis.phi), _dev(basis.phiw)
    for _ in range(12):
        L = _at_points(lam, phi)
        U = _u_of(name, L)
        w = -L[..., -1] if name.startswith("euler") else U[..., 0]
        bad = ~(w.amin(1) > w.amax(1) / 3) | ~(w.amin(1) > 0) | ~(U[..., 0].amin(1) > U[..., 0].amax(1) / 100)
        if not bool(bad.any()):
            break
        lam[:, 1:] = torch.where(bad[:, None, None], 0.5 * lam[:, 1:], lam[:, 1:])
    u = _project(_u_of(name, _at_points(lam, phi)), phiw)
    return lam, u, _plain_start(name, u)


def _orders(case, seed, basis, n):
    """Per-cell moment counts a run starts with, or None."""
    if case.get("orders") == "levels":
        return np.full(n, basis.ntotal_per_level[-1], np.int32)
    if case.get("orders") == "mixed":
        return np.asarray(basis.ntotal_per_level, np.int32)[workloads.cell_orders(n, seed, case["degree"]) - 1]
    return None


def _network(case, seed, basis, cl):
    """A network with the weights and normalisation of the seed."""
    net = native.WarmStartNet(cl, hidden=case["hidden"], seed=seed % 1000 + 1)
    k, o = net.dims[0], net.dims[-1]
    net.set_params(None, np.concatenate([np.zeros(k), np.ones(k), np.zeros(o), np.full(o, 0.01)]).astype(np.float32))
    return net


def prepare(case, seed):
    basis = _basis(case)
    name, path = _closure_name(case), case["path"]
    cl = _handle(case, basis)
    s = {"path": path, "cl": cl}
    if path in ("host", "closure", "predict"):
        n = case["cells"]
        _, u, lam0 = _cells_of_duals(name, seed, basis, n)
        if path == "host":
            s.update(u=u.cpu().numpy(), lam0=lam0.cpu().numpy())
        elif path == "closure":
            s.update(u=u, lam0=lam0, lam=torch.empty_like(u), status=torch.zeros(n, dtype=torch.int32, device="cuda"))
        else:
            s.update(u=u, lam=torch.empty_like(u), net=_network(case, seed, basis, cl))
    elif path == "grad":
        gen = torch.Generator(device="cuda").manual_seed(seed)
        net = _network(case, seed, basis, cl)
        real = cl.S * basis.M
        x, t = (torch.zeros(case["rows"], w, device="cuda") for w in (net.dims[0], net.dims[-1]))
        for a in (x, t):
            a[:, :real] = torch.randn(case["rows"], real, device="cuda", generator=gen)
        s.update(net=net, x=x, t=t, real=real, grad=torch.empty(net.n_params, device="cuda"))
    else:
        mesh = _mesh(case)
        n = mesh.n_cells
        u0 = _flow_moments(case, seed, basis, mesh)
        lam0 = _plain_start(name, u0)
        s.update(prob=_problem(case), mesh=native.DeviceMesh(mesh), u=torch.empty_like(u0),
                 uq=torch.empty(n, basis.Q, cl.S, dtype=torch.float64, device="cuda"))
        if path == "sweeps":
            # duals of a flow under way: the mean's, with a higher part of its moments' size
            ratio = u0[:, 1:] / u0.abs().amax(dim=(0, 1))
            lam0[:, 1:] = 0.1 * ratio * lam0[:, :1].abs()
            s.update(lam=lam0, unew=torch.zeros_like(u0),
                     mv=torch.empty(n, 2 * cl.S, dtype=torch.float64, device="cuda"))
        else:
            s.update(u0=u0, lam0=lam0, lam=torch.empty_like(u0), scratch=torch.empty_like(u0),
                     status=torch.zeros(n, dtype=torch.int32, device="cuda"), steps=case["steps"], nt=None)
            nt0 = _orders(case, seed, basis, n)
            if nt0 is not None:
                s.update(nt0=_dev(nt0), nt=_dev(nt0))
            if case["orders"] == "levels":
                cl.set_refinement(basis.ntotal_per_level, 2e-3, 4e-4)
    return s


def run(s):
    cl, path = s["cl"], s["path"]
    if path == "host":
        lam = s["lam0"].copy()
        status, _ = cl.solve_host(s["u"], lam)
        return {"lam": lam, "status": status}
    if path == "closure":
        s["lam"].copy_(s["lam0"])
        failed = cl.solve(s["u"], s["lam"], s["status"])
        return {"lam": s["lam"], "status": s["status"], "failed": failed}
    if path == "loop":
        s["u"].copy_(s["u0"])
        s["lam"].copy_(s["lam0"])
        if s["nt"] is not None:
            s["nt"].copy_(s["nt0"])
        cl.invalidate_factors()  # a new run: the kept factorisations belong to the old duals
        r = cl.run_steps(s["prob"], s["mesh"], s["u"], s["lam"], s["uq"], s["scratch"], s["status"], nt_cell=s["nt"],
                         max_steps=s["steps"])
        out = {"u": s["u"], "lam": s["lam"], "status": s["status"], "t": r["t"], "residual": r["residual"],
               "steps": r["steps"], "failed": r["nfail"]}
        if s["nt"] is not None:
            out["nt"] = s["nt"]
        return out
    if path == "sweeps":
        cl.eval_uq(s["lam"], s["uq"])
        cl.reconstruct(s["uq"], s["u"])
        dt = cl.compute_dt(s["prob"], s["mesh"], s["uq"])
        cl.advance(s["prob"], s["mesh"], dt, s["u"], s["uq"], s["unew"])
        cl.mean_var(s["lam"], s["mv"])
        return {"uq": s["uq"], "u": s["u"], "dt": dt, "unew": s["unew"], "mean_var": s["mv"]}
    lib, p = native.lib(), native._p
    if path == "predict":
        if lib.uqk_mlp_predict(s["net"].h, s["u"].shape[0], p(s["u"]), p(s["lam"])) != 0:
            raise RuntimeError(cl.error())
        return {"lam": s["lam"]}
    loss = native.C.c_double()
    if lib.uqk_mlp_loss_grad(s["net"].h, s["x"].shape[0], p(s["x"]), p(s["t"]), s["real"], native.C.byref(loss),
                             p(s["grad"])) != 0:
        raise RuntimeError(cl.error())
    return {"loss": loss.value, "grad": s["grad"]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
# Newton steps of a cell from the plain start (damped: alpha = 1/2 contracts by a half) and in a time step
_COLD_STEPS = {"euler1d": 36.0, "euler2d": 4.0, "sw2d": 4.0, "sw2d_barrier": 4.0, "burgers": 5.0}
_LOOP_STEPS = {"burgers": 0.5, "naca": 0.7, "dambreak": 0.25}


def work(case):
    basis = _basis(case)
    S, M, Q = native.STATES[KIND[_closure_name(case)]], basis.M, basis.Q
    if case.get("orders") == "mixed":
        M = float(np.mean(basis.ntotal_per_level))
    n = S * M
    gradient = 4.0 * Q * S * M
    newton = Q * n * (n + 1) + n ** 3 / 3 + 2 * n * n + gradient
    path = case["path"]
    if path in ("host", "closure"):
        cells = case["cells"]
        return {"bytes": cells * (24.0 * n + 4), "flops": cells * (gradient + _COLD_STEPS[case["closure"]] * newton)}
    if path in ("predict", "grad"):
        k, h = (S * M + 31) // 32 * 32, case["hidden"]
        weights = 2 * k * h + 3 * h * h
        if path == "predict":
            return {"bytes": case["cells"] * 16.0 * n + 2.0 * weights, "flops": 2.0 * case["cells"] * weights}
        return {"bytes": case["rows"] * 8.0 * k + 8.0 * weights, "flops": 6.0 * case["rows"] * weights}
    cells, edges, dim = _n_cells(case), 2 if case["flow"] == "burgers" else 4, 1 if case["flow"] == "burgers" else 2
    geometry = 4.0 * edges + 16.0 * edges * dim + 12 + 8 * dim
    flux = 30.0 * edges * S * Q + 2.0 * Q * S * M
    if path == "sweeps":
        return {"bytes": cells * (8.0 * (n + Q * S + n + n + 2 * S) + geometry), "flops": cells * (2 * gradient + flux)}
    per_step = gradient + _LOOP_STEPS[case["flow"]] * newton + flux
    return {"bytes": case["steps"] * cells * (32.0 * n + 8.0 * Q * S + geometry),
            "flops": case["steps"] * cells * per_step}


# ---------------------------------------------------------------------------
# the same outputs in plain 64-bit torch
# ---------------------------------------------------------------------------
def _exact_loop(case, seed):
    basis, name, flow = _basis(case), _closure_name(case), case["flow"]
    if _n_cells(case) * case["steps"] * (basis.M * native.STATES[KIND[name]]) ** 2 > 1e10:
        return None  # the plain Newton would take too long
    mesh = _mesh(case)
    m = _mesh_tensors(mesh)
    phi, phiw, xi = _dev(basis.phi), _dev(basis.phiw), _dev(basis.xi)
    u = _flow_moments(case, seed, basis, mesh)
    lam = _plain_start(name, u)
    cfl = {"burgers": 0.5, "naca": 0.4, "dambreak": 0.45}[flow]
    nt = _orders(case, seed, basis, mesh.n_cells)
    nt = None if nt is None else _dev(nt)
    levels = _dev(np.asarray(basis.ntotal_per_level, np.int64))
    index = torch.arange(basis.M, device="cuda")

    def mask_of(counts):
        return None if counts is None else (index[None, :] < counts[:, None]).to(torch.float64)

    t, residual = 0.0, 0.0
    for _ in range(case["steps"]):
        mask = mask_of(nt)
        _newton(name, phi, phiw, u, lam, mask)
        uq = _u_of(name, _at_points(lam if mask is None else lam * mask[..., None], phi))
        if case["orders"] == "levels":
            lev = torch.searchsorted(levels, nt.long())
            low = torch.where(lev == 0, torch.ones_like(lev), levels[(lev - 1).clamp(min=0)])
            added = (index[None, :] >= low[:, None]) & (index[None, :] < nt[:, None])
            size = (u[..., 0].abs() * added).sum(1)
            lev = torch.where((size > 2e-3) & (lev < len(levels) - 1), lev + 1,
                              torch.where((size < 4e-4) & (lev > 0), lev - 1, lev))
            nt = levels[lev].to(torch.int32)
            mask = mask_of(nt)
        rec = _project(uq, phiw)
        rate = _project(_rates(flow, m, uq, xi), phiw)
        if mask is not None:
            rec, rate = rec * mask[..., None], rate * mask[..., None]
        dt = _time_step(flow, cfl, m, uq)
        new = rec - (dt / m["area"])[:, None, None] * rate
        residual = float(((new - u)[:, 0, 0].abs() * m["area"]).sum())
        t += dt
        u = new
    out = {"u": u, "lam": lam, "status": None, "t": t, "residual": residual, "steps": None, "failed": None}
    return out


def _gelu(z):
    return 0.5 * z * (1 + torch.tanh(0.7978845608028654 * (z + 0.044715 * z ** 3)))


def _layers(case, net):
    """The network's 64-bit weights (the BF16 values that its products use) and biases."""
    p, _ = net.get_params()
    p, at, out = torch.as_tensor(p, device="cuda"), 0, []
    for k, o in zip(net.dims[:-1], net.dims[1:]):
        W = p[at:at + k * o].reshape(o, k).bfloat16().double()
        out.append((W, p[at + k * o:at + k * o + o].double()))
        at += k * o + o
    return out


def exact(case, seed):
    path = case["path"]
    if path == "loop":
        return _exact_loop(case, seed)
    basis, name = _basis(case), _closure_name(case)
    phi, phiw, xi = _dev(basis.phi), _dev(basis.phiw), _dev(basis.xi)
    if path in ("host", "closure"):
        lam, _, _ = _cells_of_duals(name, seed, basis, case["cells"])
        return {"lam": lam, "status": None, "failed": None}
    if path == "sweeps":
        mesh = _mesh(case)
        m = _mesh_tensors(mesh)
        s = prepare(case, seed)
        uq = _u_of(name, _at_points(s["lam"], phi))
        u = _project(uq, phiw)
        dt = _time_step(case["flow"], 0.4 if case["flow"] == "naca" else 0.45, m, uq)
        unew = u - (dt / m["area"])[:, None, None] * _project(_rates(case["flow"], m, uq, xi), phiw)
        mean = _project(uq, phiw[:, :1])[:, 0]
        var = _project((uq - mean[:, None]) ** 2, phiw[:, :1])[:, 0]
        return {"uq": uq, "u": u, "dt": dt, "unew": unew, "mean_var": torch.cat([mean, var], 1)}
    s = prepare(case, seed)
    layers = _layers(case, s["net"])
    S, M = s["cl"].S, basis.M
    if path == "predict":
        u = s["u"]
        u0 = u[:, 0]
        if name.startswith("euler"):
            rho = u0[:, 0]
            T = (GAMMA - 1) * (u0[:, -1] - 0.5 * (u0[:, 1:-1] ** 2).sum(-1) / rho) / rho
            D = torch.stack([rho] + [rho * torch.sqrt(T)] * (S - 2) + [rho * T], -1)
            scale = D / rho[:, None]
        else:
            a = torch.sqrt(GRAVITY * u0[:, 0])
            D = torch.stack([u0[:, 0], u0[:, 0] * a, u0[:, 0] * a], -1)
            scale = torch.stack([1 / a ** 2, 1 / a, 1 / a], -1)
        h = torch.zeros(len(u), s["net"].dims[0], dtype=torch.float64, device="cuda")
        h[:, :S * M] = (u / D[:, None]).reshape(len(u), -1)
        for i, (W, b) in enumerate(layers):
            h = h @ W.T + b
            h = _gelu(h) if i + 1 < len(layers) else h
        ds = _ds_of(name, u0)
        _, DU = _u_of(name, ds, True)
        lin = torch.linalg.solve(DU, u.transpose(1, 2)).transpose(1, 2).contiguous()
        lin[:, 0] = ds
        return {"lam": lin + 0.01 * h[:, :S * M].reshape(len(u), M, S) / scale[:, None]}
    flat = []
    for W, b in layers:
        W.requires_grad_(True)
        b.requires_grad_(True)
        flat += [W, b]
    h = s["x"].double()
    for i, (W, b) in enumerate(layers):
        h = h @ W.T + b
        h = _gelu(h) if i + 1 < len(layers) else h
    real = s["real"]
    loss = ((h[:, :real] - s["t"].double()[:, :real]) ** 2).mean()
    g = torch.autograd.grad(loss, flat)
    return {"loss": float(loss.detach()), "grad": torch.cat([x.reshape(-1) for x in g])}
