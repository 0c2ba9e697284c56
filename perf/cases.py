"""Workloads that stand for what programs do with this framework.

Every case is one pass of a program through the public entry points of
``ddc_amd``: builders, evaluators and their adjoints, on device tensors and
plans that the program keeps between calls.  ``listed()`` names twelve cases
between the smallest calls and the largest; ``draw`` takes another one of the
same ranges.  ``exact`` restates the spline mathematics with dense collocation
matrices and the Cox-de Boor recursion in plain 64-bit torch and numpy.

Meshes: "uniform"; "jitter" (break points within 0.3 of a cell of the uniform
ones); "random" (sorted uniform-random break points); "stretched" (cells that
grow by 5 % from the left end).
"""
import math

import numpy as np
import torch

import ddc_amd as D
from ddc_amd.autograd import interpolate

P, G, H = D.SplineBuilderClosure.PERIODIC, D.SplineBuilderClosure.GREVILLE, D.SplineBuilderClosure.HERMITE


def listed():
    return [
        # A 1D step of a small kinetic grid: 32 cells and 1000 lines, the
        # smallest grid that the reference's spline benchmark sweeps; its time
        # is launches and host calls.
        {"name": "line_32", "family": "line", "cells": 32, "lines": 1000, "degree": 3, "mesh": "uniform",
         "layout": "batch", "points": 32},
        # The middle of that sweep: non-uniform periodic, even degree, sizes
        # that are no multiple of any tile.
        {"name": "line_nonuniform", "family": "line", "cells": 501, "lines": 1000, "degree": 4, "mesh": "jitter",
         "layout": "batch", "points": 501},
        # 1000 x 1000 with the interpolation dimension contiguous: a program
        # that keeps its lines as rows.
        {"name": "line_rows", "family": "line", "cells": 1000, "lines": 1000, "degree": 3, "mesh": "uniform",
         "layout": "interp", "points": 1000},
        # The headline: 512 MiB of values, 2^26 evaluation points.
        {"name": "line_large", "family": "line", "cells": 1024, "lines": 65536, "degree": 3, "mesh": "uniform",
         "layout": "batch", "points": 1024},
        # One semi-Lagrangian advection step on 512 x 512 as one call, the
        # feet computed from one shift per line.
        {"name": "advect_512", "family": "advect", "cells": 512, "lines": 512, "degree": 3},
        # The same step differentiated: forward through torch.autograd, then
        # the gradients of the values and of the feet.
        {"name": "gradient_512", "family": "gradient", "cells": 512, "lines": 512, "degree": 3},
        # A bounded domain on a random mesh: build, values and first
        # derivatives (a field solve needs both).
        {"name": "greville_deriv", "family": "greville", "cells": 1024, "lines": 65536, "degree": 3, "mesh": "random",
         "layout": "batch", "points": 1024},
        # Both adjoints at scale: the backward pass of a large batch, quintic.
        {"name": "adjoint_large", "family": "adjoint", "cells": 1024, "lines": 65536, "degree": 5, "mesh": "uniform",
         "layout": "batch", "points": 1024},
        # Long lines with prescribed end derivatives on a stretched mesh (a
        # boundary layer), quintic, build only.
        {"name": "hermite_2048", "family": "hermite", "cells": 2048, "lines": 32768, "degree": 5},
        # Tensor-product 2D with scattered points (particles): build, values
        # and the full adjoint, non-uniform x periodic.
        {"name": "tensor_2d", "family": "tensor2d", "cells1": 1024, "cells2": 1024, "batch": 16, "points": 1 << 22},
        # A 2D semi-Lagrangian step: one foot per grid point, close to it.
        {"name": "advect_2d", "family": "advect2d", "cells1": 512, "cells2": 512, "batch": 8, "degree": 3},
        # Tensor-product 3D: build, values and the mixed derivative at
        # scattered points, and the integral.
        {"name": "tensor_3d", "family": "tensor3d", "cells": 128, "batch": 4, "points": 1 << 22},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["line", "line", "line", "advect", "gradient", "greville", "adjoint", "hermite", "tensor2d",
                         "advect2d", "tensor3d"])
    c = {"family": family}
    if family in ("line", "greville", "adjoint"):
        c["cells"] = _log_int(rng, 32, 1024)
        c["lines"] = _log_int(rng, 1000, min(100000, (1024 * 65536) // c["cells"]))
        c["mesh"] = "random" if family == "greville" else rng.choice(["uniform", "uniform", "jitter"])
        c["degree"] = rng.choice([3, 3, 5] if family == "greville" else [3, 3, 4, 5])
        c["layout"] = rng.choice(["batch", "batch", "interp"])
        c["points"] = c["cells"]
    elif family == "advect":
        c.update(cells=_log_int(rng, 300, 1024), lines=_log_int(rng, 256, 16384), degree=rng.choice([3, 3, 4, 5]))
    elif family == "gradient":
        c.update(cells=_log_int(rng, 64, 1024), lines=_log_int(rng, 64, 4096), degree=rng.choice([3, 3, 4, 5]))
    elif family == "hermite":
        c.update(cells=_log_int(rng, 256, 2048), lines=_log_int(rng, 1000, 32768), degree=rng.choice([3, 5]))
    elif family == "tensor2d":
        c.update(cells1=_log_int(rng, 100, 1024), cells2=_log_int(rng, 100, 1024), batch=rng.randint(1, 16),
                 points=_log_int(rng, 1 << 16, 1 << 22))
    elif family == "advect2d":
        c.update(cells1=_log_int(rng, 100, 1024), cells2=_log_int(rng, 100, 1024), batch=rng.randint(1, 8),
                 degree=rng.choice([3, 3, 5]))
    else:
        c.update(cells=_log_int(rng, 32, 128), batch=rng.randint(1, 4), points=_log_int(rng, 1 << 16, 1 << 22))
    return c


# ---- plans and inputs


def _breaks(mesh, n):
    rng = np.random.default_rng(0xDDC0 + n)
    x = np.linspace(0.0, 1.0, n + 1)
    if mesh == "jitter":
        x[1:-1] += rng.uniform(-0.3, 0.3, n - 1) / n
    elif mesh == "random":
        x[1:-1] = np.sort(rng.uniform(0.0, 1.0, n - 1))
    elif mesh == "stretched":
        x = (1.05 ** np.arange(n + 1, dtype=np.float64) - 1.0) / (1.05 ** n - 1.0)
    return x


def _basis(mesh, n, degree, periodic):
    if mesh == "uniform":
        return D.UniformBSplines(degree, 0.0, 1.0, n, periodic=periodic)
    return D.NonUniformBSplines(degree, _breaks(mesh, n), periodic=periodic)


def _rand(shape, gen):
    return torch.rand(shape, dtype=torch.float64, device="cuda", generator=gen)


def _randn(shape, gen):
    return torch.randn(shape, dtype=torch.float64, device="cuda", generator=gen)


def _line_values(m, lines, axis, gen):
    """sin(2 pi k_y x) + 0.1 N(0, 1) with k_y in 1..8, one line per y."""
    x = torch.arange(m, dtype=torch.float64, device="cuda") / m
    k = torch.randint(1, 9, (lines,), device="cuda", generator=gen).to(torch.float64)
    phase = x[:, None] * k[None, :] if axis == 0 else k[:, None] * x[None, :]
    return torch.sin(2 * math.pi * phase) + 0.1 * _randn(phase.shape, gen)


def _line_shape(case):
    """(rows, axis) to shape: lines are columns ("batch") or rows ("interp")."""
    axis = 0 if case.get("layout", "batch") == "batch" else 1
    lines = case["lines"]
    return axis, (lambda rows: (rows, lines) if axis == 0 else (lines, rows))


def _closure(case):
    return {"greville": (False, G), "hermite": (False, H)}.get(case["family"], (True, P))


def _mesh(case):
    return "stretched" if case["family"] == "hermite" else case.get("mesh", "uniform")


def _inputs(case, seed):
    """The arrays of one pass, from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    family = case["family"]
    s = {}
    if family == "tensor2d":
        n1, n2 = case["cells1"] + 3, case["cells2"]
        s["vals"] = _randn((case["batch"], n1, n2), gen)
        s["coords"] = _rand((case["batch"], case["points"], 2), gen)
        s["w"] = _randn((case["batch"], case["points"]), gen)
    elif family == "advect2d":
        nb, n1, n2 = case["batch"], case["cells1"], case["cells2"]
        off = 0.0 if case["degree"] % 2 else 0.5
        x = (torch.arange(n1, dtype=torch.float64, device="cuda") + off) / n1
        y = (torch.arange(n2, dtype=torch.float64, device="cuda") + off) / n2
        a = 0.01 + 0.02 * _rand((nb, 1, 1), gen)  # each entry's rotation, about a cell or more at the edge
        s["vals"] = torch.sin(2 * math.pi * x)[None, :, None] * torch.cos(2 * math.pi * y)[None, None, :] \
            + 0.1 * _randn((nb, n1, n2), gen)
        fx = x[None, :, None] + a * (y[None, None, :] - 0.5)
        fy = y[None, None, :] - a * (x[None, :, None] - 0.5)
        s["coords"] = torch.stack([fx.expand(nb, n1, n2), fy.expand(nb, n1, n2)], dim=-1).reshape(nb, n1 * n2, 2)
        s["coords"] = s["coords"].contiguous()
    elif family == "tensor3d":
        n, nb = case["cells"], case["batch"]
        s["vals"] = _randn((nb, n + 3, n, n + 3), gen)
        s["coords"] = _rand((nb, case["points"], 3), gen)
    else:
        periodic, closure = _closure(case)
        axis, shape = _line_shape(case)
        n, d = case["cells"], case["degree"]
        m = n if periodic else n + 1 if closure == H else n + d
        s["vals"] = _line_values(m, case["lines"], axis, gen)
        if family == "advect":
            y = torch.arange(case["lines"], dtype=torch.float64, device="cuda") / case["lines"]
            s["shift"] = 0.01 * torch.sin(2 * math.pi * (y + _rand((1,), gen)))
        elif family == "gradient":
            off = 0.0 if d % 2 else 0.5
            x = (torch.arange(n, dtype=torch.float64, device="cuda") + off) / n
            y = torch.arange(case["lines"], dtype=torch.float64, device="cuda") / case["lines"]
            s["coords"] = x[:, None] - 0.01 * torch.sin(2 * math.pi * (y + _rand((1,), gen)))[None, :]
            s["w"] = _randn(shape(n), gen)
        elif family == "hermite":
            s["dmin"], s["dmax"] = _randn(shape(d // 2), gen), _randn(shape(d // 2), gen)
        else:
            s["coords"] = _rand(shape(case["points"]), gen)
        if family == "adjoint":
            s["coef"] = _randn(shape(n + d), gen)
            s["w"] = _randn(shape(case["points"]), gen)
            del s["vals"]
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    family = case["family"]
    s["family"] = family
    per, null = D.PeriodicExtrapolationRule(), D.NullExtrapolationRule()

    def new(*shape):
        return torch.empty(shape, dtype=torch.float64, device="cuda")

    if family == "tensor2d":
        n1, n2, nb, pts = case["cells1"], case["cells2"], case["batch"], case["points"]
        b1, b2 = _basis("random", n1, 3, False), _basis("uniform", n2, 3, True)
        s["builder"] = D.SplineBuilder2D(D.SplineBuilder(b1, G, G), D.SplineBuilder(b2))
        s["eval"] = D.SplineEvaluator2D(D.SplineEvaluator(b1, null, null), D.SplineEvaluator(b2, per, per))
        s.update(coef=new(nb, n1 + 3, n2 + 3), out=new(nb, pts), gx=new(nb, pts, 2), gcoef=new(nb, n1 + 3, n2 + 3),
                 gvals=new(nb, n1 + 3, n2))
    elif family == "advect2d":
        n1, n2, nb, d = case["cells1"], case["cells2"], case["batch"], case["degree"]
        b1, b2 = _basis("uniform", n1, d, True), _basis("uniform", n2, d, True)
        s["builder"] = D.SplineBuilder2D(D.SplineBuilder(b1), D.SplineBuilder(b2))
        s["eval"] = D.SplineEvaluator2D(D.SplineEvaluator(b1, per, per), D.SplineEvaluator(b2, per, per))
        s.update(coef=new(nb, n1 + d, n2 + d), out=new(nb, n1 * n2))
    elif family == "tensor3d":
        n, nb = case["cells"], case["batch"]
        bs = [_basis("random", n, 3, False), _basis("uniform", n, 3, True), _basis("uniform", n, 3, False)]
        s["builder"] = D.SplineBuilder3D(D.SplineBuilder(bs[0], G, G), D.SplineBuilder(bs[1]),
                                         D.SplineBuilder(bs[2], G, G))
        s["eval"] = D.SplineEvaluator3D(D.SplineEvaluator(bs[0], null, null), D.SplineEvaluator(bs[1], per, per),
                                        D.SplineEvaluator(bs[2], null, null))
        s.update(coef=new(nb, n + 3, n + 3, n + 3), out=new(nb, case["points"]), dout=new(nb, case["points"]),
                 integral=new(nb))
    else:
        periodic, closure = _closure(case)
        s["axis"], shape = _line_shape(case)
        n, d = case["cells"], case["degree"]
        bs = _basis(_mesh(case), n, d, periodic)
        s["builder"] = D.SplineBuilder(bs, closure, closure)
        s["eval"] = D.SplineEvaluator(bs, per, per) if periodic else D.SplineEvaluator(bs, null, null)
        if family == "gradient":
            s["vals"].requires_grad_(True)
            s["coords"].requires_grad_(True)
        elif family == "adjoint":
            s.update(gx=new(*shape(case["points"])), gcoef=new(*shape(n + d)), gvals=new(*shape(n)))
        elif family == "advect":
            s["out"] = new(*shape(n))
        else:
            s["coef"] = new(*shape(n + d))
            if family != "hermite":
                s["out"] = new(*shape(case["points"]))
            if family == "greville":
                s["dout"] = new(*shape(case["points"]))
    return s


def run(s):
    family, builder, ev = s["family"], s["builder"], s["eval"]
    if family == "line":
        builder(s["coef"], s["vals"], axis=s["axis"])
        ev(s["out"], s["coords"], s["coef"], axis=s["axis"])
        return {"coef": s["coef"], "out": s["out"]}
    if family == "advect":
        D.advect(builder, ev, s["out"], s["vals"], s["shift"])
        return {"out": s["out"]}
    if family == "gradient":
        out = interpolate(builder, ev, s["vals"], s["coords"])
        gvals, gx = torch.autograd.grad(out, [s["vals"], s["coords"]], s["w"])
        return {"out": out.detach(), "gvals": gvals, "gx": gx}
    if family == "greville":
        builder(s["coef"], s["vals"], axis=s["axis"])
        ev(s["out"], s["coords"], s["coef"], axis=s["axis"])
        ev.deriv(1, s["dout"], s["coords"], s["coef"], axis=s["axis"])
        return {"coef": s["coef"], "out": s["out"], "dout": s["dout"]}
    if family == "adjoint":
        ev.eval_vjp(s["coords"], s["w"], s["coef"], s["gx"], s["gcoef"], axis=s["axis"])
        builder.build_vjp(s["gcoef"], s["gvals"], axis=s["axis"])
        return {"gx": s["gx"], "gcoef": s["gcoef"], "gvals": s["gvals"]}
    if family == "hermite":
        builder(s["coef"], s["vals"], s["dmin"], s["dmax"])
        return {"coef": s["coef"]}
    if family == "tensor2d":
        builder(s["coef"], s["vals"])
        ev(s["out"], s["coords"], s["coef"])
        ev.eval_vjp(s["coords"], s["w"], s["coef"], s["gx"], s["gcoef"])
        builder.build_vjp(s["gcoef"], s["gvals"])
        return {"coef": s["coef"], "out": s["out"], "gx": s["gx"], "gcoef": s["gcoef"], "gvals": s["gvals"]}
    if family == "advect2d":
        builder(s["coef"], s["vals"])
        ev(s["out"], s["coords"], s["coef"])
        return {"coef": s["coef"], "out": s["out"]}
    builder(s["coef"], s["vals"])
    ev(s["out"], s["coords"], s["coef"])
    ev.deriv((1, 1, 1), s["dout"], s["coords"], s["coef"])
    ev.integrate(s["integral"], s["coef"])
    return {"coef": s["coef"], "out": s["out"], "dout": s["dout"], "integral": s["integral"]}


def work(case):
    """Each input read once and each output written once.  A solved row costs
    about 4 d multiply-adds (two banded sweeps), a 1D basis about 3 d (d + 1)
    operations."""
    family = case["family"]
    if family == "tensor2d":
        n1, n2, nb, pts = case["cells1"] + 3, case["cells2"], case["batch"], case["points"]
        vals, coef, np_ = nb * n1 * n2, nb * n1 * (n2 + 3), nb * pts
        # vals, coords, w in; coef, out, gx, gcoef, gvals out
        return {"bytes": 8 * (2 * vals + 2 * coef + np_ * (2 + 1 + 1 + 2)),
                "flops": 2 * 2 * 24 * vals + np_ * (2 * 2 * 36 + 2 * 16 + 4 * 2 * 16)}
    if family == "advect2d":
        d, nb = case["degree"], case["batch"]
        vals = nb * case["cells1"] * case["cells2"]
        coef = nb * (case["cells1"] + d) * (case["cells2"] + d)
        return {"bytes": 8 * (vals + coef + 3 * vals),
                "flops": vals * (2 * 8 * d + 2 * 3 * d * (d + 1) + 2 * (d + 1) ** 2)}
    if family == "tensor3d":
        n, nb = case["cells"], case["batch"]
        vals, coef, np_ = nb * (n + 3) * n * (n + 3), nb * (n + 3) ** 3, nb * case["points"]
        return {"bytes": 8 * (vals + coef + np_ * (3 + 1 + 1) + nb),
                "flops": 3 * 24 * vals + np_ * 2 * (3 * 36 + 2 * 84) + 2 * coef}
    n, d, lines = case["cells"], case["degree"], case["lines"]
    solve, basis = 8 * d * n * lines, 3 * d * (d + 1) + 2 * (d + 1)
    if family == "hermite":
        return {"bytes": 8 * lines * (n + 1 + 2 * (d // 2) + n + d), "flops": solve}
    if family == "advect":
        return {"bytes": 8 * lines * (2 * n + 1), "flops": solve + basis * n * lines}
    if family == "gradient":  # vals, coords, w in; out, gvals, gx out
        return {"bytes": 8 * 6 * n * lines, "flops": 2 * solve + 4 * basis * n * lines}
    p = case["points"] * lines
    if family == "adjoint":  # coords, w, coef in; gx, gcoef, gvals out
        return {"bytes": 8 * (3 * p + 2 * (n + d) * lines + n * lines), "flops": solve + 3 * basis * p}
    m = n + d if family == "greville" else n
    outs = 2 if family == "greville" else 1
    return {"bytes": 8 * ((m + n + d) * lines + (1 + outs) * p), "flops": solve + outs * basis * p}


# ---- the same results in plain 64-bit torch and numpy


class _Exact1D:
    """A spline space and its interpolation problem with dense matrices."""

    def __init__(self, mesh, n, d, periodic, closure):
        self.n, self.d, self.periodic = n, d, periodic
        br = _breaks(mesh, n)
        if mesh == "uniform":
            knots = np.arange(-d, n + d + 1) / n
        elif periodic:
            knots = np.concatenate([br[n - d:n] - 1.0, br, br[1:d + 1] + 1.0])
        else:
            knots = np.concatenate([[br[0]] * d, br, [br[-1]] * d])
        if mesh == "uniform" and periodic:
            pts = (np.arange(n) + (0.0 if d % 2 else 0.5)) / n
        elif mesh == "uniform":  # odd degrees: averages of the clamped knots at the ends, break points inside
            ends = np.array([i * (i + 1) / (2.0 * d) for i in range(d // 2 + 1)]) / n
            pts = np.concatenate([ends, br[1:-1], 1.0 - ends[::-1]])
        else:
            nb = n if periodic else n + d
            pts = np.array([knots[i + 1:i + 1 + d].mean() for i in range(nb)])
            if periodic:
                pts = np.sort(np.where(pts < br[0], pts + 1.0, pts))
            elif closure == H:  # one point less for each end derivative
                pts = pts[d // 2:nb - d // 2]
        self.knots = torch.from_numpy(np.ascontiguousarray(knots)).cuda()
        self.points = torch.from_numpy(np.ascontiguousarray(pts)).cuda()
        nu = n if periodic else n + d
        lead = d // 2 if closure == H else 0  # derivative equations at each end
        a = np.zeros((len(pts) + 2 * lead, nu))
        cell, b = self.basis(self.points)
        self._put(a, lead, cell.cpu().numpy(), b.cpu().numpy())
        for i in range(lead):
            for row, x in ((i, br[:1]), (lead + len(pts) + i, br[-1:])):
                cell, b = self.basis(torch.from_numpy(x).cuda(), i + d % 2)
                self._put(a, row, cell.cpu().numpy(), b.cpu().numpy())
        self.scale = 1.0 / np.abs(a).max(1)  # derivative rows on a stretched mesh are huge
        a *= self.scale[:, None]
        self.a = torch.from_numpy(a).cuda()
        self.inv = torch.from_numpy(np.linalg.inv(a)).cuda()
        self.scale = torch.from_numpy(self.scale).cuda()

    def _put(self, a, row, cell, b):
        for j in range(self.d + 1):
            np.add.at(a, (row + np.arange(cell.size), (cell + j) % a.shape[1]), b[j])

    def basis(self, x, order=0):
        """The cell of each x and its d + 1 basis values or derivatives."""
        d, k = self.d, self.knots
        if self.periodic:
            x = x - torch.floor(x)
        cell = (torch.searchsorted(k[d:d + self.n + 1].contiguous(), x.contiguous(), right=True) - 1).clamp(0, self.n - 1)
        m = cell + d
        p = d - order
        vals = [torch.ones_like(x)]
        for q in range(1, p + 1):
            nxt = [torch.zeros_like(x) for _ in range(q + 1)]
            for r in range(q):
                lo, hi = k[m + r + 1 - q], k[m + r + 1]
                t = vals[r] / (hi - lo)
                nxt[r] += (hi - x) * t
                nxt[r + 1] += (x - lo) * t
            vals = nxt
        for q in range(p + 1, d + 1):  # one derivative per degree regained
            nxt = [torch.zeros_like(x) for _ in range(q + 1)]
            for r in range(q):  # the function of degree q - 1 that starts at knot m - q + 1 + r
                t = q * vals[r] / (k[m + r + 1] - k[m - q + 1 + r])
                nxt[r] -= t
                nxt[r + 1] += t
            vals = nxt
        return cell, torch.stack(vals)

    def solve(self, rhs, transpose=False):
        """rhs (equations, ...) to spline coefficients (n + d, ...), or the
        transposed problem on coefficient gradients (n + d, ...)."""
        shape = rhs.shape[1:]
        b = rhs.reshape(rhs.shape[0], -1)
        if transpose:
            if self.periodic:
                b = torch.cat([b[:self.d] + b[self.n:], b[self.d:self.n]])
            a, inv = self.a.T, self.inv.T
        else:
            b = b * self.scale[:, None]
            a, inv = self.a, self.inv
        x = inv @ b
        x += inv @ (b - a @ x)
        if transpose:
            x = x * self.scale[:, None]
        elif self.periodic:
            x = torch.cat([x, x[:self.d]])
        return x.reshape((x.shape[0],) + shape)

    def along(self, rhs, axis, transpose=False):
        return self.solve(rhs.movedim(axis, 0), transpose).movedim(0, axis).contiguous()

    def eval(self, x, coef, order=0):
        """x (points, lines), coef (n + d, lines)."""
        out = torch.empty_like(x)
        step = max(1, (1 << 24) // x.shape[1])
        for i in range(0, x.shape[0], step):
            cell, b = self.basis(x[i:i + step], order)
            out[i:i + step] = sum(b[j] * coef.gather(0, cell + j) for j in range(self.d + 1))
        return out

    def scatter(self, x, w, lines):
        g = torch.zeros((self.n + self.d, lines), dtype=torch.float64, device="cuda")
        step = max(1, (1 << 24) // x.shape[1])
        for i in range(0, x.shape[0], step):
            cell, b = self.basis(x[i:i + step])
            for j in range(self.d + 1):
                g.scatter_add_(0, cell + j, b[j] * w[i:i + step])
        return g


def _tensor_eval(spaces, coords, coef, orders):
    """coords (points, N), coef (size_1, ..., size_N) of one batch entry."""
    out = torch.empty(coords.shape[0], dtype=torch.float64, device="cuda")
    flat = coef.reshape(-1)
    for i in range(0, coords.shape[0], 1 << 22):
        part = [s.basis(coords[i:i + (1 << 22), k], o) for k, (s, o) in enumerate(zip(spaces, orders))]

        def level(k, index):
            cell, b = part[k]
            total = 0
            for j in range(spaces[k].d + 1):
                at = index * coef.shape[k] + (cell + j)
                total = total + b[j] * (flat[at] if k + 1 == len(part) else level(k + 1, at))
            return total

        out[i:i + (1 << 22)] = level(0, 0)
    return out


def exact(case, seed):
    s = _inputs(case, seed)
    family = case["family"]
    if family in ("tensor2d", "advect2d"):
        if family == "tensor2d":
            s1, s2 = _Exact1D("random", case["cells1"], 3, False, G), _Exact1D("uniform", case["cells2"], 3, True, P)
        else:
            s1, s2 = (_Exact1D("uniform", case[k], case["degree"], True, P) for k in ("cells1", "cells2"))
        coef = s2.along(s1.along(s["vals"], 1), 2)
        out = torch.stack([_tensor_eval((s1, s2), c, f, (0, 0)) for c, f in zip(s["coords"], coef)])
        if family == "advect2d":
            return {"coef": coef, "out": out}
        gx, gcoef = torch.empty_like(s["coords"]), torch.zeros_like(coef)
        for e in range(coef.shape[0]):
            c, w = s["coords"][e], s["w"][e]
            gx[e, :, 0] = w * _tensor_eval((s1, s2), c, coef[e], (1, 0))
            gx[e, :, 1] = w * _tensor_eval((s1, s2), c, coef[e], (0, 1))
            (c1, b1), (c2, b2) = s1.basis(c[:, 0]), s2.basis(c[:, 1])
            flat = gcoef[e].view(-1)
            for i in range(4):
                for j in range(4):
                    flat.index_add_(0, (c1 + i) * coef.shape[2] + c2 + j, w * b1[i] * b2[j])
        gvals = s1.along(s2.along(gcoef, 2, True), 1, True)
        return {"coef": coef, "out": out, "gx": gx, "gcoef": gcoef, "gvals": gvals}
    if family == "tensor3d":
        n = case["cells"]
        sp = (_Exact1D("random", n, 3, False, G), _Exact1D("uniform", n, 3, True, P), _Exact1D("uniform", n, 3, False, G))
        coef = s["vals"]
        for k in range(3):
            coef = sp[k].along(coef, k + 1)
        out = torch.stack([_tensor_eval(sp, c, f, (0, 0, 0)) for c, f in zip(s["coords"], coef)])
        dout = torch.stack([_tensor_eval(sp, c, f, (1, 1, 1)) for c, f in zip(s["coords"], coef)])
        # two Gauss points per cell integrate a cubic
        node = torch.tensor([0.5 - 0.5 / math.sqrt(3.0), 0.5 + 0.5 / math.sqrt(3.0)], dtype=torch.float64, device="cuda")
        integral = coef
        for e in sp:
            t = e.knots[e.d:e.d + e.n + 1]
            h = t[1:] - t[:-1]
            x = (t[:-1, None] + h[:, None] * node[None, :]).reshape(-1)
            cell, b = e.basis(x)
            weights = torch.zeros(e.n + e.d, dtype=torch.float64, device="cuda")
            for j in range(e.d + 1):
                weights.index_add_(0, cell + j, b[j] * (0.5 * h).repeat_interleave(2))
            integral = (integral * weights.view((1, -1) + (1,) * (integral.dim() - 2))).sum(1)
        return {"coef": coef, "out": out, "dout": dout, "integral": integral}
    periodic, closure = _closure(case)
    axis, _ = _line_shape(case)
    sp = _Exact1D(_mesh(case), case["cells"], case["degree"], periodic, closure)

    def col(t):
        return t.T if axis == 1 else t

    if family == "adjoint":
        x, w, coef = col(s["coords"]), col(s["w"]), col(s["coef"])
        g = sp.scatter(x, w, case["lines"])
        res = {"gx": w * sp.eval(x, coef, 1), "gcoef": g, "gvals": sp.solve(g, True)}
        return {k: col(v).contiguous() for k, v in res.items()}
    if family == "hermite":
        return {"coef": sp.solve(torch.cat([s["dmin"], s["vals"], s["dmax"]]))}
    coef = sp.solve(col(s["vals"]))
    if family == "advect":
        return {"out": sp.eval(sp.points[:, None] - s["shift"][None, :], coef)}
    x = col(s["coords"])
    if family == "gradient":
        g = sp.scatter(x, s["w"], case["lines"])
        return {"out": sp.eval(x, coef), "gvals": sp.solve(g, True), "gx": s["w"] * sp.eval(x, coef, 1)}
    res = {"coef": coef, "out": sp.eval(x, coef)}
    if family == "greville":
        res["dout"] = sp.eval(x, coef, 1)
    return {k: col(v).contiguous() for k, v in res.items()}
