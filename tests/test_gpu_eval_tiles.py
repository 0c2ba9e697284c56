"""Evaluators and their adjoint where a tile's points do not fill its threads,
where the divisor products of a non-uniform basis are out of range, at the knots
themselves, and at the sizes at which the adjoint changes kernel.  Tolerances as
in the other evaluator tests: 1e-13 for values and coordinate gradients, ten
times more per derivative, 1e-12 for coefficient gradients (sums in any order)."""
import numpy as np
import pytest

import oracle as O
from cases import G, P, breaks_for
from conftest import rel_err

pytestmark = pytest.mark.gpu


def _space(degree, cells, scale=1.0, mesh="random", seed=3):
    """A bounded non-uniform space (or uniform periodic) and its oracle."""
    import ddc_amd as D

    if mesh == "uniform":
        return (D.UniformBSplines(degree, 0.0, 1.0, cells, periodic=True),
                O.Spline(degree, True, P, P, ncells=cells, rmin=0.0, rmax=1.0))
    br = breaks_for(mesh, cells, seed=seed) * scale
    return D.NonUniformBSplines(degree, br), O.Spline(degree, False, G, G, breaks=br)


def _cus(cuda):
    import torch

    return torch.cuda.get_device_properties(cuda).multi_processor_count


def _some(nbatch):
    return np.unique(np.concatenate([[0, 1, nbatch - 2, nbatch - 1], np.random.default_rng(0).integers(0, nbatch, 30)]))


@pytest.mark.parametrize("degree,scale", [(1, 1.0), (3, 1.0), (5, 1.0), (6, 1.0), (3, 1e-60), (5, 1e-60), (7, 1e-40)])
@pytest.mark.parametrize("axis", [0, 1])
def test_few_points(degree, scale, axis, cuda):
    """Values (some outside) and two derivatives at 64, 65 and 200 points a line:
    narrow tiles, 16-line tiles and the streaming kernel."""
    import torch

    import ddc_amd as D

    cus = _cus(cuda)
    bs, orc = _space(degree, 120, scale)
    ev = D.SplineEvaluator(bs, D.ConstantExtrapolationRule(), D.NullExtrapolationRule())
    rng = np.random.default_rng(1)
    for nbatch in (9, 8 * cus + 13, 32 * cus + 16):
        some = _some(nbatch)
        coef = rng.standard_normal((orc.size, nbatch))
        tc = torch.from_numpy(coef if axis == 0 else np.ascontiguousarray(coef.T)).to(cuda)
        for npts in (64, 65, 200):
            x = rng.uniform(-0.02, 1.02, (npts, nbatch)) * scale
            for order in range(0, min(degree, 2) + 1):
                if order:
                    x = np.clip(x, orc.rmin, orc.rmax)
                tx = torch.from_numpy(x if axis == 0 else np.ascontiguousarray(x.T)).to(cuda)
                out = torch.full_like(tx, np.nan)
                (ev(out, tx, tc, axis=axis) if order == 0 else ev.deriv(order, out, tx, tc, axis=axis))
                got = out.cpu().numpy() if axis == 0 else out.cpu().numpy().T
                assert np.all(np.isfinite(got)), (nbatch, npts, order)
                ref = orc.eval(x[:, some], coef[:, some], deriv=order, extrap=("constant", "null"))
                assert rel_err(got[:, some], ref) <= 1e-13 * 10 ** order, (nbatch, npts, order)


@pytest.mark.parametrize("degree", [3, 5])
@pytest.mark.parametrize("scale", [1e-100, 1e-40, 1e100])
def test_derivatives_at_extreme_scales(degree, scale, cuda):
    """deriv(1) and the adjoint where the divisors' product leaves the range of a
    double (test_nonuniform_values_at_extreme_scales for the values)."""
    import torch

    import ddc_amd as D

    bs, orc = _space(degree, 200, scale, seed=12)
    ev = D.SplineEvaluator(bs)
    rng = np.random.default_rng(13)
    for nbatch in (3, 37):  # the per-point kernel and a tile
        coef, w = rng.standard_normal((orc.size, nbatch)), rng.standard_normal((400, nbatch))
        x = rng.uniform(orc.rmin, orc.rmax, (400, nbatch))
        tx, tw, tc = (torch.from_numpy(a).to(cuda) for a in (x, w, coef))
        out, gx, gc = torch.full_like(tx, np.nan), torch.full_like(tx, np.nan), torch.full_like(tc, np.nan)
        ev.deriv(1, out, tx, tc)
        assert rel_err(out.cpu().numpy(), orc.eval(x, coef, deriv=1)) <= 1e-12
        ev.eval_vjp(tx, tw, tc, gx, gc)
        ref_c, ref_x = orc.eval_vjp(x, w, coef)
        assert rel_err(gx.cpu().numpy(), ref_x) <= 1e-12 and rel_err(gc.cpu().numpy(), ref_c) <= 1e-12


def _edges(br):
    """Break points, the edges of equal buckets, and their neighbours."""
    lo, hi = br[0], br[-1]
    base = np.concatenate([br, lo + np.arange(len(br)) * ((hi - lo) / (len(br) - 1))])
    return np.clip(np.concatenate([base, np.nextafter(base, np.inf), np.nextafter(base, -np.inf)]), lo, hi)


@pytest.mark.parametrize("mesh,cells", [("random", 300), ("jitter", 200), ("geometric", 340)])
@pytest.mark.parametrize("axis", [0, 1])
def test_first_derivative_at_knots(mesh, cells, axis, cuda):
    """The slope of a degree-1 spline jumps at every knot: a point in a
    neighbouring cell shows, in the per-point kernel, the tiles and the streaming
    kernel, in deriv(1) and in the adjoint."""
    import torch

    import ddc_amd as D

    bs, orc = _space(1, cells, mesh=mesh, seed=11)
    ev = D.SplineEvaluator(bs)
    x1 = _edges(orc.knots()[1:-1])
    c1 = np.random.default_rng(5).standard_normal(orc.size)
    ref = orc.eval(x1[:, None], c1[:, None], deriv=1)
    for nbatch in (2, 9, 32 * _cus(cuda) + 16):
        if axis == 1 and nbatch > 9:
            continue
        for part in np.array_split(np.arange(len(x1)), 3):  # up to 1152 points for the streaming kernel
            shape = (lambda n: (n, nbatch)) if axis == 0 else (lambda n: (nbatch, n))
            col = (lambda a: a[:, None]) if axis == 0 else (lambda a: a[None, :])
            tx = torch.from_numpy(col(x1[part])).to(cuda).expand(shape(len(part))).contiguous()
            tc = torch.from_numpy(col(c1)).to(cuda).expand(shape(orc.size)).contiguous()
            out, gx, gc = torch.empty_like(tx), torch.empty_like(tx), torch.empty_like(tc)
            ev.deriv(1, out, tx, tc, axis=axis)
            want = torch.from_numpy(col(ref[part, 0])).to(cuda)
            assert float((out - want).abs().max()) <= 1e-12 * np.abs(ref).max(), nbatch
            ev.eval_vjp(tx, torch.ones_like(tx), tc, gx, gc, axis=axis)
            assert float((gx - want).abs().max()) <= 1e-12 * np.abs(ref).max(), nbatch


@pytest.mark.parametrize("degree", [1, 3])
def test_binned_points_at_knots(degree, cuda):
    """The count pass finds the cells of several points together, the tile pass
    one by one: points at the knots of both dimensions against the kernel
    without binning."""
    import torch

    import ddc_amd as D
    from ddc_amd._lib import call
    import ctypes as C

    (b1, o1), (b2, o2) = _space(degree, 90, mesh="random", seed=2), _space(degree, 70, mesh="geometric")
    e1, e2 = D.SplineEvaluator(b1), D.SplineEvaluator(b2)
    x1, x2 = _edges(o1.knots()[degree:-degree]), _edges(o2.knots()[degree:-degree])
    x = np.stack(np.meshgrid(x1, x2, indexing="ij"), axis=-1).reshape(1, -1, 2)
    npts = x.shape[1]
    rng = np.random.default_rng(0)
    tx, tw = torch.from_numpy(x).to(cuda), torch.from_numpy(rng.standard_normal((1, npts))).to(cuda)
    coef = torch.from_numpy(rng.standard_normal((1, b1.size(), b2.size()))).to(cuda)

    def run(name, *work):
        gx, gc = torch.full_like(tx, np.nan), torch.full_like(coef, np.nan)
        call(name, e1._h, e2._h, tx.data_ptr(), tw.data_ptr(), gx.data_ptr(), npts, coef.data_ptr(), gc.data_ptr(),
             *coef.stride(), 1, *work, None)
        torch.cuda.synchronize()
        return gx.cpu().numpy(), gc.cpu().numpy()

    need = C.c_int64(0)
    call("ddcx_evaluator2d_eval_vjp_workspace", e1._h, e2._h, npts, 1, C.byref(need))
    ws = torch.empty(need.value, dtype=torch.uint8, device=cuda)
    gx, gc = run("ddcx_evaluator2d_eval_vjp")
    bx, bc = run("ddcx_evaluator2d_eval_vjp_binned", ws.data_ptr(), need.value)
    assert np.array_equal(gx, bx) and np.abs(gc - bc).max() <= 1e-12 * np.abs(gc).max()


@pytest.mark.parametrize("degree,mesh", [(1, "uniform"), (3, "uniform"), (5, "uniform"), (3, "random")])
@pytest.mark.parametrize("cells", [150, 400, 700])
def test_adjoint_by_size(degree, mesh, cells, cuda):
    """The adjoint on 256, 512 and 1024 threads and on 16-line tiles, around the
    batch sizes and point counts at which they change, rows a power of two apart
    and not."""
    import torch

    import ddc_amd as D

    cus = _cus(cuda)
    bs, orc = _space(degree, cells, mesh=mesh)
    ev = D.SplineEvaluator(bs, D.ConstantExtrapolationRule(), D.NullExtrapolationRule())
    rng = np.random.default_rng(4)
    size = orc.size
    for nbatch, npts in ((8 * cus, 64), (8 * cus + 1, 100), (32 * cus - 1, size // 4), (32 * cus, size // 4),
                         (32 * cus, size), (32 * cus, size + 1), (32 * cus + 9, size // 4), (32 * cus + 9, size // 4 + 1)):
        if npts < 64:
            continue
        some = _some(nbatch)
        coef = rng.standard_normal((size, nbatch))
        if mesh == "uniform":
            coef[-degree:] = coef[:degree]
        x, w = rng.uniform(-0.02, 1.02, (npts, nbatch)), rng.standard_normal((npts, nbatch))
        tx, tw, tc = (torch.from_numpy(a).to(cuda) for a in (x, w, coef))
        gx, gc = torch.full_like(tx, np.nan), torch.full_like(tc, np.nan)
        ev.eval_vjp(tx, tw, tc, gx, gc)
        assert bool(torch.isfinite(gx).all()) and bool(torch.isfinite(gc).all()), (nbatch, npts)
        ref_c, ref_x = orc.eval_vjp(x[:, some], w[:, some], coef[:, some], extrap=("constant", "null"))
        assert rel_err(gx.cpu().numpy()[:, some], ref_x) <= 1e-13, (nbatch, npts)
        assert rel_err(gc.cpu().numpy()[:, some], ref_c) <= 1e-12, (nbatch, npts)
