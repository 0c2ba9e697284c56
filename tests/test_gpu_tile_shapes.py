"""Builds and their adjoints where the tiled kernels change shape: main blocks
of up to 64 rows (8 segments of 4 or 8), and the batch sizes at which the 8-line
tiles of small batches hand over to the 16- and 32-line ones, against the CPU
oracle (relative error in the max norm <= 1e-13, as for every FP64 build)."""
import numpy as np
import pytest

from cases import Case, G, H, HH, P
from conftest import rel_err
from test_gpu_build import _run
from test_gpu_vjp import _vjp

pytestmark = pytest.mark.gpu
TOL = 1e-13

# ncells around the sizes at which nq (ncells less the border) crosses 32 and 64
SHORT = [Case(3, True, P, ncells=n) for n in (6, 32, 33, 34, 64, 65, 66)] + [
    Case(1, True, P, ncells=20),
    Case(2, False, G, ncells=31, mesh="random"),
    Case(3, False, H, ncells=33, mesh="random"),
    Case(4, False, P, ncells=63, mesh="jitter"),
    Case(5, True, P, ncells=30),
    Case(5, False, G, ncells=40, mesh="jitter"),
    Case(5, False, HH, ncells=62, mesh="uniform"),
]


@pytest.mark.parametrize("case", SHORT, ids=lambda c: c.id)
@pytest.mark.parametrize("layout", ["batch_contiguous", "interp_contiguous"])
@pytest.mark.parametrize("nbatch", [1, 33])
def test_short_lines(case, layout, nbatch, cuda):
    got, ref = _run(case, nbatch, layout, cuda, seed=3)
    assert rel_err(got, ref) <= TOL
    got, ref = _vjp(case, nbatch, layout, cuda, seed=4)
    assert rel_err(got, ref) <= TOL


@pytest.mark.parametrize("case,tiles", [(Case(3, True, P, ncells=300), 1), (Case(3, False, G, ncells=1000), 1),
                                        (Case(5, True, P, ncells=700), 1), (Case(4, False, P, ncells=501, mesh="jitter"), 1),
                                        (Case(3, True, P, ncells=200), 2), (Case(5, False, H, ncells=180, mesh="jitter"), 2)],
                         ids=lambda c: getattr(c, "id", None))
@pytest.mark.parametrize("layout", ["batch_contiguous", "interp_contiguous"])
def test_batch_thresholds(case, tiles, layout, cuda):
    import torch

    limit = 8 * tiles * torch.cuda.get_device_properties(cuda).multi_processor_count
    for nbatch in (9, limit - 7, limit + 1):
        got, ref = _run(case, nbatch, layout, cuda, seed=5)
        assert rel_err(got, ref) <= TOL, nbatch
        got, ref = _vjp(case, nbatch, layout, cuda, seed=6)
        assert np.all(np.isfinite(got)) and rel_err(got, ref) <= TOL, nbatch


@pytest.mark.parametrize("case", [Case(3, True, P, ncells=300), Case(5, True, P, ncells=1000)], ids=lambda c: c.id)
def test_advect_thresholds(case, cuda):
    """The fused step on 4, 8 and 16 lines per workgroup."""
    import torch

    import ddc_amd as D

    orc = case.oracle()
    bs, builder = case.product()
    ev = D.SplineEvaluator(bs)
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    rng = np.random.default_rng(1)
    for nbatch in (3, 4 * cus + 1, 8 * cus + 1):
        f = rng.standard_normal((orc.npts, nbatch))
        shift = rng.uniform(-0.03, 0.03, nbatch)
        ref = orc.eval(builder.interpolation_points()[:, None] - shift[None, :], orc.build(f))
        out = torch.full((orc.npts, nbatch), np.nan, dtype=torch.float64, device=cuda)
        D.advect(builder, ev, out, torch.from_numpy(f).to(cuda), torch.from_numpy(shift).to(cuda))
        assert rel_err(out.cpu().numpy(), ref) <= TOL, nbatch


@pytest.mark.parametrize("case", [Case(3, True, P, ncells=90), Case(2, True, G, ncells=70), Case(5, True, P, ncells=300),
                                  Case(4, False, P, ncells=101, mesh="jitter"), Case(3, False, G, ncells=1000)],
                         ids=lambda c: c.id)
@pytest.mark.parametrize("axis", [0, 1])
def test_eval_thresholds(case, axis, cuda):
    """Values and first derivatives on 4, 8 and 16 lines per workgroup, with
    points outside the domain for the values."""
    import torch

    import ddc_amd as D

    orc = case.oracle()
    bs, _ = case.product()
    ev = D.SplineEvaluator(bs, D.ConstantExtrapolationRule(), D.NullExtrapolationRule())
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    rng = np.random.default_rng(2)

    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a if axis == 0 else a.T)).to(cuda)

    for nbatch in (8, 4 * cus - 1, 4 * cus + 1, 8 * cus - 3, 8 * cus + 1):
        coef = rng.standard_normal((orc.size, nbatch))
        if case.periodic:
            coef[-case.degree:] = coef[:case.degree]
        x = rng.uniform(-0.05, 1.05, (67, nbatch))
        out = torch.empty_like(dev(x))
        ev(out, dev(x), dev(coef), axis=axis)
        got = out.cpu().numpy() if axis == 0 else out.cpu().numpy().T
        ref = orc.eval(x, coef, extrap=("constant", "null"))
        assert rel_err(got, ref) <= TOL, nbatch
        x = np.clip(x, 0.0, 1.0)
        ev.deriv(1, out, dev(x), dev(coef), axis=axis)
        got = out.cpu().numpy() if axis == 0 else out.cpu().numpy().T
        assert rel_err(got, orc.eval(x, coef, deriv=1, extrap=("constant", "null"))) <= 10 * TOL, nbatch


@pytest.mark.parametrize("case", [Case(3, True, P, ncells=450), Case(4, False, G, ncells=600, mesh="jitter"),
                                  Case(3, True, G, ncells=1100), Case(5, False, H, ncells=1100, mesh="jitter")],
                         ids=lambda c: c.id)
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("npts,extra", [(450, 1), (600, 15)])
def test_eval_wide_batches(case, axis, npts, extra, cuda):
    """Past the small batches: the 16-line tile, the streaming kernel's 768-point
    form (rows that start at 128-byte lines) and the narrow tiles of the others."""
    import torch

    import ddc_amd as D

    orc = case.oracle()
    bs, _ = case.product()
    ev = D.SplineEvaluator(bs, D.ConstantExtrapolationRule(), D.NullExtrapolationRule())
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    rng = np.random.default_rng(4)
    for nbatch in (8 * cus + extra, 32 * cus + 16 * extra):
        coef = rng.standard_normal((orc.size, nbatch))
        if case.periodic:
            coef[-case.degree:] = coef[:case.degree]
        x = rng.uniform(0.0, 1.0, (npts, nbatch))
        tx, tc = ((torch.from_numpy(a).to(cuda) if axis == 0 else torch.from_numpy(np.ascontiguousarray(a.T)).to(cuda))
                  for a in (x, coef))
        out = torch.full_like(tx, float("nan"))
        for order in (0, 1):
            (ev(out, tx, tc, axis=axis) if order == 0 else ev.deriv(1, out, tx, tc, axis=axis))
            got = out.cpu().numpy() if axis == 0 else out.cpu().numpy().T
            assert rel_err(got, orc.eval(x, coef, deriv=order, extrap=("constant", "null"))) <= TOL * 10 ** order


@pytest.mark.parametrize("case", [Case(3, True, P, ncells=100), Case(5, True, G, ncells=128),
                                  Case(3, False, G, ncells=128), Case(5, False, P, ncells=90, mesh="jitter")],
                         ids=lambda c: c.id)
@pytest.mark.parametrize("axis", [0, 1])
def test_eval_vjp_short_lines(case, axis, cuda):
    """The adjoint on 256 threads (up to 384 points) and on 1024, with odd numbers
    of 8-line tiles; coordinates <= 1e-13, coefficients <= 1e-12."""
    import torch

    import ddc_amd as D

    orc = case.oracle()
    bs, _ = case.product()
    ev = D.SplineEvaluator(bs, D.ConstantExtrapolationRule(), D.NullExtrapolationRule())
    nbatch = 8 * torch.cuda.get_device_properties(cuda).multi_processor_count + 13
    rng = np.random.default_rng(3)

    def dev(a):
        return torch.from_numpy(np.ascontiguousarray(a if axis == 0 else a.T)).to(cuda)

    for npts in (64, 384, 385):
        coef = rng.standard_normal((orc.size, nbatch))
        if case.periodic:
            coef[-case.degree:] = coef[:case.degree]
        x, w = rng.uniform(-0.02, 1.02, (npts, nbatch)), rng.standard_normal((npts, nbatch))
        gx, gc = torch.full_like(dev(x), float("nan")), torch.full_like(dev(coef), float("nan"))
        ev.eval_vjp(dev(x), dev(w), dev(coef), gx, gc, axis=axis)
        got_c, got_x = ((t.cpu().numpy() if axis == 0 else t.cpu().numpy().T) for t in (gc, gx))
        ref_c, ref_x = orc.eval_vjp(x, w, coef, extrap=("constant", "null"))
        assert rel_err(got_x, ref_x) <= 1e-13 and rel_err(got_c, ref_c) <= 1e-12, npts
