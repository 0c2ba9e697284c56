"""The fused build and evaluation where its tables and tiles fill the LDS: long
quartic lines (128 segments without room for their transfer products), and
quintic lines whose 16-line tile does not fit.  Every case must run at any batch
size, with and without a coefficient array, and agree with the oracle."""
import numpy as np
import pytest

from cases import Case, G, P
from conftest import rel_err

pytestmark = pytest.mark.gpu
CASES = [Case(4, False, P, ncells=1100, mesh="jitter"), Case(4, False, P, ncells=1990, mesh="jitter"),
         Case(4, False, G, ncells=1500, mesh="random"), Case(5, False, P, ncells=938, mesh="jitter"),
         Case(5, False, P, ncells=1000, mesh="jitter"), Case(3, False, G, ncells=1900, mesh="random"),
         Case(5, True, P, ncells=2000)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: c.id)
def test_fused_steps(case, cuda):
    import torch

    import ddc_amd as D

    orc = case.oracle()
    bs, builder = case.product()
    ev = D.SplineEvaluator(bs) if case.periodic else \
        D.SplineEvaluator(bs, D.ConstantExtrapolationRule(), D.ConstantExtrapolationRule())
    rule = None if case.periodic else ("constant", "constant")
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    rng = np.random.default_rng(7)
    pts = builder.interpolation_points()
    for nbatch in (3, 4 * cus + 3, 8 * cus + 5):
        some = np.unique(np.concatenate([[0, 1, nbatch - 2, nbatch - 1], rng.integers(0, nbatch, 12)]))
        f = rng.standard_normal((orc.npts, nbatch))
        shift = rng.uniform(-0.03, 0.03, nbatch)
        coef = orc.build(f[:, some])
        feet = pts[:, None] - shift[None, some]
        ref = orc.eval(feet, coef) if rule is None else orc.eval(feet, coef, extrap=rule)
        tf, ts = torch.from_numpy(f).to(cuda), torch.from_numpy(shift).to(cuda)
        for spline in (None, torch.full((orc.size, nbatch), np.nan, dtype=torch.float64, device=cuda)):
            out = torch.full_like(tf, np.nan)
            D.advect(builder, ev, out, tf, ts, spline=spline)
            assert bool(torch.isfinite(out).all())
            assert rel_err(out.cpu().numpy()[:, some], ref) <= 1e-13, nbatch
            if spline is not None:
                assert rel_err(spline.cpu().numpy()[:, some], coef) <= 1e-13, nbatch
        x = rng.uniform(orc.rmin, orc.rmax, (67, nbatch))
        tx = torch.from_numpy(x).to(cuda)
        for spline in (None, torch.full((orc.size, nbatch), np.nan, dtype=torch.float64, device=cuda)):
            out = torch.full_like(tx, np.nan)
            D.build_eval(builder, ev, out, tx, tf, spline=spline)
            assert rel_err(out.cpu().numpy()[:, some], orc.eval(x[:, some], coef)) <= 1e-13, nbatch
            if spline is not None:
                assert rel_err(spline.cpu().numpy()[:, some], coef) <= 1e-13, nbatch
