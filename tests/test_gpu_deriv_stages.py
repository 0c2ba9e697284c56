"""First derivatives of non-uniform bases on both sides of the rule for the
points per thread and stage: one or several, whole and partial last groups, in
both layouts, aligned rows and not, narrow and wide tiles."""
import numpy as np
import pytest

from cases import Case, G, P
from conftest import rel_err

pytestmark = pytest.mark.gpu
CASES = [Case(3, False, P, ncells=40, mesh="jitter"), Case(5, False, G, ncells=750, mesh="jitter"),
         Case(6, False, P, ncells=100, mesh="jitter"), Case(1, False, G, ncells=1500, mesh="jitter")]


@pytest.mark.parametrize("npts", [64, 65, 127, 129, 192, 257, 300, 513, 1025])
@pytest.mark.parametrize("case", CASES, ids=lambda c: c.id)
def test_first_derivative(case, npts, cuda):
    import torch

    import ddc_amd as D

    orc = case.oracle()
    bs, _ = case.product()
    ev = D.SplineEvaluator(bs) if case.periodic else \
        D.SplineEvaluator(bs, D.ConstantExtrapolationRule(), D.ConstantExtrapolationRule())
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    rng = np.random.default_rng(npts)
    for nbatch in (9, 8 * cus + 3, 9 * cus):
        some = np.unique(np.concatenate([[0, nbatch - 1], rng.integers(0, nbatch, 6)]))
        x = rng.uniform(orc.rmin, orc.rmax, (npts, nbatch))
        c = rng.standard_normal((orc.size, nbatch))
        ref = orc.eval(x[:, some], c[:, some], deriv=1)
        tx, tc = torch.from_numpy(x).to(cuda), torch.from_numpy(c).to(cuda)
        for axis in (0, 1):
            ax, ac = (tx, tc) if axis == 0 else (tx.t().contiguous(), tc.t().contiguous())
            out = torch.full_like(ax, np.nan)
            ev.deriv(1, out, ax, ac, axis=axis)
            got = (out if axis == 0 else out.t()).cpu().numpy()
            assert np.isfinite(got).all()
            assert rel_err(got[:, some], ref) <= 1e-12, (nbatch, axis)
