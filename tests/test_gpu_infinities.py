"""Builds of lines that hold an infinity or NaN: the non-finite coefficients of a
line are the same in both layouts (rows that only pad the tiles add none), and
other lines are untouched."""
import numpy as np
import pytest

from cases import Case, G, P

pytestmark = pytest.mark.gpu
CASES = [Case(d, u, b, ncells=n, mesh="jitter")
         for d, u, b, n in ((1, True, G, 37), (3, True, G, 40), (3, True, P, 75), (3, False, G, 130), (4, False, P, 203),
                            (5, True, G, 300), (3, True, G, 1000), (3, True, P, 1030), (5, False, G, 700))]
CASES += [Case(d, u, b, ncells=n, mesh="jitter") for n in range(64, 71) for d, u, b in
          ((3, True, G), (3, True, P), (5, False, P), (4, False, G))]


@pytest.mark.parametrize("case", CASES, ids=lambda c: c.id)
def test_same_rows_in_both_layouts(case, cuda):
    import torch

    orc = case.oracle()
    bs, builder = case.product()
    n = orc.npts
    for nbatch in (3, 37, 9000):
        rng = np.random.default_rng(nbatch)
        f = rng.standard_normal((n, nbatch))
        clean = torch.from_numpy(f).to(cuda)
        bad = {0: (n - 1, np.inf), nbatch - 1: (n - 1, -np.inf), nbatch // 2: (n // 2, np.nan)}
        if nbatch > 30:
            bad |= {2 + k: (n - 2 - k, np.inf) for k in range(6)} | {20 + k: (k, np.inf) for k in range(6)}
        for line, (row, v) in bad.items():
            f[row, line] = v
        vals = torch.from_numpy(f).to(cuda)
        coef = torch.empty(orc.size, nbatch, dtype=torch.float64, device=cuda)
        base = torch.empty_like(coef)
        lines = torch.empty(nbatch, orc.size, dtype=torch.float64, device=cuda)
        builder(coef, vals)
        builder(base, clean)
        builder(lines, vals.t().contiguous(), axis=1)
        b = sorted(bad)
        assert bool((torch.isfinite(coef[:, b]) == torch.isfinite(lines.t()[:, b])).all()), nbatch
        assert bool((torch.isnan(coef[:, b]) == torch.isnan(lines.t()[:, b])).all()), nbatch
        keep = np.setdiff1d(np.arange(nbatch), b)
        assert bool((coef[:, keep] == base[:, keep]).all()) and bool(torch.isfinite(coef[:, keep]).all()), nbatch
