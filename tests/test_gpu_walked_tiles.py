"""Builds of long lines where a workgroup walks several tiles: second and third
trips, a last trip that only some workgroups make, a last tile of a few lines,
both line counts of a tile, rows a multiple of 8 KiB apart (where the tiles are
walked from a larger batch on) and other pitches."""
import numpy as np
import pytest

from cases import Case, G, H, P
from conftest import rel_err

pytestmark = pytest.mark.gpu
# 64 segments of 32 rows in 16-line tiles, then 32 segments in 16- and 32-line tiles
CASES = [Case(3, True, H, ncells=1100), Case(3, True, P, ncells=2048), Case(3, False, H, ncells=1990, mesh="jitter"),
         Case(5, False, P, ncells=1030, mesh="jitter"), Case(3, True, P, ncells=300), Case(3, False, G, ncells=1000, mesh="jitter"),
         Case(7, True, P, ncells=1000)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: c.id)
def test_trips(case, cuda):
    import torch

    orc = case.oracle()
    bs, builder = case.product()
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    rng = np.random.default_rng(11)
    wide = case.ncells <= 1024
    for nbatch, pitch in ((32 * cus + 5, 32 * cus + 5), (40 * cus + 33, 40 * cus + 64), (48 * cus + 1, 64 * cus),
                          (72 * cus, 72 * cus), *(((130 * cus + 3, 136 * cus),) if wide else ())):
        some = np.unique(np.concatenate([[0, 1, 16 * cus - 1, 16 * cus, nbatch - 2, nbatch - 1],
                                         rng.integers(0, nbatch, 24)]))
        g = torch.Generator(device=cuda).manual_seed(3)
        vals = torch.rand(orc.npts, pitch, dtype=torch.float64, device=cuda, generator=g)[:, :nbatch]
        coef = torch.full((orc.size, pitch), np.nan, dtype=torch.float64, device=cuda)
        der = {}
        ref = {}
        if case.bcl == H:
            for k, n in (("derivs_xmin", builder.s_nbv_xmin), ("derivs_xmax", builder.s_nbv_xmax)):
                d = rng.uniform(-1, 1, (n, nbatch))
                der[k], ref[k] = torch.from_numpy(d).to(cuda), d[:, some]
        builder(coef[:, :nbatch], vals, **der)
        ref = orc.build(vals[:, torch.from_numpy(some).to(cuda)].cpu().numpy(), *ref.values())
        assert rel_err(coef[:, torch.from_numpy(some).to(cuda)].cpu().numpy(), ref) <= 1e-13, (nbatch, pitch)
        assert bool(torch.isfinite(coef[:, :nbatch]).all()) and bool(torch.isnan(coef[:, nbatch:]).all())
