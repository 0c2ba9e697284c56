"""Binned points whose tile ranges are filled in one part or in one per XCD
(64 chunks of 4096 points per batch entry and more, given the workspace for
it): against the kernels without binning.  Values and coordinate gradients are
the same bits; coefficient gradients add the same terms in another order."""
import ctypes as C

import numpy as np
import pytest

import ddc_amd as D
from ddc_amd._lib import DDCXError, call

pytestmark = pytest.mark.gpu
LIMIT = 64 * 4096
NULL = D.NullExtrapolationRule


def _evaluator(degree, cells, periodic):
    bs = D.UniformBSplines(degree, 0.0, 1.0, cells, periodic=periodic)
    return bs, D.SplineEvaluator(bs) if periodic else D.SplineEvaluator(bs, NULL(), NULL())


def _inputs(sizes, nb, npts, nd, cuda):
    import torch

    rng = np.random.default_rng(npts)
    coef = torch.from_numpy(rng.standard_normal((nb, *sizes))).to(cuda)
    x = torch.from_numpy(rng.uniform(-0.05, 1.05, (nb, npts, nd))).to(cuda)  # some outside: no tile
    return coef, x, torch.from_numpy(rng.standard_normal((nb, npts))).to(cuda)


@pytest.mark.parametrize("npts", [LIMIT - 1, LIMIT, LIMIT + 4097])
@pytest.mark.parametrize("cells", [(40, 70), (1100, 1061)])
def test_adjoint_2d(cells, npts, cuda):
    import torch

    (bs1, e1), (bs2, e2) = _evaluator(3, cells[0], False), _evaluator(2, cells[1], True)
    nb = 2
    coef, x, w = _inputs((bs1.size(), bs2.size()), nb, npts, 2, cuda)

    def run(name, *work):
        gx, gc = torch.full_like(x, np.nan), torch.full_like(coef, np.nan)
        call(name, e1._h, e2._h, x.data_ptr(), w.data_ptr(), gx.data_ptr(), npts, coef.data_ptr(), gc.data_ptr(),
             *coef.stride(), nb, *work, None)
        torch.cuda.synchronize()
        return gx.cpu().numpy(), gc.cpu().numpy()

    need = C.c_int64(0)
    call("ddcx_evaluator2d_eval_vjp_workspace", e1._h, e2._h, npts, nb, C.byref(need))
    gx, gc = run("ddcx_evaluator2d_eval_vjp")
    per = 3 * ((4 * nb * 35 * 34 + 255) // 256 * 256 + 256)  # above the tables of one group, 32 x 32 cells per tile
    least = need.value if npts < LIMIT else nb * npts * 30 + 5 * 256 + per
    for size in sorted({least, need.value - (npts >= LIMIT), need.value}):
        ws = torch.empty(size, dtype=torch.uint8, device=cuda)
        bx, bc = run("ddcx_evaluator2d_eval_vjp_binned", ws.data_ptr(), size)
        assert np.array_equal(bx, gx), size
        assert np.abs(bc - gc).max() <= 1e-12 * np.abs(gc).max(), size
    with pytest.raises(DDCXError, match="workspace too small"):
        run("ddcx_evaluator2d_eval_vjp_binned", ws.data_ptr(), nb * npts * 30)


@pytest.mark.parametrize("npts", [LIMIT - 1, LIMIT, LIMIT + 4097])
@pytest.mark.parametrize("cells", [(9, 17, 40), (170, 165, 161)])
def test_values_3d(cells, npts, cuda):
    import torch

    pairs = [_evaluator(3, n, k == 1) for k, n in enumerate(cells)]
    ev = D.SplineEvaluatorND(*[e for _, e in pairs])
    nb = 2
    coef, x, _ = _inputs([bs.size() for bs, _ in pairs], nb, npts, 3, cuda)
    direct, binned = torch.full((nb, npts), np.nan, dtype=torch.float64, device=cuda), None
    ev.deriv([0, 0, 0], direct, x, coef, binned=False)
    need = C.c_int64(0)
    call("ddcx_evaluatornd_eval_workspace", ev._hs, 3, npts, nb, C.byref(need))
    st = (C.c_int64 * 3)(*coef.stride()[1:])
    for size in (need.value - (npts >= LIMIT), need.value):
        binned = torch.full_like(direct, np.nan)
        ws = torch.empty(size, dtype=torch.uint8, device=cuda)
        call("ddcx_evaluatornd_eval_binned", ev._hs, 3, None, binned.data_ptr(), x.data_ptr(), npts, coef.data_ptr(),
             coef.stride(0), st, nb, ws.data_ptr(), size, None)
        torch.cuda.synchronize()
        assert np.array_equal(binned.cpu().numpy(), direct.cpu().numpy()), size
    with pytest.raises(DDCXError, match="workspace"):
        call("ddcx_evaluatornd_eval_binned", ev._hs, 3, None, binned.data_ptr(), x.data_ptr(), npts, coef.data_ptr(),
             coef.stride(0), st, nb, ws.data_ptr(), nb * npts * 30, None)
