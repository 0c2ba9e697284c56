"""Every 1D entry point on views that are not plain arrays: rows padded beyond
the batch, two batch dimensions around the row dimension, and unit-stride rows
with a gap, at a small batch (narrow tiles) and at one of more 32-line tiles
than CUs (workgroups that walk tiles), against the oracle on the first, the
last and some lines between.  Nothing outside a view may be written."""
import numpy as np
import pytest

from cases import Case, G, H, P
from conftest import rel_err

pytestmark = pytest.mark.gpu
KINDS = ["padded", "middle", "rows"]


class _View:
    """A (rows, lines) array stored as `kind`; t is the view passed on."""

    def __init__(self, kind, rows, outer, inner, pad, cuda, data=None):
        import torch

        shape = {"padded": (rows, outer * inner + pad), "middle": (outer, rows, inner + pad),
                 "rows": (outer * inner, rows + pad)}[kind]
        self.axis = {"padded": 0, "middle": 1, "rows": 1}[kind]
        self.base = torch.full(shape, 7.5, dtype=torch.float64, device=cuda)
        self.t = self.base[..., :shape[-1] - pad]
        self.kind, self.rows, self.outer, self.inner = kind, rows, outer, inner
        if data is not None:
            d = {"padded": lambda: data, "middle": lambda: data.reshape(rows, outer, inner).transpose(1, 0, 2),
                 "rows": lambda: data.T}[kind]()
            self.t.copy_(torch.from_numpy(np.ascontiguousarray(d)))
        else:
            self.t.fill_(float("nan"))

    def numpy(self):
        pad = self.base.shape[-1] - self.t.shape[-1]
        assert pad == 0 or bool((self.base[..., -pad:] == 7.5).all()), "written outside the view"
        a = self.t.cpu().numpy()
        if self.kind == "middle":
            a = a.transpose(1, 0, 2).reshape(self.rows, -1)
        elif self.kind == "rows":
            a = a.T
        assert np.all(np.isfinite(a)), "not fully written"
        return a


@pytest.mark.parametrize("case", [Case(3, True, P, ncells=40), Case(3, True, P, ncells=300),
                                  Case(4, False, G, ncells=301, mesh="jitter"),
                                  Case(5, False, H, ncells=1000, mesh="jitter")], ids=lambda c: c.id)
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("large", [False, True], ids=["small", "large"])
def test_views(case, kind, large, cuda):
    import torch

    import ddc_amd as D

    orc = case.oracle()
    bs, builder = case.product()
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    outer, inner = (5, 8 * cus + 1) if large else (7, 45)
    nb = outer * inner
    rng = np.random.default_rng(8)
    some = np.unique(np.concatenate([[0, 1, nb - 2, nb - 1], rng.integers(0, nb, 40)]))

    def view(rows, pad, data=None):
        return _View(kind, rows, outer, inner, pad, cuda, data)

    hermite = case.bcl == H
    f = rng.standard_normal((orc.npts, nb))
    dl, dr = (rng.standard_normal((n, nb)) if hermite else None for n in (orc.nbv_l, orc.nbv_r))
    tf, tc = view(orc.npts, 3, f), view(orc.size, 2)
    axis = tf.axis
    td = [view(len(d), 1, d).t if hermite else None for d in (dl, dr)]
    builder(tc.t, tf.t, *td, axis=axis)
    got = tc.numpy()
    ref = orc.build(f[:, some], dl[:, some] if hermite else None, dr[:, some] if hermite else None)
    assert rel_err(got[:, some], ref) <= 1e-13, "build"

    g = rng.standard_normal((orc.size, nb))
    gv = view(orc.npts, 4)
    gd = [view(n, 1) if hermite else None for n in (orc.nbv_l, orc.nbv_r)]
    builder.build_vjp(view(orc.size, 1, g).t, gv.t, *[v.t if hermite else None for v in gd], axis=axis)
    ref = orc.build_vjp(g[:, some])
    got = np.concatenate([gv.numpy()[:, some]] + [v.numpy()[:, some] for v in gd if hermite])
    assert rel_err(got, np.concatenate([ref[0]] + ([ref[1], ref[2]] if hermite else []))) <= 1e-13, "build adjoint"

    ev = D.SplineEvaluator(bs, D.ConstantExtrapolationRule(), D.NullExtrapolationRule())
    coef = rng.standard_normal((orc.size, nb))
    if case.periodic:
        coef[-case.degree:] = coef[:case.degree]
    x, w = rng.uniform(0.0, 1.0, (130, nb)), rng.standard_normal((130, nb))
    vc, vx, out = view(orc.size, 6, coef), view(130, 5, x), view(130, 5)
    rule = ("constant", "null")
    ev(out.t, vx.t, vc.t, axis=axis)
    assert rel_err(out.numpy()[:, some], orc.eval(x[:, some], coef[:, some], extrap=rule)) <= 1e-13, "eval"
    ev.deriv(1, out.t, vx.t, vc.t, axis=axis)
    ref = orc.eval(x[:, some], coef[:, some], deriv=1, extrap=rule)
    assert rel_err(out.numpy()[:, some], ref) <= 1e-12, "deriv"
    gx, gc = view(130, 5), view(orc.size, 6)
    ev.eval_vjp(vx.t, view(130, 5, w).t, vc.t, gx.t, gc.t, axis=axis)
    ref_c, ref_x = orc.eval_vjp(x[:, some], w[:, some], coef[:, some], extrap=rule)
    assert rel_err(gx.numpy()[:, some], ref_x) <= 1e-13, "eval adjoint, coordinates"
    assert rel_err(gc.numpy()[:, some], ref_c) <= 1e-12, "eval adjoint, coefficients"
