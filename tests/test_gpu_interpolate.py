"""interpolate() as one autograd node against the composition of SplineBuild and
SplineEval: the same values and gradients for every choice of inputs that
require a gradient, with strided values and saved-tensor hooks."""
import numpy as np
import pytest

from cases import Case, H, P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [Case(3, True, P, ncells=40), Case(3, False, H, ncells=70, mesh="jitter")],
                         ids=lambda c: c.id)
@pytest.mark.parametrize("wanted", ["vals", "coords", "derivs", "vals coords derivs"])
def test_one_node_matches_composition(case, wanted, cuda):
    import torch

    import ddc_amd as D
    from ddc_amd.autograd import SplineBuild, SplineEval, interpolate

    if wanted == "derivs" and case.bcl != H:
        pytest.skip("no derivative inputs")
    bs, builder = case.product()
    ev = D.SplineEvaluator(bs)
    n, nb = 70, 9
    rng = np.random.default_rng(0)

    def new(rows, name):
        t = torch.from_numpy(rng.uniform(0.05, 0.95, (nb, rows))).to(cuda).T  # strided: lines are rows of memory
        return t.requires_grad_(name in wanted)

    vals, coords = new(builder.npoints(), "vals"), new(n, "coords")
    nd = builder.s_nbv_xmin
    dl, dr = (new(nd, "derivs"), new(nd, "derivs")) if nd else (None, None)
    w = torch.from_numpy(rng.standard_normal((n, nb))).to(cuda)
    inputs = [t for t in (vals, coords, dl, dr) if t is not None and t.requires_grad]
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.clone(), lambda t: t):
        got = interpolate(builder, ev, vals, coords, dl, dr)
    assert len(packed) == 2
    ref = SplineEval.apply(ev, coords, SplineBuild.apply(builder, vals, dl, dr, 0), 0)
    assert torch.equal(got, ref)
    for a, b in zip(torch.autograd.grad(got, inputs, w), torch.autograd.grad(ref, inputs, w)):
        # the coefficient gradients are sums of LDS atomics in any order
        assert a.shape == b.shape and (a - b).abs().max() <= 1e-13 * b.abs().max()
