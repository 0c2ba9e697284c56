"""Rounding of the basis weights themselves.  A line whose coefficients are 1 at
every (D + 1)-th index and 0 elsewhere returns one weight per point, so the
evaluators show their basis arithmetic without a sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _derivative_weights(knots, degree, x):
    """First-derivative weights (points, D + 1) in 80 bits, and the cells."""
    t = knots.astype(np.longdouble)
    cell = np.clip(np.searchsorted(knots, x, side="right") - 1, degree, len(knots) - degree - 2)
    z = x.astype(np.longdouble)
    v = [np.ones_like(z)]
    for q in range(1, degree):
        nxt = [np.zeros_like(z) for _ in range(q + 1)]
        for r in range(q):
            lo, hi = t[cell + r + 1 - q], t[cell + r + 1]
            nxt[r] += (hi - z) / (hi - lo) * v[r]
            nxt[r + 1] += (z - lo) / (hi - lo) * v[r]
        v = nxt
    d = [np.zeros_like(z) for _ in range(degree + 1)]
    for r in range(degree):
        s = degree * v[r] / (t[cell + r + 1] - t[cell + r + 1 - degree])
        d[r] -= s
        d[r + 1] += s
    return np.stack(d, axis=1), cell - degree


@pytest.mark.parametrize("degree", [3, 5, 6])
@pytest.mark.parametrize("lines", ["one", "tile", "stream"])
def test_first_derivative_weights_nonuniform(degree, lines, cuda):
    """deriv(1) and the adjoint's w f'(x) on a random mesh.  A weight is the
    result of about 5 roundings for each of its D levels (two knot differences,
    a reciprocal, a product, a fused update), each of rms 2^-53 / sqrt(3):
    together sqrt(5 D) * 6.4e-17 of the cell's largest weight."""
    import torch

    import ddc_amd as D

    n, npts = 300, 1000
    cus = torch.cuda.get_device_properties(cuda).multi_processor_count
    # whole sets of D + 1 lines: the per-point kernel, the tiles, the streaming kernel
    sets = {"one": 1, "tile": 6, "stream": (2 * 16 * cus) // (degree + 1) + 2}[lines]
    rng = np.random.default_rng(degree)
    breaks = np.concatenate([[0.0], np.sort(rng.uniform(0, 1, n - 1)), [1.0]])
    bs = D.NonUniformBSplines(degree, breaks)
    ev = D.SplineEvaluator(bs)
    x = rng.uniform(0.0, 1.0, npts)
    ref, jmin = _derivative_weights(bs.knots(), degree, x)
    nb = sets * (degree + 1)
    rows = torch.arange(bs.size(), device=cuda) % (degree + 1)
    coef = (rows[:, None] == torch.arange(nb, device=cuda)[None, :] % (degree + 1)).to(torch.float64)
    tx = torch.from_numpy(x).to(cuda)[:, None].expand(npts, nb).contiguous()
    out, gx, gc = torch.empty_like(tx), torch.empty_like(tx), torch.empty_like(coef)
    ev.deriv(1, out, tx, coef)
    ev.eval_vjp(tx, torch.ones_like(tx), coef, gx, gc)
    for name, got in (("deriv", out), ("eval_vjp", gx)):
        a = got.cpu().numpy().reshape(npts, sets, degree + 1)
        w = np.empty_like(ref)  # the line that holds weight i of the point
        for i in range(degree + 1):
            w[np.arange(npts), (jmin + i) % (degree + 1)] = ref[:, i]
        err = np.abs(a - w[:, None, :]) / np.abs(ref).max(1)[:, None, None]
        rms = float(np.sqrt((err.astype(float) ** 2).mean()))
        assert rms <= np.sqrt(5 * degree) * 2.0 ** -53 / np.sqrt(3.0), (name, rms)
