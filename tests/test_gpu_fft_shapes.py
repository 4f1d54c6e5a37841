"""The FFT solver's plane pairs, mirror-image orbits and transform lengths at
the sizes where they can go wrong: odd and even, one and two cells along a
transformed axis, odd and even plane counts along every tridiagonal axis, more
than one block of modes, against the oracle (1e-11 of the solution, as the
solver's other tests)."""
import itertools

import numpy as np
import pytest

from briscola_amd import bmg
from oracle import fft_ref as F

pytestmark = pytest.mark.gpu

PAIRS = {"N": (F.NEU, F.NEU), "D": (F.DIR, F.DIR), "P": (F.PER, F.PER),
         "Q": (F.DIR, F.NEU), "R": (F.NEU, F.DIR)}


def vertices(n, stretch):
    verts = [np.linspace(0.0, 1.0 + d, q + 1) for d, q in enumerate(n)]
    if stretch is not None and n[stretch] > 1:
        t = np.linspace(-1.0, 1.0, n[stretch] + 1)
        verts[stretch] = np.tanh(1.5 * t) / np.tanh(1.5)
    return verts


def shapes():
    """(n, stretched axis, kinds): periodic axes are uniform, and the
    tridiagonal axis has at least two cells (three if periodic)."""
    out = []
    for n, stretch, kinds in itertools.product(
            [(7, 9, 11), (6, 5, 8), (3, 2, 1), (2, 1, 3), (5, 70, 67)],
            [0, 1, 2, None],
            ["NDP", "PPN", "QRD", "PQP", "DNR", "PPP", "NNN", "RPQ"]):
        if stretch is not None and kinds[stretch] == "P":
            continue
        s = F.plan(vertices(n, stretch))[0]
        if n[s] >= (3 if kinds[s] == "P" else 2):
            out.append((n, stretch, kinds))
    return out


@pytest.mark.parametrize("n,stretch,kinds", shapes())
def test_odd_and_small_sizes(gpu, n, stretch, kinds):
    verts = vertices(n, stretch)
    bc = [k for a in kinds for k in PAIRS[a]]
    print(f"[fft shapes] n={n} kinds={kinds} stretch={stretch}", flush=True)
    rng = np.random.default_rng(4)
    b = np.zeros(tuple(q + 2 for q in n))
    b[1:-1, 1:-1, 1:-1] = rng.standard_normal(n)
    if F.DIR not in bc:
        # a compatible source: the pinned row of the zero mode else amplifies
        # rounding by the condition of the singular operator
        w = [np.diff(v) for v in verts]
        vol = w[0][:, None, None] * w[1][None, :, None] * w[2][None, None, :]
        b[1:-1, 1:-1, 1:-1] -= (vol * b[1:-1, 1:-1, 1:-1]).sum() / vol.sum()
    x0 = np.zeros_like(b)
    ref = np.asarray(F.solve(b, x0, bc, verts))
    x = bmg.FFT(verts, bc).solve(b.copy(), x0.copy())
    got = x[1:-1, 1:-1, 1:-1]
    assert np.abs(got - ref).max() <= 1e-11 * np.abs(ref).max()


@pytest.mark.parametrize("kinds", ["DRP", "NPD", "PNR"])
@pytest.mark.parametrize("n", [(4, 70000, 3), (140000, 3, 4)])
def test_axes_beyond_the_grid_limit(gpu, n, kinds):
    """An axis of more cells, rows or plane pairs than the 65536 workgroups
    that a launch takes along y or z: the seven-point operator on the result
    (its ghosts included) gives back the source.  Its rounding is that of a
    few sums of terms of the size of x/h^2, and the transforms add log2 of
    their length roundings, so the bound is 64 eps max|x|/h^2."""
    h = 0.125
    verts = [np.arange(q + 1)*h for q in n]
    bc = [k for a in kinds for k in PAIRS[a]]
    b = np.zeros(tuple(q + 2 for q in n))
    b[1:-1, 1:-1, 1:-1] = np.random.default_rng(5).standard_normal(n)
    print(f"[fft long] n={n} kinds={kinds}", flush=True)
    x = bmg.FFT(verts, bc).solve(b.copy(), np.zeros_like(b))
    c = (slice(1, -1),)*3
    lap = -6.0*x[c]
    for d in range(3):
        for e in (slice(None, -2), slice(2, None)):
            lap += x[c[:d] + (e,) + c[d + 1:]]
    err = np.abs(lap/h**2 + b[c]).max()
    bound = 64*np.finfo(float).eps*np.abs(x).max()/h**2
    print(f"[fft long] residual {err:.2e}, bound {bound:.2e}", flush=True)
    assert err <= bound
