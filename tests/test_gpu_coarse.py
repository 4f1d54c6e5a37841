"""Coarsest-level direct solves of more than 64 cells, where one wavefront no
longer holds a row per lane: the FP64 substitutions bit for bit against the
oracle, and the FP32 cycles' inverse through whole solves.

Sizes: 72 cells (one whole block of 64 columns and a remainder), 216 (a 6^3
level, under every 3*2^k size), 384 and 512 (either side of the two columns a
product thread keeps ahead), 1728 (beyond the staged products).
"""
import numpy as np
import pytest

import oracle
from briscola_amd import workloads as W

pytestmark = pytest.mark.gpu

N, D, P = W.NEUMANN, W.DIRICHLET, W.PERIODIC
OPTS = dict(rel_tol=1e-10, tolerance=0.0, n_sweeps_pre=2, n_sweeps_post=2,
            cycle=oracle.VCYCLE, coarse_mode=oracle.COARSE_DIRECT)


def problem(n, bc, seed):
    verts = [np.arange(q + 1) / q for q in n]
    rng = np.random.default_rng(seed)
    b = np.zeros(tuple(q + 2 for q in n))
    b[1:-1, 1:-1, 1:-1] = rng.uniform(-1, 1, n) / np.prod(n)
    if D not in bc:
        b[1:-1, 1:-1, 1:-1] -= b[1:-1, 1:-1, 1:-1].mean()
    return verts, bc, b


@pytest.mark.parametrize("n,coarse_level,cells,bc", [
    ((6, 8, 12), 1, 72, (N, N, D, N, P, P)),
    ((12, 12, 12), 1, 216, (N,) * 6),
    ((12, 12, 12), 1, 216, (P, P, D, D, N, N)),
    ((16, 16, 12), 2, 384, (D, N, P, P, N, N)),
    ((16, 16, 16), 2, 512, (P, P, P, P, D, D)),
    ((24, 24, 24), 2, 1728, (N, D, P, P, N, N)),
])
def test_substitutions_bitwise(gpu, n, coarse_level, cells, bc):
    print(f"[coarse solve] n={n} cells={cells} bc={bc}", flush=True)
    verts, bc, _ = problem(n, bc, 1)
    opts = dict(OPTS, coarse_level=coarse_level)
    o = oracle.Oracle(verts, bc)
    o.set_opts(**opts)
    o.assemble(None)
    ctx = gpu.Context(verts, bc, **opts)
    ctx.set_laplacian(None)
    o.pin_and_eliminate()
    o.prepare_coarse()
    ctx.prepare()
    lc = o.nlevels - 1 - coarse_level
    assert np.prod(ctx.shapes[lc]) == cells
    rng = np.random.default_rng(2)
    for which, v in ((oracle.X, np.zeros(o.padded(lc))),
                     (oracle.B, rng.uniform(-1, 1, o.padded(lc)))):
        o.set_field(which, lc, v)
        ctx.upload(which, lc, v)
    o.coarse_solve()
    ctx.coarse_solve()
    assert np.array_equal(ctx.download(0, lc), o.field(oracle.X, lc))


@pytest.mark.parametrize("n,coarse_level,bc", [
    ((8, 8, 8), 1, (N, D, P, P, N, N)),          # 64 cells
    ((24, 32, 48), 1, (N, N, D, D, P, P)),       # 72
    ((48, 48, 48), 1, (P, P, P, P, D, N)),       # 216
    ((48, 48, 48), 1, (N, N, P, P, N, N)),       # 216, singular
    ((32, 32, 32), 2, (P, P, P, P, P, P)),       # 512, singular
    ((16, 4, 4), 1, (N, N, D, N, D, D)),         # 16
])
@pytest.mark.parametrize("krylov", [0, 1], ids=["mg", "fcg"])
def test_inverse_in_mixed_solves(gpu, n, coarse_level, bc, krylov):
    """The mixed cycle preconditions as the FP64 one does: the iteration
    counts agree to one, a wrong row, coupling or ghost of the coarse
    correction costs several; the solution agrees to the stopping test (the
    residual bound times the condition of at most (2 n)^2)."""
    print(f"[mixed] n={n} bc={bc} krylov={krylov}", flush=True)
    verts, bc, b = problem(n, bc, 3)
    out = []
    for prec in (gpu.FP64, gpu.MIXED):
        ctx = gpu.Context(verts, bc, **dict(OPTS, coarse_level=coarse_level,
                                            precision=prec, krylov=krylov))
        # the reference's order in both, so that the counts compare
        ctx.set_periodic_smoothing(0)
        ctx.set_laplacian(None)
        x, st = ctx.solve(b.copy())
        x2, st2 = ctx.solve(b.copy(), const_matrix=True)
        assert st2.iters == st.iters and np.array_equal(x, x2)
        x3, st3 = ctx.solve(b.copy())        # refactorised
        assert st3.iters == st.iters and np.array_equal(x, x3)
        xi = x[1:-1, 1:-1, 1:-1]
        out.append((xi - xi.mean() if D not in bc else xi, st.iters))
    (a, ia), (m, im) = out
    assert abs(ia - im) <= 1, (ia, im)
    assert np.linalg.norm(a - m) <= 1e-10 * (2 * max(n))**2 * np.linalg.norm(a)
