"""The small levels of a V-cycle in one workgroup, against the oracle bit for
bit (FP64: whole solves, replayed) and, for the FP32 cycles, against the same
cycle run as one launch per step.

Shapes: level 1 of exactly 4096 cells and just above (the leg then starts a
level lower), flat and long ones, periodic axes of two cells (boundary planes
that touch) and of eight and more (wrapped in FP32)."""
import numpy as np
import pytest

import oracle
from briscola_amd import workloads as W

pytestmark = pytest.mark.gpu

N, D, P = W.NEUMANN, W.DIRICHLET, W.PERIODIC


def problem(n, bc, seed):
    verts = [np.cumsum(np.concatenate(([0.0], 1.0 + 0.2*np.sin(np.arange(q)))))
             / q for q in n]
    rng = np.random.default_rng(seed)
    b = np.zeros(tuple(q + 2 for q in n))
    b[1:-1, 1:-1, 1:-1] = rng.uniform(-1, 1, n) / np.prod(n)
    if D not in bc:
        b[1:-1, 1:-1, 1:-1] -= b[1:-1, 1:-1, 1:-1].mean()
    return verts, b


@pytest.mark.parametrize("n,bc,pre,post,coarse_level", [
    ((32, 32, 32), (N,) * 6, 2, 2, 1),             # level 1: 4096 cells
    ((32, 32, 32), (P, P, D, N, P, P), 2, 2, 1),
    ((48, 32, 24), (N, N, D, D, P, P), 2, 2, 1),   # level 1: 4608
    ((8, 64, 64), (D, D, P, P, N, N), 1, 2, 1),    # flat: axes stop halving
    ((16, 8, 64), (P, P, P, P, D, N), 0, 1, 0),
    ((24, 24, 24), (P, P, P, P, P, P), 3, 1, 1),
    ((16, 16, 16), (N, D, N, D, P, P), 1, 0, 0),
    ((8, 8, 8), (P, P, N, N, D, D), 2, 3, 0),
])
def test_solve_bitwise(gpu, n, bc, pre, post, coarse_level):
    print(f"[tail] n={n} bc={bc} sweeps={pre},{post}", flush=True)
    opts = dict(rel_tol=1e-9, tolerance=0.0, n_sweeps_pre=pre,
                n_sweeps_post=post, cycle=oracle.VCYCLE, max_iter=6,
                coarse_mode=oracle.COARSE_DIRECT, coarse_level=coarse_level)
    verts, b0 = problem(n, bc, 5)
    o = oracle.Oracle(verts, bc)
    o.set_opts(**opts)
    o.assemble(None)
    o.set_field(oracle.B, 0, b0)
    it, _, _ = o.solve()
    ctx = gpu.Context(verts, bc, **opts)
    ctx.set_laplacian(None)
    for _ in range(3):
        x, st = ctx.solve(b0.copy())
        assert st.iters == it
        assert np.array_equal(x, o.field(oracle.X, 0))


@pytest.mark.parametrize("bc", [(N,) * 6, (D, N, P, P, N, D), (P,) * 6])
@pytest.mark.parametrize("n", [(16, 16, 16), (24, 16, 32), (32, 32, 32),
                               (48, 16, 32)])
@pytest.mark.parametrize("coarse_level", [0, 1])
def test_fp32_leg_equals_launches(gpu, n, bc, coarse_level):
    """Mixed solves: the leg against one launch per step (fused smoothing,
    which changes no bits, keeps the cycles to launches).  The FP32 row
    products are contracted as each kernel's compilation chooses, so a
    correction may differ by its rounding, 2^-24 per operation of a sweep's
    some twenty: 2e-6 of x, and of the residual, which later corrections
    reduce alike, far less than the 1e-3 a wrong ghost or weight changes."""
    print(f"[tail fp32] n={n} bc={bc} coarse_level={coarse_level}", flush=True)
    verts, b0 = problem(n, bc, 9)
    out = []
    for mode in (0, 2):
        ctx = gpu.Context(verts, bc, rel_tol=1e-12, tolerance=0.0,
                          max_iter=5, n_sweeps_pre=2, n_sweeps_post=2,
                          cycle=gpu.VCYCLE, coarse_mode=gpu.COARSE_DIRECT,
                          coarse_level=coarse_level, precision=gpu.MIXED)
        ctx.set_fused_smoothing(mode)
        ctx.set_laplacian(None)
        x, st = ctx.solve(b0.copy())
        out.append((x, st.final_residual))
    (a, ra), (b, rb) = out
    assert np.abs(a - b).max() <= 2e-6 * np.abs(a).max()
    assert abs(ra - rb) <= 1e-3 * ra


@pytest.mark.parametrize("bc", [(N, D, D, N, N, D), (P, P, N, D, D, D),
                                (P, P, P, P, D, N), (P,) * 6, (N,) * 6,
                                (D, D, P, P, N, N)])
@pytest.mark.parametrize("n,cycle", [((64, 32, 32), oracle.VCYCLE),
                                     ((48, 64, 32), oracle.WCYCLE),
                                     ((32, 48, 96), oracle.FCYCLE)])
def test_ghosts_formed_by_prolongation(gpu, n, cycle, bc):
    """Levels of more than 4096 cells, whose ghosts the prolongation forms
    itself: faces of every kind next to each other (edges and corners of
    mixed kinds), bit for bit."""
    opts = dict(rel_tol=1e-9, tolerance=0.0, n_sweeps_pre=1, n_sweeps_post=1,
                cycle=cycle, max_iter=3, coarse_mode=oracle.COARSE_DIRECT,
                coarse_level=1)
    verts, b0 = problem(n, bc, 7)
    o = oracle.Oracle(verts, bc)
    o.set_opts(**opts)
    o.assemble(None)
    o.set_field(oracle.B, 0, b0)
    it, _, _ = o.solve()
    ctx = gpu.Context(verts, bc, **opts)
    ctx.set_laplacian(None)
    for _ in range(2):
        x, st = ctx.solve(b0.copy())
        assert st.iters == it
        assert np.array_equal(x, o.field(oracle.X, 0))


@pytest.mark.parametrize("bc", [(N, D, P, P, N, N), (P, P, D, N, P, P)])
@pytest.mark.parametrize("faces", [False, True])
def test_residual_restricted_as_formed(gpu, faces, bc):
    """A level of more than 32768 cells below the finest: its residual by
    axis factors or face coefficients, restricted in the same launch, bit for
    bit (coarse rows of 24 cells, packed; the levels below are stencils)."""
    n = (64, 96, 96)
    opts = dict(rel_tol=1e-9, tolerance=0.0, n_sweeps_pre=1, n_sweeps_post=1,
                cycle=oracle.VCYCLE, max_iter=2,
                coarse_mode=oracle.COARSE_DIRECT, coarse_level=1)
    verts, b0 = problem(n, bc, 11)
    lam = None
    if faces:
        rng = np.random.default_rng(12)
        lam = [10.0**rng.uniform(-1, 1, b0.shape) for _ in range(3)]
        for d in range(3):
            if bc[2*d] == P:
                # one coefficient for the two sides of a periodic face
                m = np.moveaxis(lam[d], d, 0)
                m[n[d] + 1] = m[1]
    o = oracle.Oracle(verts, bc)
    o.set_opts(**opts)
    o.assemble(lam)
    o.set_field(oracle.B, 0, b0)
    it, _, _ = o.solve()
    ctx = gpu.Context(verts, bc, **opts)
    ctx.set_laplacian(lam)
    x, st = ctx.solve(b0.copy())
    assert st.iters == it
    assert np.array_equal(x, o.field(oracle.X, 0))
