"""New operators in a context that already has one.

Buffers of the old operator are kept where the new one needs them in the same
sizes; levels of at most 32768 cells are stored as stencils through a scratch
that all of them share.  Whatever a context held before, the new operator's
stencils on every level and its solve have to be those of a fresh context, bit
for bit.
"""
import numpy as np
import pytest

from briscola_amd import bmg, unet

pytestmark = pytest.mark.gpu


def context(n, precision):
    verts = [np.arange(q + 1)/max(n) for q in n]
    faces = (bmg.NEUMANN, bmg.DIRICHLET, bmg.NEUMANN, bmg.NEUMANN,
             bmg.PERIODIC, bmg.PERIODIC)
    return bmg.Context(verts, faces, rel_tol=1e-8, tolerance=0.0,
                       coarse_mode=bmg.COARSE_DIRECT, coarse_level=1,
                       precision=precision, krylov=bmg.KRYLOV_FCG)


def coefficients(shape, seed):
    rng = np.random.default_rng(seed)
    return [10.0**rng.uniform(-2, 2, shape) for _ in range(3)]


# extents: every level a stencil; one level of faces or axis factors; two
@pytest.mark.parametrize("n", [(16, 24, 32), (48, 32, 24), (96, 64, 48)])
@pytest.mark.parametrize("precision", [bmg.FP64, bmg.MIXED])
def test_update_equals_fresh(gpu, n, precision):
    used = context(n, precision)
    shape = used.padded(0)
    steps = [dict(lam=coefficients(shape, 1)),
             dict(lam=coefficients(shape, 2), ddt=(0.01, 1.0)),
             dict(lam=None, ddt=(0.02, 0.5)),
             dict(lam=None),
             dict(lam=coefficients(shape, 3)),
             None,                                   # stored stencils
             dict(lam=coefficients(shape, 4))]
    rng = np.random.default_rng(5)
    b = rng.standard_normal(shape)
    for step in steps:
        fresh = context(n, precision)
        if step is None:
            src = context(n, precision)
            src.set_laplacian(coefficients(shape, 6))
            for l in range(src.nlevels):
                for c in (used, fresh):
                    c.set_stencil(l, src.stencil(l))
            src.close()
        else:
            used.set_laplacian(**step)
            fresh.set_laplacian(**step)
        for l in range(used.nlevels):
            np.testing.assert_array_equal(used.stencil(l), fresh.stencil(l))
        xu, su = used.solve(b.copy())
        xf, sf = fresh.solve(b.copy())
        assert su.iters == sf.iters
        np.testing.assert_array_equal(xu, xf)
        fresh.close()
    used.close()


@pytest.mark.parametrize("n", [(8, 8, 8), (24, 32, 16)])
def test_learned_channel_follows_operator(gpu, n):
    """The network's coefficient channel is that of the current operator."""
    verts = [np.arange(q + 1)/max(n) for q in n]
    b = np.random.default_rng(3).standard_normal([q + 2 for q in n])

    def make():
        c = bmg.Context(verts, (bmg.NEUMANN, bmg.DIRICHLET)*3, rel_tol=1e-8,
                        tolerance=0.0, coarse_mode=bmg.COARSE_DIRECT,
                        coarse_level=1, krylov=bmg.KRYLOV_FCG_LEARNED)
        net = unet.Net(seed=5)
        net.attach(c)
        return c, net
    used, net = make()
    shape = used.padded(0)
    for lam in (None, coefficients(shape, 7), coefficients(shape, 8), None):
        fresh, net2 = make()
        used.set_laplacian(lam)
        fresh.set_laplacian(lam)
        xu, su = used.solve(b.copy())
        xf, sf = fresh.solve(b.copy())
        assert (su.iters, su.learned_guess_residual) == (
            sf.iters, sf.learned_guess_residual)
        np.testing.assert_array_equal(xu, xf)
        fresh.close()
    used.close()
