"""Learned preconditioner on the device: the BF16 matrix-core convolution
kernels against the CPU reference (oracle/unet_ref.py) -- forward, data
gradient and weight gradient --, a training step that lowers the loss, and
the learned flexible-CG solve, which must reach the same tolerance and the
same solution as the plain FP64 solve (the fall-back to MG cycles keeps it
convergent whatever the network predicts)."""
import numpy as np
import pytest

from oracle import unet_ref as U
from briscola_amd import bmg, unet, workloads as W

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev_bf16(a):
    """float32 array of BF16 values -> bfloat16 cuda tensor (same bits)."""
    t = torch.from_numpy(U.bf16_bits(a).view(np.int16)).to("cuda:0")
    return t.view(torch.bfloat16)


def host(t):
    return t.float().cpu().numpy()


def close(gpu, ref, rel=2e-2):
    scale = np.abs(ref).max() + 1e-30
    err = np.abs(gpu - ref).max() / scale
    assert err < rel, f"max error {err:.3e} of the largest value"


@pytest.mark.parametrize("shape,cin,cout,relu", [
    ((8, 8, 8), 16, 16, True),
    ((8, 16, 8), 8, 32, False),
    ((16, 8, 8), 48, 48, True),
    ((8, 8, 16), 192, 64, True),
    # partial output tiles (x, y and z extents not multiples of the tile)
    ((6, 10, 20), 32, 96, True),
    ((4, 6, 12), 96, 192, False),
    ((3, 5, 7), 8, 128, True),
])
def test_conv_forward(gpu, shape, cin, cout, relu):
    r = np.random.default_rng(cin + cout)
    x = U.to_bf16(r.standard_normal(shape + (cin,)).astype(np.float32))
    kp = unet.round32(27 * cin)
    w = np.zeros((cout, kp), np.float32)
    w[:, :27 * cin] = U.to_bf16(
        (r.standard_normal((cout, 27 * cin)) / np.sqrt(27 * cin)).astype(np.float32))
    bias = r.standard_normal(cout).astype(np.float32)
    ref = U.conv(x, w[:, :27 * cin], bias, relu)
    y = unet.op_conv(dev_bf16(x), dev_bf16(w),
                     torch.from_numpy(bias).to("cuda:0"), cout, relu)
    close(host(y), ref)


@pytest.mark.parametrize("cin,cout", [(16, 32), (48, 16), (96, 32)])
def test_conv_data_gradient(gpu, cin, cout):
    r = np.random.default_rng(7 + cin)
    shape = (8, 8, 16)
    dz = U.to_bf16(r.standard_normal(shape + (cout,)).astype(np.float32))
    kp = unet.round32(27 * cin)
    w = np.zeros((cout, kp), np.float32)
    w[:, :27 * cin] = U.to_bf16(
        (r.standard_normal((cout, 27 * cin)) / np.sqrt(27 * cout)).astype(np.float32))
    ref = U.conv_dgrad(dz, w[:, :27 * cin], cin)
    dx = unet.op_conv_dgrad(dev_bf16(dz), dev_bf16(w), cin)
    close(host(dx), ref)


@pytest.mark.parametrize("cin,cout,chunk", [(8, 16, 256), (32, 64, 160),
                                            (48, 16, 1024)])
def test_conv_weight_gradient(gpu, cin, cout, chunk):
    r = np.random.default_rng(11 + cin)
    shape = (8, 16, 8)
    x = U.to_bf16(r.standard_normal(shape + (cin,)).astype(np.float32))
    dz = U.to_bf16(r.standard_normal(shape + (cout,)).astype(np.float32))
    kp = unet.round32(27 * cin)
    ref = U.conv_wgrad(x, dz, kp)
    dw = unet.op_conv_wgrad(dev_bf16(x), dev_bf16(dz), kp, chunk)
    got = dw.cpu().numpy()
    # FP32 accumulation of exact BF16 products
    assert np.abs(got - ref).max() < 1e-4 * np.abs(ref).max()
    assert np.all(got[:, 27 * cin:] == 0.0)


def small_problem(n=16, seed=3):
    return W.spheres(n, seed=seed, nspheres=4)


def test_training_lowers_the_loss(gpu):
    prob = small_problem()
    ctx = bmg.Context(prob.vertices, prob.bc, prob.bc_value, rel_tol=1e-10,
                      tolerance=0.0, max_iter=500, n_sweeps_pre=2,
                      n_sweeps_post=2, cycle=bmg.VCYCLE, coarse_level=1,
                      krylov=bmg.KRYLOV_FCG)
    ctx.set_laplacian(prob.lam)
    x, _ = ctx.solve(prob.b.copy())
    f, c, t, _, _ = unet.scaled_pair(prob, x)
    net = unet.Net(seed=1)
    d = lambda a: torch.from_numpy(a).to("cuda:0")
    F, C, T = d(f), d(c), d(t)
    losses = [net.train_step(F, C, T, 1e-3) for _ in range(40)]
    assert np.isfinite(losses).all()
    assert losses[-1] < 0.5 * losses[0], losses[::8]
    # the forward entry point gives the trained prediction
    p = net.forward(F, C).cpu().numpy()
    e = p - p.mean() - t
    assert np.mean(e * e) < losses[0]


@pytest.mark.parametrize("seed", [1, 4])
def test_network_gradient_matches_oracle(gpu, seed):
    """One training step's gradient (every convolution's weights and bias,
    the head; bmg_unet_get_grads) and loss against the float64 restatement
    of the whole network (oracle/unet_ref.py, pinned by central differences
    in tests/test_unet_oracle.py) with BF16 rounding where the device stores
    BF16, on a 16^3 input: the backward kernels of the ReLU, pooling,
    upsampling, concatenation, head, bias sums and loss all enter it."""
    D = 16
    r = np.random.default_rng(seed)
    f = r.standard_normal((D, D, D)).astype(np.float32)
    c = r.uniform(-1, 1, (D, D, D)).astype(np.float32)
    t = r.standard_normal((D, D, D)).astype(np.float32)
    net = unet.Net(seed=seed)
    P = net.params().astype(np.float64)
    d = lambda a: torch.from_numpy(a).to("cuda:0")
    loss = net.train_step(d(f), d(c), d(t), 0.0)
    G = net.grads().astype(np.float64)
    L, Gr = U.net_loss_grad(P, f.astype(np.float64), c.astype(np.float64),
                            t.astype(np.float64), bf16=True)
    L0, G0 = U.net_loss_grad(P, f.astype(np.float64), c.astype(np.float64),
                             t.astype(np.float64))
    lay, hoff, n = U.param_layout()
    names = ["E0", "E1", "E2", "E3", "D2", "D1", "D0"]
    rows = [("loss", abs(loss - L) / L, 1.0)]
    groups = []
    for name, (wo, bo, kp), (cin, cout, _, _) in zip(names, lay, U.CONVS):
        groups.append((name + " w", slice(wo, wo + cout * kp)))
        groups.append((name + " b", slice(bo, bo + cout)))
    groups.append(("head", slice(hoff, hoff + 17)))
    worst = 0.0
    for name, sl in groups:
        g, gr, g0 = G[sl], Gr[sl], G0[sl]
        rel = np.linalg.norm(g - gr) / np.linalg.norm(gr)
        cos = float(g @ gr / (np.linalg.norm(g) * np.linalg.norm(gr)))
        rel0 = np.linalg.norm(g - g0) / np.linalg.norm(g0)
        rows.append((name, rel, cos, rel0))
        worst = max(worst, rel)
    print(f"\n[unet grad] seed {seed}: loss device {loss:.6g} oracle {L:.6g}")
    for row in rows[1:]:
        print(f"[unet grad] {row[0]:7s} rel err vs BF16 oracle {row[1]:.2e} "
              f"cos {row[2]:.6f}; vs exact float64 {row[3]:.2e}")
    assert abs(loss - L) <= 1e-3 * L and abs(L - L0) <= 2e-2 * L0
    for name, rel, cos, rel0 in rows[1:]:
        assert rel < 0.05 and cos > 0.998, (name, rel, cos)
        assert rel0 < 0.15, (name, rel0)
    # the padded channels of the first convolution get no gradient
    w0 = G[lay[0][0]:lay[0][1]].reshape(16, lay[0][2])
    assert not w0[:, 27 * 8:].any()
    assert not w0[:, :27 * 8].reshape(16, 27, 8)[:, :, 2:].any()
    net.close()


@pytest.mark.parametrize("precision", [bmg.FP64, bmg.MIXED], ids=["fp64", "mixed"])
def test_learned_fcg_reaches_tolerance(gpu, precision):
    prob = W.spheres(32, seed=2, nspheres=6)
    base = dict(rel_tol=1e-8, tolerance=0.0, max_iter=500, n_sweeps_pre=2,
                n_sweeps_post=2, cycle=bmg.VCYCLE, coarse_level=1,
                precision=precision)
    ref = bmg.Context(prob.vertices, prob.bc, prob.bc_value,
                      **dict(base, krylov=bmg.KRYLOV_FCG, rel_tol=1e-12,
                             precision=bmg.FP64))
    ref.set_laplacian(prob.lam)
    xr, _ = ref.solve(prob.b.copy())
    ctx = bmg.Context(prob.vertices, prob.bc, prob.bc_value,
                      **dict(base, krylov=bmg.KRYLOV_FCG_LEARNED))
    ctx.set_laplacian(prob.lam)
    net = unet.Net(seed=5)
    net.attach(ctx)
    x, st = ctx.solve(prob.b.copy())
    assert st.final_residual / st.initial_residual <= 1e-8
    xi, ri = x[1:-1, 1:-1, 1:-1], xr[1:-1, 1:-1, 1:-1]
    err = np.linalg.norm((xi - xi.mean()) - (ri - ri.mean())) / np.linalg.norm(ri - ri.mean())
    assert err < 1e-5
    assert st.learned_fallback != -1 or st.learned_iters == st.iters
    # and against an FP64 direct solve of the oracle's eliminated system
    import oracle
    from oracle import direct
    o = oracle.Oracle(prob.vertices, prob.bc, prob.bc_value)
    o.assemble(prob.lam)
    o.pin_and_eliminate()
    xs = direct.solve_sparse(o.stencil(0), prob.b, prob.bc)
    err_d = direct.rel_error(xi, xs, True)
    print(f"[learned fcg] precision={precision}: {st.iters} iterations, "
          f"error vs sparse direct {err_d:.2e}", flush=True)
    assert err_d < 1e-5


def guess_error(net, prob, xr):
    """Relative L2 error (mean removed) of the network's initial guess
    x = U(b / rms(b)) * rms(b) / (h s) against the solution xr."""
    f, c, _, rms, hs = unet.scaled_pair(prob)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    u = net.forward(d(f), d(c)).cpu().numpy().astype(np.float64)
    g = (u - u.mean()) * rms / hs
    ri = xr[1:-1, 1:-1, 1:-1]
    ri = ri - ri.mean()
    return float(np.linalg.norm(g - ri) / np.linalg.norm(ri))


def test_what_training_gains(gpu, capsys):
    """What the trained network gains over the method without it, measured
    on held-out problems of its training distribution (spheres, density
    ratio 1000, 32^3; trained on 32 other seeds with the project's own
    kernels).  Training must bring the network's initial guess closer to the
    solution than the untrained network's and than the zero guess FCG starts
    from without a network.  The learned flexible-CG solve is then timed
    against FCG with the MG cycle alone and both iteration counts are
    printed: at this training budget the guess is still tens of percent off,
    the solver keeps it only when it lowers the residual, and the learned
    solve reaches the tolerance in no more iterations than the method without
    the network plus the fall-back's restart."""
    from briscola_amd import train_unet
    net, hist, _, _ = train_unet.train(32, 32, 20, lr=2e-3, verbose=False)
    raw = unet.Net(seed=7)
    assert hist[-1] < 0.2 * hist[0], hist
    rows = []
    for s in range(2):
        prob = W.spheres(32, seed=9000 + s)
        ref = train_unet.solver(prob, bmg.KRYLOV_FCG, 1e-12)
        xr, _ = ref.solve(prob.b.copy())
        ref.close()
        e_trained = guess_error(net, prob, xr)
        e_raw = guess_error(raw, prob, xr)
        # the zero guess has relative error 1
        assert e_trained < 1.0 and e_trained < e_raw, (e_trained, e_raw)
        it = {}
        for name, kry in (("fcg", bmg.KRYLOV_FCG),
                          ("fcg_learned", bmg.KRYLOV_FCG_LEARNED)):
            ctx = train_unet.solver(prob, kry, 1e-8, bmg.MIXED)
            if kry == bmg.KRYLOV_FCG_LEARNED:
                net.attach(ctx)
            _, st = ctx.solve(prob.b.copy())
            ctx.close()
            assert st.final_residual / st.initial_residual <= 1e-8
            it[name] = (st.iters, st.learned_guess_residual)
        assert it["fcg_learned"][0] <= it["fcg"][0] + 2, it
        rows.append((s, e_trained, e_raw, it))
    with capsys.disabled():
        for s, et, er, it in rows:
            print(f"\n[learned gain] held-out seed {s}: guess error trained "
                  f"{et:.3f} / untrained {er:.3g} / zero 1; FCG iterations "
                  f"{it['fcg'][0]} without the network, "
                  f"{it['fcg_learned'][0]} with it (guess residual "
                  f"{it['fcg_learned'][1]:.3g} of the zero guess's)")


@pytest.mark.parametrize("shape", [(3, 5, 7), (6, 9, 16), (5, 17, 33),
                                   (4, 8, 40), (2, 4, 8)])
@pytest.mark.parametrize("cin,cout", [(8, 16), (16, 32), (48, 16), (32, 64),
                                      (64, 128)])
def test_wgrad_tiles(gpu, shape, cin, cout):
    """The tiled weight gradient at rows of every residue grouping (at most 8,
    9 to 16, above), partial tiles on each axis and all output groupings;
    exact BF16 products summed in FP32 (bound as above)."""
    r = np.random.default_rng(cin + cout)
    x = U.to_bf16(r.standard_normal(shape + (cin,)).astype(np.float32))
    dz = U.to_bf16(r.standard_normal(shape + (cout,)).astype(np.float32))
    kp = unet.round32(27 * cin)
    ref = U.conv_wgrad(x, dz, kp)
    got = unet.op_conv_wgrad(dev_bf16(x), dev_bf16(dz), kp).cpu().numpy()
    assert np.abs(got - ref).max() < 1e-4 * np.abs(ref).max()
    assert np.all(got[:, 27 * cin:] == 0.0)


@pytest.mark.parametrize("shape,cin,cout", [((4, 6, 20), 192, 64),
                                            ((8, 8, 8), 64, 128),
                                            ((5, 3, 17), 48, 48),
                                            ((16, 16, 16), 64, 192)])
def test_small_grid_forward(gpu, shape, cin, cout):
    """Grids of few tiles take output channels in groups over workgroups."""
    r = np.random.default_rng(cin)
    x = U.to_bf16(r.standard_normal(shape + (cin,)).astype(np.float32))
    kp = unet.round32(27 * cin)
    w = np.zeros((cout, kp), np.float32)
    w[:, :27 * cin] = U.to_bf16(
        (r.standard_normal((cout, 27 * cin)) / np.sqrt(27 * cin)).astype(
            np.float32))
    bias = r.standard_normal(cout).astype(np.float32)
    ref = U.conv(x, w[:, :27 * cin], bias, relu=True)
    y = unet.op_conv(dev_bf16(x), dev_bf16(w), torch.from_numpy(bias).cuda(),
                     cout, True).float().cpu().numpy()
    # one BF16 rounding of the result and FP32 sums
    assert np.abs(y - ref).max() <= 2.0**-8 * np.abs(ref).max()


@pytest.mark.parametrize("shape", [(8, 8, 8), (16, 24, 40), (8, 48, 16),
                                   (32, 32, 64), (64, 64, 64)])
def test_inference_pass(gpu, shape):
    """The inference pass (first convolution from the FP32 inputs, upsampling
    and skips read in place, averages and output projection in the epilogues)
    against the float64 restatement with the same BF16 roundings; partial
    tiles at every level, one and several tiles.  FP32 sums flip the rounding
    of some activations, by 2^-9 of a value each; were every activation of the
    eight layers one rounding apart, the output would be off by about
    sqrt(8) 2^-9 = 0.0055, the bound 2^-7 (a wrong tap or row is of order
    one).  The same after a training step, whose buffers the pass shares."""
    r = np.random.default_rng(sum(shape))
    f = r.standard_normal(shape).astype(np.float32)
    c = np.where(r.uniform(size=shape) > 0.5, 1.0, -1.0).astype(np.float32)
    net = unet.Net(seed=5)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    F, C = dev(f), dev(c)
    for step in range(2):
        if step:
            if np.prod(shape) > 20000:
                break
            net.train_step(F, C, dev(f), 1e-3)
        ref, _ = U.net_forward(net.params().astype(np.float64),
                               f.astype(np.float64), c.astype(np.float64),
                               bf16=True)
        got = host(net.forward(F, C))
        rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert rel < 2.0**-7, rel
    net.close()


def jacobi_net(alpha):
    """A network with U(f, c) = alpha f: the first convolution's centre tap
    gives the two signs of f, the last one passes them on, the head subtracts
    them."""
    net = unet.Net(seed=0)
    lay, hoff, n = U.param_layout()
    P = np.zeros(n, np.float32)
    wo, _, kp = lay[0]
    P[wo + 13*8], P[wo + kp + 13*8] = 1.0, -1.0
    wo, _, kp = lay[6]
    P[wo + 13*48 + 32], P[wo + kp + 13*48 + 33] = 1.0, 1.0
    P[hoff], P[hoff + 1] = alpha, -alpha
    net.set_params(P)
    return net


def test_learned_solve_after_the_buffers_moved(gpu):
    """A learned solve repeats bit for bit after its network's activations
    were replaced: by a training step (learning rate 0) on the same grid, and
    by a context of another size on the same network.  The solve's captured
    iteration refers to the activations, so it has to be captured anew."""
    net = jacobi_net(-1.0/7.0)
    ctxs, bs = [], []
    for n in ((16, 16, 16), (24, 16, 32)):
        c = bmg.Context([np.arange(q + 1)/16.0 for q in n], (0, 0, 1, 1, 0, 1),
                        rel_tol=1e-8, tolerance=0.0, n_sweeps_pre=2,
                        n_sweeps_post=2, cycle=bmg.VCYCLE, coarse_level=1,
                        krylov=bmg.KRYLOV_FCG_LEARNED)
        c.set_laplacian(None)
        net.attach(c)
        b = np.zeros(c.padded(0))
        b[1:-1, 1:-1, 1:-1] = np.random.default_rng(1).standard_normal(n)
        ctxs.append(c)
        bs.append(b)
    first = []
    for c, b in zip(ctxs, bs):
        x, st = c.solve(b.copy())
        assert st.learned_iters > 0, st.learned_guess_residual
        first.append(x)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    for k in (0, 1, 0, 0, 1):
        x, st = ctxs[k].solve(bs[k].copy())
        assert st.learned_iters > 0 and np.array_equal(x, first[k])
        f = dev(bs[k][1:-1, 1:-1, 1:-1].astype(np.float32))
        net.train_step(f, torch.ones_like(f), f, 0.0)
        x, st = ctxs[k].solve(bs[k].copy())
        assert st.learned_iters > 0 and np.array_equal(x, first[k])
    for c in ctxs:
        c.close()
    net.close()


def test_infinite_input_stays_infinite(gpu):
    """With positive weights throughout, one infinite input gives infinities
    and no NaN: the matrix instructions' padding multiplies no value of the
    tile by its zeros."""
    shape = (16, 8, 24)
    net = unet.Net(seed=0)
    net.set_params(np.abs(net.params()))
    f = np.random.default_rng(2).uniform(0.0, 1.0, shape).astype(np.float32)
    f[5, 3, 13] = np.inf
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    got = host(net.forward(dev(f), torch.ones(shape, device="cuda:0")))
    assert np.isinf(got[5, 3, 13]) and not np.isnan(got).any()
    net.close()


@pytest.mark.parametrize("shape", [(6, 10, 20), (4, 16, 32)])
@pytest.mark.parametrize("c0,c1", [(0, 16), (32, 16), (64, 32)])
@pytest.mark.parametrize("tile", [(4, 8), (4, 4), (2, 8), (1, 8), (1, 4)])
def test_inference_convolution_tiles(gpu, tile, c0, c1, shape):
    """Every tile of the inference pass's convolution, with and without the
    averages and (16 channels) the output projection, from a tensor of half
    the extents and a slice of a wider one, into a slice: partial and whole
    tiles, one group of output channels and two.  y against float64 sums of
    the BF16 products (one BF16 rounding, 2^-8 of the largest value, as
    above); the averages and the projection bit for bit from y, in the order
    of the training pass."""
    r = np.random.default_rng(c0 + tile[0])
    cin, cout = c0 + c1, 16*tile[0]*(2 if tile[0] < 4 else 1)
    coarse = tuple(n // 2 for n in shape)
    rnd = lambda s: U.to_bf16(r.standard_normal(s).astype(np.float32))
    u, x = rnd(coarse + (c0,)), rnd(shape + (c1,))
    w = np.zeros((cout, unet.round32(27*cin)), np.float32)
    w[:, :27*cin] = U.to_bf16((r.standard_normal((cout, 27*cin))
                               / np.sqrt(27*cin)).astype(np.float32))
    bias = r.standard_normal(cout).astype(np.float32)
    cat = np.concatenate([U.up(u), x], axis=3)
    ref = U.conv(cat, w[:, :27*cin], bias, relu=True)
    # the fine tensor and the output as slices of wider ones
    wide = dev_bf16(np.concatenate([np.zeros_like(x), x], axis=3))
    y = torch.full(shape + (cout + 16,), 7.0, dtype=torch.bfloat16,
                   device="cuda:0")
    pool = torch.zeros(coarse + (cout,), dtype=torch.bfloat16, device="cuda:0")
    args = (dev_bf16(u) if c0 else None, wide[..., c1:], dev_bf16(w),
            torch.from_numpy(bias).to("cuda:0"))
    unet.op_conv_rows(*args, y=y[..., 16:], tile=tile)
    got = host(y[..., 16:])
    assert np.abs(got - ref).max() <= 2.0**-8*np.abs(ref).max()
    assert bool((y[..., :16] == 7.0).all())
    y2 = torch.zeros_like(y)
    unet.op_conv_rows(*args, y=y2[..., 16:], pool=pool, tile=tile)
    assert np.array_equal(host(y2[..., 16:]), got)
    s = np.zeros(coarse + (cout,), np.float32)
    for d in range(8):
        s += got[d >> 2::2, (d >> 1) & 1::2, d & 1::2]
    assert np.array_equal(host(pool), U.to_bf16(np.float32(0.125)*s))
    if tile[0] > 1:
        return
    # the output projection: the first 16 channels' convolution
    h = r.standard_normal(17).astype(np.float32)
    out = torch.zeros(shape, device="cuda:0")
    unet.op_conv_rows(args[0], args[1], args[2][:16].contiguous(), args[3][:16],
                      head=torch.from_numpy(h).to("cuda:0"), out=out, tile=tile)
    e = np.full(shape, h[16])
    for c in range(16):
        e = e + h[c]*got[..., c]
    assert e.dtype == np.float32 and np.array_equal(host(out), e)


def test_inference_convolution_refuses_other_tiles(gpu):
    x = torch.zeros((2, 8, 16, 16), dtype=torch.bfloat16, device="cuda:0")
    w = torch.zeros((32, 448), dtype=torch.bfloat16, device="cuda:0")
    y = torch.zeros((2, 8, 16, 32), dtype=torch.bfloat16, device="cuda:0")
    b = torch.zeros(32, device="cuda:0")
    for tile in ((4, 8), (3, 8), (2, 4), (1, 2)):
        with pytest.raises(bmg.BmgError):
            unet.op_conv_rows(None, x, w, b, y=y, tile=tile)


@pytest.mark.parametrize("cin,cout,chunk", [(24, 16, 32), (24, 40, 100),
                                            (40, 16, 1000), (16, 24, 7),
                                            (8, 20, 4096)])
def test_general_weight_gradient(gpu, cin, cout, chunk):
    """Channel counts the tiled weight gradient does not take, in chunks that
    do not divide the 315 voxels, larger ones and ones below a K step; exact
    BF16 products summed in FP32, bound as above."""
    r = np.random.default_rng(cin + chunk)
    shape = (5, 7, 9)
    x = U.to_bf16(r.standard_normal(shape + (cin,)).astype(np.float32))
    dz = U.to_bf16(r.standard_normal(shape + (cout,)).astype(np.float32))
    kp = unet.round32(27 * cin)
    ref = U.conv_wgrad(x, dz, kp)
    got = unet.op_conv_wgrad(dev_bf16(x), dev_bf16(dz), kp, chunk).cpu().numpy()
    assert np.abs(got - ref).max() < 1e-4 * np.abs(ref).max()
    assert np.all(got[:, 27 * cin:] == 0.0)
