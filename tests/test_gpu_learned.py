"""Learned gauge-covariant preconditioner on the GPU, through the C ABI,
against the oracle's layers (oracle/wilson_oracle.c or_net_layer*).

Bars (relative 2-norm):
  * layer forward / adjoint vs the oracle that rounds the transported values
    to bfloat16 exactly as the matrix-core operands are: 1e-4.  The residue
    is the transported values whose FP32 (device) and FP64 (oracle) forms
    round to different bf16 neighbours: probability ~1e-7/2^-8 each, error
    2^-8 each, ~3e-5 in the 2-norm over 288 products per output;
  * the same vs the unrounded FP64 oracle: 1e-2 (bf16 has 8 significant bits);
  * weight gradient (FP32 VALU) vs the FP64 oracle: 1e-5;
  * network gradient vs central finite differences of the FP64 oracle loss
    along random weight directions: 3e-2 (bf16 forward and adjoint);
  * gauge covariance of M: 2e-2 (different bf16 roundings of rotated fields).
"""
import os

import numpy as np
import pytest

import iroiro_amd as ii
from oracle import oracle as orc
from tests.wilson_math import GAMMAS, random_su3, shift_index

pytestmark = pytest.mark.gpu

DIMS = (4, 4, 4, 8)
WIDTHS = (1, 8, 8, 8, 1)


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(b))


def bf16_weights(rng, shape, scale=0.3):
    w = scale * (rng.normal(size=shape) + 1j * rng.normal(size=shape))
    return orc.bf16_round(w.real) + 1j * orc.bf16_round(w.imag)


@pytest.fixture(scope="module")
def env():
    lat = orc.Lattice(DIMS)
    u = lat.apbc(lat.gauge_expH(0.4, 2024))
    ctx = ii.Context(DIMS)
    ctx.upload_gauge(u)
    net = ii.LearnedPreconditioner(ctx)
    yield lat, u, ctx, net
    ctx.close()


@pytest.mark.parametrize("layer", [0, 1, 3])
def test_layer_forward_vs_oracle(env, layer):
    lat, u, ctx, net = env
    rng = np.random.default_rng(10 + layer)
    cin, cout = WIDTHS[layer], WIDTHS[layer + 1]
    w = bf16_weights(rng, (9, cout, cin, 4, 4))
    net.set_weights(layer, w)
    x = rng.normal(size=cin * lat.full_size).astype(np.float32).astype(np.float64)
    got = net.layer_apply(layer, x)
    assert rel(got, lat.net_layer(u, w, x, round_bf16=True)) < 1e-4
    assert rel(got, lat.net_layer(u, w, x)) < 1e-2


@pytest.mark.parametrize("layer", [1, 3])
def test_layer_adjoint_vs_oracle(env, layer):
    lat, u, ctx, net = env
    rng = np.random.default_rng(20 + layer)
    cin, cout = WIDTHS[layer], WIDTHS[layer + 1]
    w = bf16_weights(rng, (9, cout, cin, 4, 4))
    net.set_weights(layer, w)
    g = rng.normal(size=cout * lat.full_size).astype(np.float32).astype(np.float64)
    got = net.layer_apply(layer, g, adjoint=True)
    assert rel(got, lat.net_layer_adj(u, w, g, round_bf16=True)) < 1e-4
    assert rel(got, lat.net_layer_adj(u, w, g)) < 1e-2


@pytest.mark.parametrize("layer", [0, 1, 3])
def test_layer_weight_gradient_vs_oracle(env, layer):
    lat, u, ctx, net = env
    rng = np.random.default_rng(30 + layer)
    cin, cout = WIDTHS[layer], WIDTHS[layer + 1]
    x = rng.normal(size=cin * lat.full_size).astype(np.float32).astype(np.float64)
    g = rng.normal(size=cout * lat.full_size).astype(np.float32).astype(np.float64)
    got = net.layer_wgrad(layer, x, g)
    ref = lat.net_layer_wgrad(u, cin, cout, x, g)
    assert rel(got, ref) < 1e-5


@pytest.mark.parametrize("dims", [(2, 2, 2, 2), (4, 2, 2, 6), (6, 4, 2, 10)])
@pytest.mark.parametrize("layer", [0, 1, 3])
def test_layer_weight_gradient_partial_stages(dims, layer):
    """Lattices of 16, 96 and 480 sites against the kernel's stages of 32: a
    stage with sites missing, a parity boundary inside a stage, blocks of one
    stage.  Bar 1e-6: FP32 sums of 192 terms a stage (2^-24 sqrt(192) = 8e-7)."""
    lat = orc.Lattice(dims)
    u = lat.apbc(lat.gauge_expH(0.4, 31))
    rng = np.random.default_rng(50 + layer)
    cin, cout = WIDTHS[layer], WIDTHS[layer + 1]
    x = rng.normal(size=cin * lat.full_size).astype(np.float32).astype(np.float64)
    g = rng.normal(size=cout * lat.full_size).astype(np.float32).astype(np.float64)
    ctx = ii.Context(dims)
    ctx.upload_gauge(u)
    got = ii.LearnedPreconditioner(ctx).layer_wgrad(layer, x, g)
    ctx.close()
    assert rel(got, lat.net_layer_wgrad(u, cin, cout, x, g)) < 1e-6


def test_network_gradient_vs_oracle_finite_differences(env):
    lat, u, ctx, net = env
    rng = np.random.default_rng(40)
    ws = [bf16_weights(rng, (9, WIDTHS[l + 1], WIDTHS[l], 4, 4), 0.15) for l in range(4)]
    for l, w in enumerate(ws):
        net.set_weights(l, w)
    pairs = [(rng.normal(size=lat.half_size), rng.normal(size=lat.half_size)) for _ in range(2)]
    pairs = [(b.astype(np.float32).astype(np.float64), y.astype(np.float32).astype(np.float64))
             for b, y in pairs]
    loss, grads = net.loss_grad([p[0] for p in pairs], [p[1] for p in pairs])
    ref_loss, ref_grads = orc.Net(lat, u, ws).loss_and_grad(pairs)
    assert abs(loss - ref_loss) < 2e-2 * ref_loss
    for l in range(4):
        assert rel(grads[l], ref_grads[l]) < 3e-2, l
    # directional finite differences of the FP64 oracle loss
    h = 1e-4
    for trial in range(3):
        dirs = [rng.normal(size=w.shape) + 1j * rng.normal(size=w.shape) for w in ws]
        wp = [w + h * d for w, d in zip(ws, dirs)]
        wm = [w - h * d for w, d in zip(ws, dirs)]
        fd = (orc.Net(lat, u, wp).loss_and_grad(pairs)[0] -
              orc.Net(lat, u, wm).loss_and_grad(pairs)[0]) / (2 * h)
        an = sum(float(np.sum(g.real * d.real + g.imag * d.imag)) for g, d in zip(grads, dirs))
        assert abs(an - fd) < 3e-2 * abs(fd), (trial, an, fd)


def test_neumann_init_weights_and_series(env):
    lat, u, ctx, net = env
    kappa = 0.125
    net.init_neumann(kappa, noise=0.0)
    w0 = net.get_weights(0)
    for mu in range(4):
        np.testing.assert_allclose(w0[2 * mu + 1, 1, 0], kappa * (np.eye(4) - GAMMAS[mu]),
                                   atol=1e-7)
        np.testing.assert_allclose(w0[2 * mu + 2, 1, 0], kappa * (np.eye(4) + GAMMAS[mu]),
                                   atol=1e-7)
    # M r = even part of sum_{k<=4} (kappa H)^k (r, 0), kappa H = 1 - D
    r = orc.gauss_field(lat.half_size, 7)
    f = lat.merge(r, np.zeros(lat.half_size))
    acc = f.copy()
    term = f.copy()
    for _ in range(4):
        term = term - lat.dirac_full(u, term, 0, kappa)
        acc += term
    ref = lat.split(acc)[0]
    assert rel(net.apply(r), ref) < 1e-2


def test_preconditioner_gauge_covariance(env):
    lat, u, ctx, net = env
    net.init_neumann(0.125, noise=0.5, seed=3)
    rng = np.random.default_rng(50)
    V = lat.V
    gt = random_su3(V, rng)
    U = u.reshape(4, V, 3, 3, 2)
    Uc = U[..., 0] + 1j * U[..., 1]
    Ug = np.empty_like(Uc)
    for mu in range(4):
        fw = shift_index(DIMS, mu, +1)
        Ug[mu] = gt @ Uc[mu] @ np.conj(np.transpose(gt[fw], (0, 2, 1)))
    ug = np.stack([Ug.real, Ug.imag], axis=-1).ravel()
    e, o = lat.eo_tables()

    def rot_even(h):
        c = h.reshape(-1, 4, 3, 2)
        c = c[..., 0] + 1j * c[..., 1]
        r = np.einsum("xab,xsb->xsa", gt[e], c)
        return np.stack([r.real, r.imag], axis=-1).ravel()

    r = orc.gauss_field(lat.half_size, 9)
    z = net.apply(r)
    ctx2 = ii.Context(DIMS)
    try:
        ctx2.upload_gauge(ug)
        net2 = ii.LearnedPreconditioner(ctx2)
        for l in range(4):
            net2.set_weights(l, net.get_weights(l))
        z2 = net2.apply(rot_even(r))
    finally:
        ctx2.close()
    assert rel(z2, rot_even(z)) < 2e-2


def test_fgcr_plain_and_preconditioned(env):
    lat, u, ctx, net = env
    kappa = 0.125
    b = orc.gauss_field(lat.half_size, 11)
    res = {}
    for use_net in (False, True):
        if use_net:
            net.init_neumann(kappa, noise=0.0)
        x = np.empty_like(b)
        out = ii.Solver_FGCR(ctx, kappa, tol=1e-10, maxiter=500, nkrylov=16,
                             use_net=use_net).solve(x, b)
        true = rel(lat.dirac_eo(u, x, 0, kappa), b)
        assert true < 1e-10, (use_net, true)
        res[use_net] = out.Iterations
    assert res[True] < res[False], res


def test_training_reduces_loss_and_iterations(tmp_path):
    """Ablation on an 8^3x16 heat-bath field near kappa_c: the trained
    network lowers the loss below the Neumann start and the flexible GCR
    needs fewer directions with it than with no preconditioner."""
    dims = (8, 8, 8, 16)
    kappa = 0.1355
    ctx = ii.Context(dims)
    try:
        ctx.unit_gauge()
        ctx.heatbath(5.8, 99, 60)
        ctx.apply_apbc()
        net = ii.LearnedPreconditioner(ctx)
        rep = net.train(kappa, npairs=16, epochs=6, batch=4, lr=2e-3, pair_tol=1e-8, seed=5)
        assert rep["loss_last"] < rep["loss_first"], rep
        path = os.path.join(str(tmp_path), "net.bin")
        net.save(path)
        lat = orc.Lattice(dims)
        b = orc.gauss_field(lat.half_size, 12345)
        its = {}
        for use_net in (False, True):
            x = np.empty_like(b)
            out = ii.Solver_FGCR(ctx, kappa, tol=1e-10, maxiter=2000, nkrylov=16,
                                 use_net=use_net).solve(x, b)
            its[use_net] = out.Iterations
        assert its[True] < its[False], its
        z1 = net.apply(b)
        net.init_neumann(kappa)
        net.load(path)
        assert np.array_equal(net.apply(b), z1)
    finally:
        ctx.close()


@pytest.mark.parametrize("dims,nrhs", [((4, 4, 4, 8), 5), ((6, 2, 2, 6), 3), ((8, 8, 32, 32), 3)])
def test_batched_apply_vs_oracle(dims, nrhs):
    """ii_net_apply_batched (all rhs per launch; layers regrouped by parity
    with composite weights, e4m3 activation records and Y with one
    power-of-two scale per site and group of 8 channels or paths, bfloat16
    links, inputs, weights and transports) against Net.apply_device_form,
    the oracle of that evaluation step by step with the same roundings (only
    its sums are exact where the device's are FP32), and against the exact
    FP64 network; on a lattice whose half volume is a whole number of
    16-site tiles and on one that is not (6x2x2x6: 72 sites), and on
    8x8x32x32, where on a 256-CU device the blocks own several z-planes
    each, with the autotuned rhs grouping and three forced ones
    (bit-identical).
    Bounds: 1e-2 against the device form (measured 4e-8 to 4e-3: a rounding
    step that lands the other way because of the FP32 sums moves one value
    by a unit of its format); 5e-2 against the exact network (measured
    0.030-0.032: the e4m3 records, 4 significant bits).  A network with one
    transport path of one layer dropped is 0.17-0.19 from the device form,
    more than ten bounds."""
    lat = orc.Lattice(dims)
    u = lat.apbc(lat.gauge_expH(0.4, 77))
    ctx = ii.Context(dims)
    try:
        ctx.upload_gauge(u)
        net = ii.LearnedPreconditioner(ctx)
        net.init_neumann(0.13, noise=0.3, seed=5)
        ws = [net.get_weights(layer).astype(np.complex128) for layer in range(4)]
        rng = np.random.default_rng(3)
        b = rng.normal(size=(nrhs, lat.half_size))
        rg, report = net.tune(nrhs)
        print("autotuned rhs groups %s: %s" % (rg, report))
        assert all(1 <= v <= 12 for v in rg)
        got = net.apply_batched(b)
        single = np.stack([net.apply(b[k]) for k in range(nrhs)])
        ref = orc.Net(lat, u, ws)
        wrong = [w.copy() for w in ws]
        wrong[1][8] = 0.0
        bad = orc.Net(lat, u, wrong)
        want = [ref.apply(b[k]) for k in range(nrhs)]
        wantd = [ref.apply_device_form(b[k]) for k in range(nrhs)]
        for k in range(nrhs):
            ed, e = rel(got[k], wantd[k]), rel(got[k], want[k])
            print("rhs %d: vs device-form oracle %.2e, vs exact %.4f" % (k, ed, e))
            assert ed < 1e-2, (k, ed)
            assert e < 5e-2, (k, e)
            assert rel(got[k], single[k]) < 5e-2
            assert rel(bad.apply_device_form(b[k]), wantd[k]) > 1e-1
        # every grouping of the rhs gives the same result (the work order
        # changes, not the arithmetic of a site)
        for force in [(1, 1, 1, 1), (2, 3, 4, 12), (12, 6, 1, 2)]:
            net.tune(nrhs, force)
            assert np.array_equal(net.apply_batched(b), got), force
    finally:
        ctx.close()


def test_batched_apply_beyond_64_rhs():
    """Batches of more than 64 rhs take the stages' static work order (the
    work queues hold up to 64 live rhs): 66 rhs on 4^3x8 give, rhs by rhs,
    bitwise the result of a batch of 3 (dynamic order) for the rhs they
    share, and every rhs matches the device-form oracle."""
    dims = (4, 4, 4, 8)
    lat = orc.Lattice(dims)
    u = lat.apbc(lat.gauge_expH(0.4, 78))
    ctx = ii.Context(dims)
    try:
        ctx.upload_gauge(u)
        net = ii.LearnedPreconditioner(ctx)
        net.init_neumann(0.13, noise=0.3, seed=6)
        ws = [net.get_weights(layer).astype(np.complex128) for layer in range(4)]
        rng = np.random.default_rng(9)
        b = rng.normal(size=(66, lat.half_size))
        big = net.apply_batched(b)
        small = net.apply_batched(b[[0, 40, 65]])
        for k, j in enumerate((0, 40, 65)):
            assert np.array_equal(big[j], small[k]), j
        ref = orc.Net(lat, u, ws)
        worst = max(rel(big[j], ref.apply_device_form(b[j])) for j in (0, 13, 64, 65))
        print("66 rhs: max error against the device-form oracle %.2e" % worst)
        assert worst < 1e-2
    finally:
        ctx.close()


def _fgcr_setup(dims, kappa, seed=5):
    lat = orc.Lattice(dims)
    u = lat.apbc(lat.gauge_expH(0.6, seed))
    ctx = ii.Context(dims)
    ctx.upload_gauge(u)
    net = ii.LearnedPreconditioner(ctx)
    net.init_neumann(kappa, noise=0.05, seed=1)
    return lat, u, ctx, net


@pytest.mark.parametrize("use_net,use_graph,northo", [(True, False, 0), (False, False, 0),
                                                     (True, True, 0), (True, False, 3),
                                                     (True, True, 8)])
def test_fgcr_batched_point_sources(use_net, use_graph, northo):
    """The batched mixed-precision flexible GCR (every rhs per launch, FP32
    Krylov vectors, the network on bfloat16 activations, FP64 restarts): the
    12 point-source columns reach the full-operator true residual 1e-10
    (oracle) and the oracle's FP64 solution to 1e-8, with and without the
    network, with the restart cycle captured as a HIP graph, and with each
    direction orthogonalised against the previous one (default), three, or
    all of the cycle (the full GCR)."""
    dims, kappa = (8, 8, 8, 8), 0.1355
    lat, u, ctx, net = _fgcr_setup(dims, kappa)
    try:
        src = ii.DeviceField(ctx, "full", 12)
        sol = ii.DeviceField(ctx, "full", 12)
        src.point_sources((0, 0, 0, 0))
        outs = ii.PropagatorSolver(ctx, kappa, tol=1e-10, batched=True, method="fgcr",
                                   use_learned=use_net, use_graph=use_graph,
                                   nkrylov=8, northo=northo).solve(src, sol)
        print("fgcr net=%s graph=%s northo=%d: directions %s, cycles %s, fallback %s"
              % (use_net, use_graph, northo, [o.Iterations for o in outs],
                 [o.restarts for o in outs],
                 [o.inner_iterations for o in outs]))
        assert max(o.true_residual for o in outs) <= 1e-10
        for rhs in (0, 4, 11):
            b = src.download(rhs)
            x = sol.download(rhs)
            r = lat.true_residual_full(u, kappa, x, b)
            assert r <= 1e-10, (rhs, r)
            assert abs(outs[rhs].true_residual - r) < 1e-12
            xo, _ = lat.eo_invert(u, kappa, b, 1e-28, 5000)
            assert rel(x, xo) < 1e-8
    finally:
        ctx.close()


def test_fgcr_graph_equals_eager_and_network_saves_directions():
    """Graph replay of the restart cycle gives the eager solution bit for
    bit; the Neumann-initialised network needs fewer directions than the
    same flexible GCR without it; a ragged batch of 5 Gaussian sources."""
    dims, kappa = (8, 8, 8, 8), 0.1355
    lat, u, ctx, net = _fgcr_setup(dims, kappa, seed=8)
    try:
        src = ii.DeviceField(ctx, "full", 5)
        sol = ii.DeviceField(ctx, "full", 5)
        rng = np.random.default_rng(4)
        bs = [rng.normal(size=lat.full_size) for _ in range(5)]
        for k in range(5):
            src.upload(k, bs[k])
        runs = {}
        for name, net_on, graph in [("eager", True, False), ("graph", True, True),
                                    ("plain", False, False)]:
            outs = ii.PropagatorSolver(ctx, kappa, tol=1e-10, batched=True, method="fgcr",
                                       use_learned=net_on, use_graph=graph).solve(src, sol)
            runs[name] = (outs, [sol.download(k) for k in range(5)])
        for k in range(5):
            assert np.array_equal(runs["eager"][1][k], runs["graph"][1][k])
            assert lat.true_residual_full(u, kappa, runs["eager"][1][k], bs[k]) <= 1e-10
            assert lat.true_residual_full(u, kappa, runs["plain"][1][k], bs[k]) <= 1e-10
        d_net = max(o.Iterations for o in runs["eager"][0])
        d_plain = max(o.Iterations for o in runs["plain"][0])
        print("directions: network %d, none %d" % (d_net, d_plain))
        assert d_net < d_plain
    finally:
        ctx.close()


def test_loss_grad_of_pairs_in_arrays_of_their_own(env):
    """The same bits as the pairs back to back in one array."""
    import ctypes
    from iroiro_amd import _lib
    lat, u, ctx, net = env
    rng = np.random.default_rng(41)
    bs, ys = rng.normal(size=(2, 3, lat.half_size))
    loss, grads = net.loss_grad(list(bs), list(ys))
    f = np.empty(2 * sum(g.size for g in grads), np.float32)
    one = ctypes.c_double()
    assert _lib.load().ii_net_loss_grad(ctx.handle, 3, _lib.dptr(bs.ravel()),
                                        _lib.dptr(ys.ravel()), ctypes.byref(one),
                                        _lib.fptr(f)) == _lib.II_OK
    assert one.value == loss
    assert np.array_equal(f.view(np.complex64), np.concatenate([g.ravel() for g in grads]))
