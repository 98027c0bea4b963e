"""Workloads of the Wilson even/odd solve path, for timing and comparing builds.

Each case is one call (or one short chain of calls) of the public Python
interface, at sizes of this repository's configurations and at ragged ones:
operators and solvers on host arrays as the reference's Field interface hands
them over, the device-resident 12-column propagator with its contraction, the
rational (RHMC) solver, the two-flavour MD force and the network's gradient.

Gauge fields are U = exp(i eps H) with eps = 0.3 and H traceless Hermitian
Gaussian, reunitarised, antiperiodic in time; their average plaquette (0.6) is
that of a beta = 6 quenched field, and kappa = 0.1265 here takes about the
iterations that kappa = 0.1355 takes there (70 of CG, 30 of BiCGStab, 20 with
the network).
"""
import functools
import math

import numpy as np
import torch
import torch.utils.checkpoint

import iroiro_amd as ii

EPS = 0.3
WIDTHS = (1, 8, 8, 8, 1)


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one operator application from host code: the smallest call, all latency
        dict(name="dhat_4c8", kind="dhat", dims="4x4x4x8", kappa=0.12),
        # Fopr_DdagD inside a host-driven iteration (eigensolver, host CG)
        dict(name="ddagd_16c32", kind="ddagd", dims="16x16x16x32", kappa=0.1265),
        # a solve on a test-sized lattice: many short launches in a chain
        dict(name="cg_8c16", kind="cg", dims="8x8x8x16", kappa=0.1265),
        # Inverter_WilsonLike on a lattice whose rows fill no wavefront evenly
        dict(name="invert_12x10x14x18", kind="invert", dims="12x10x14x18", kappa=0.1265),
        # the reference's plain FP64 solve at a production size
        dict(name="cg_24c48", kind="cg", dims="24x24x24x48", kappa=0.1265),
        # RHMC Metropolis step, the reference's FP64 multishift recursion
        dict(name="rational_double_16c32", kind="rational", dims="16x16x16x32", kappa=0.1265,
             precision="double", degree=10),
        # the same step with the mixed-precision multishift
        dict(name="rational_half_24c48", kind="rational", dims="24x24x24x48", kappa=0.1265,
             precision="half", degree=10),
        # one MD force of two-flavour HMC: FP64 solve, force, projection
        dict(name="nf2_force_16c32", kind="nf2", dims="16x16x16x32", kappa=0.1265),
        # a 12-column propagator handed back to host code (saved or contracted there)
        dict(name="qprop_cg_single_12c24", kind="qprop", dims="12x12x12x24", kappa=0.1265,
             method="cg", precision="single", learned=False),
        # spectroscopy on the device: propagator, then the 18 meson correlators
        dict(name="mesons_bicgstab_half_24c48", kind="mesons", dims="24x24x24x48", kappa=0.1265,
             method="bicgstab", precision="half", learned=False, mode=0),
        # the headline solve: flexible GCR with the learned preconditioner, then the contraction
        dict(name="mesons_fgcr_learned_32c64", kind="mesons", dims="32x32x32x64", kappa=0.1265,
             method="fgcr", precision="half", learned=True, mode=0),
        # a minibatch of the network's training: forward, backward, weight gradients
        dict(name="net_grad_16c32", kind="net_grad", dims="16x16x16x32", kappa=0.1265, pairs=4),
    ]


#: smallest and largest volume a drawn case of each kind has
_RANGE = {
    "dhat": (512, 300000), "ddagd": (512, 700000), "cg": (512, 700000), "invert": (512, 300000),
    "rational": (2048, 700000), "nf2": (512, 300000), "qprop": (2048, 100000),
    "mesons": (4096, 700000), "net_grad": (512, 140000),
}


def draw(rng):
    kind = rng.choice(sorted(_RANGE))
    lo, hi = _RANGE[kind]
    target = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    while True:
        side = target ** 0.25
        d = [2 * max(2, int(round(0.5 * side * math.exp(rng.uniform(-0.35, 0.35))))) for _ in range(3)]
        d.append(2 * max(2, int(round(0.5 * target / (d[0] * d[1] * d[2])))))
        if lo <= d[0] * d[1] * d[2] * d[3] <= hi and d[3] <= 96:
            break
    c = dict(kind=kind, dims="x".join(map(str, d)), kappa=round(rng.uniform(0.118, 0.1275), 4))
    if kind == "rational":
        c.update(precision=rng.choice(["double", "single", "half"]), degree=rng.choice([6, 8, 10]))
    if kind in ("qprop", "mesons"):
        c.update(rng.choice([
            dict(method="cg", precision="single", learned=False),
            dict(method="cg", precision="half", learned=False),
            dict(method="bicgstab", precision="single", learned=False),
            dict(method="bicgstab", precision="half", learned=False),
            dict(method="bicgstab", precision="bf16", learned=False),
            dict(method="fgcr", precision="half", learned=False),
            dict(method="fgcr", precision="half", learned=True)]))
    if kind == "mesons":
        c.update(mode=rng.choice([0, 1, 2]))
    if kind == "net_grad":
        c.update(pairs=rng.choice([1, 2, 3, 4]))
    return c


def _dims(case):
    return tuple(int(v) for v in case["dims"].split("x"))


def _mom(case):
    d = _dims(case)
    return (2 * math.pi / d[0], 0.0, 2 * math.pi / d[2])


@functools.lru_cache(maxsize=None)
def _approx(degree):
    """x^(+-1/2) on the spectrum of Dhat^dag Dhat at these kappa: a program's plan."""
    return ii.RationalApprox(degree, degree, 1, 2, 50, 1e-3, 8.0)


# ------------------------------------------------------------------ the inputs
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(seed, part):
    g = torch.Generator(device=_device())
    g.manual_seed(1000003 * int(seed) + part)
    return g


def _cross(a, b):
    return torch.stack([a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2],
                        a[0] * b[1] - a[1] * b[0]])


def _links(dims, seed):
    """Links as [mu][row][col][T][Z][Y][X], complex128, time boundary included."""
    Lx, Ly, Lz, Lt = dims
    shape = (Lt, Lz, Ly, Lx)
    out = []
    for mu in range(4):
        r = torch.randn((9,) + shape, generator=_generator(seed, mu), device=_device(),
                        dtype=torch.float64)
        tr = (r[0] + r[1] + r[2]) / 3
        h = [[None] * 3 for _ in range(3)]
        for a in range(3):
            h[a][a] = torch.complex(r[a] - tr, torch.zeros_like(tr))
        for n, (a, b) in enumerate(((0, 1), (0, 2), (1, 2))):
            h[a][b] = torch.complex(r[3 + 2 * n], r[4 + 2 * n]) / math.sqrt(2)
            h[b][a] = h[a][b].conj()
        h = torch.stack([torch.stack([v.resolve_conj() for v in row]) for row in h])
        del r, tr
        u = torch.zeros_like(h)
        for a in range(3):
            u[a, a] = 1
        term = u.clone()
        for k in range(1, 17):  # exp(i eps H) as a series; the rows are made orthonormal below
            term = sum(term[:, b, None] * h[b] for b in range(3)) * (1j * EPS / k)
            u += term
        del h, term
        x, y = u[0], u[1]
        x = x / x.abs().square().sum(0).sqrt()
        y = y - x * (x.conj() * y).sum(0)
        y = y / y.abs().square().sum(0).sqrt()
        u = torch.stack([x, y, _cross(x, y).conj()])
        if mu == 3:
            u[:, :, -1] *= -1
        out.append(u.resolve_conj())
    return torch.stack(out)


def _host_links(u):
    """Format_G: [mu][site][row][col][re, im]."""
    v = u.permute(0, 3, 4, 5, 6, 1, 2).contiguous()
    return torch.view_as_real(v).reshape(-1).cpu().numpy()


def _even(dims):
    Lx, Ly, Lz, Lt = dims
    s = [torch.arange(n, device=_device()) for n in (Lt, Lz, Ly, Lx)]
    return (s[0][:, None, None, None] + s[1][:, None, None] + s[2][:, None] + s[3]) % 2 == 0


def _gauss(dims, seed, part, sites):
    """Host half field (esec order) or full field of unit Gaussians."""
    Lx, Ly, Lz, Lt = dims
    n = 24 * Lx * Ly * Lz * Lt // (2 if sites == "even" else 1)
    return torch.randn(n, generator=_generator(seed, 16 + part), device=_device(),
                       dtype=torch.float64).cpu().numpy()


def _site(dims, seed):
    r = np.random.default_rng(int(seed))
    return tuple(int(r.integers(n)) for n in dims)


def _pairs(case, seed):
    """Sources and targets of the network: y = b + a smooth part of b's size."""
    dims = _dims(case)
    bs = [_gauss(dims, seed, 2 * k, "even") for k in range(case["pairs"])]
    ys = [b + 0.3 * _gauss(dims, seed, 2 * k + 1, "even") for k, b in enumerate(bs)]
    return bs, ys


def _weights(kappa, seed):
    """A network near the truncated Neumann series of D^-1 (as training starts and
    ends), W[layer] complex64 [9][cout][cin][4][4]."""
    r = np.random.default_rng([int(seed), 77])
    g = _gamma_matrices()
    hop = np.zeros((9, 4, 4), complex)
    for mu in range(4):
        hop[2 * mu + 1] = kappa * (np.eye(4) - g[mu])
        hop[2 * mu + 2] = kappa * (np.eye(4) + g[mu])
    ws = []
    for l in range(4):
        cout, cin = WIDTHS[l + 1], WIDTHS[l]
        w = 0.02 * kappa * (r.standard_normal((9, cout, cin, 4, 4, 2)) @ np.array([1, 1j]))
        w[0, 0, 0] += np.eye(4)
        last = min(1, cin - 1)
        if cout > 1:
            w[0, 1, 0] += np.eye(4)
            w[:, 1, last] += hop
        else:
            w[:, 0, last] += hop
        ws.append(w.astype(np.complex64))
    return ws


def prepare(case, seed):
    dims, kind = _dims(case), case["kind"]
    mass = 0.5 / case["kappa"] - 4.0
    ctx = ii.Context(dims)
    D = ii.Dirac_Wilson_EvenOdd(mass, _host_links(_links(dims, seed)), ctx)
    torch.cuda.empty_cache()
    st = {"kind": kind, "case": case, "ctx": ctx, "D": D}
    if kind in ("dhat", "ddagd", "cg", "rational", "nf2"):
        st["b"] = _gauss(dims, seed, 0, "even")
    if kind == "ddagd":
        st["A"] = ii.Fopr_DdagD(D)
    if kind == "cg":
        st["solver"] = ii.Solver_CG(1e-20, 5000, ii.Fopr_DdagD(D))
        st["x"] = np.empty_like(st["b"])
    if kind == "invert":
        st["b"] = _gauss(dims, seed, 0, "full")
        st["x"] = np.empty_like(st["b"])
        st["solver"] = ii.Inverter_WilsonLike(D, ii.Solver_CG(1e-20, 5000, ii.Fopr_DdagD(D)))
    if kind == "rational":
        stop = 1e-20 if case["precision"] == "double" else 1e-10
        st["solver"] = ii.RationalSolver_CG(ii.MultiShiftSolver_CG(ii.Fopr_DdagD(D), stop, 5000),
                                            _approx(case["degree"]), precision=case["precision"])
        st["x"] = np.empty_like(st["b"])
    if kind == "nf2":
        st["action"] = ii.Action_Nf2(D, ii.Solver_CG(1e-20, 5000, ii.Fopr_DdagD(D)))
        st["action"].set_phi(st["b"])
    if kind in ("qprop", "mesons"):
        if case["learned"]:
            net = ii.LearnedPreconditioner(ctx)
            for l, w in enumerate(_weights(case["kappa"], seed)):
                net.set_weights(l, w)
        st["src"], st["sol"] = ii.DeviceField(ctx, "full", 12), ii.DeviceField(ctx, "full", 12)
        st["src"].point_sources(_site(dims, seed))
        st["solver"] = ii.PropagatorSolver(ctx, case["kappa"], tol=1e-10,
                                           precision=case["precision"], batched=True,
                                           method=case["method"], use_learned=case["learned"],
                                           use_graph=case["method"] == "fgcr")
    if kind == "net_grad":
        st["net"] = ii.LearnedPreconditioner(ctx)
        for l, w in enumerate(_weights(case["kappa"], seed)):
            st["net"].set_weights(l, w)
        st["bs"], st["ys"] = _pairs(case, seed)
    return st


# ------------------------------------------------------------------ one pass
def run(st):
    kind = st["kind"]
    if kind == "dhat":
        return st["D"].mult(st["b"])
    if kind == "ddagd":
        return st["A"].mult(st["b"])
    if kind == "cg":
        st["solver"].solve(st["x"], st["b"])
        return st["x"]
    if kind == "invert":
        st["solver"].invert(st["x"], st["b"])
        return st["x"]
    if kind == "rational":
        st["solver"].solve_inv(st["x"], st["b"])
        return st["x"]
    if kind == "nf2":
        return st["action"].md_force()
    if kind == "qprop":
        st["solver"].solve(st["src"], st["sol"])
        return [st["sol"].download(k) for k in range(12)]
    if kind == "mesons":
        st["solver"].solve(st["src"], st["sol"])
        return ii.meson_correlators(st["ctx"], st["sol"], st["sol"], st["case"]["mode"], 3,
                                    _mom(st["case"]))
    loss, grads = st["net"].loss_grad(st["bs"], st["ys"])
    return {"loss": loss, "grads": grads}


# ------------------------------------------------------------------ what a pass needs
#: CG iterations to |r|^2/|b|^2 = 1e-20 at these kappa (each four hops), and the hops on one
#: column that the other methods need to the same residual
_CG_ITERATIONS = 70
_COLUMN_HOPS = {"cg": 4 * 70, "bicgstab": 4 * 30, "fgcr": 2 * 53}


def work(case):
    dims, kind = _dims(case), case["kind"]
    v = dims[0] * dims[1] * dims[2] * dims[3]
    half, links = 96.0 * v, 576.0 * v   # bytes: an FP64 half field, the FP64 links
    hop = 1320.0 * v / 2                # flops of one hop
    # FP64 solves: a hop reads every link, a half field and writes one; a CG step has six
    # vector reads and three writes besides
    hop64 = links + 2 * half
    it64 = 4 * hop64 + 9 * half
    if kind == "dhat":
        return {"bytes": links + 2 * half, "flops": 2 * hop}
    if kind == "ddagd":
        return {"bytes": links + 2 * half, "flops": 4 * hop}
    if kind in ("cg", "invert"):
        return {"bytes": _CG_ITERATIONS * it64 + 4 * half, "flops": _CG_ITERATIONS * 4 * hop}
    if kind == "nf2":
        return {"bytes": _CG_ITERATIONS * it64 + 2 * links + 4 * half,
                "flops": _CG_ITERATIONS * 4 * hop}
    if kind == "rational":
        n, it, real = case["degree"], 0.6 * _CG_ITERATIONS, 8 if case["precision"] == "double" else 4
        return {"bytes": it * (it64 + 4 * n * half) * real / 8, "flops": it * 4 * hop}
    if kind in ("qprop", "mesons"):
        real = 2 if case["precision"] == "half" and case["method"] != "fgcr" else 4
        if case["precision"] == "bf16":
            real = 2
        n = _COLUMN_HOPS[case["method"]] * (0.4 if case["learned"] else 1.0)
        b = n * (links * 2 / 3 + 12 * 2 * half) * real / 8 + 24 * half
        f = n * 12 * hop
        if case["learned"]:  # each direction: one evaluation on 12 columns, 8-channel e4m3 records
            b += n / 2 * 12 * (v / 2) * 2112.0
            f += n / 2 * 12 * (v / 2) * 2 * 9 * 3 * 16 * 16 * 8.0
        return {"bytes": b, "flops": f}
    # network: per pair the four layers, their adjoints and the weight gradients; each FP32
    # activation written once and read by the next layer and by its weight gradient
    n = case["pairs"]
    macs = 9 * 3 * 16 * (8 + 64 + 64 + 8)
    return {"bytes": n * v * 96.0 * (1 + 8 * 3 * 3 + 8 * 3 * 2), "flops": n * v * macs * 8.0 * 3}


def tolerance(case):
    kind = case["kind"]
    if kind in ("dhat", "ddagd"):
        return {"rel": 1e-14, "max": 1e-12}
    # solves stop at a residual of 1e-10: the solution is 3e-10 to 5e-10 off exact(), on the
    # side that its own roundings take it, in the largest component by up to ten times that
    if kind in ("cg", "invert", "nf2", "qprop"):
        return {"rel": 2e-9, "max": 1e-7}
    # the same, damped by the sum over poles or over a time slice
    if kind in ("rational", "mesons"):
        return {"rel": 1e-9, "max": 1e-7}
    # bfloat16 operands: 2e-2 off exact(); a transported value whose FP32 rounding differs in
    # the last bit may round to the other bfloat16 neighbour
    return {"rel": 1e-2, "max": 1e-1}


# ------------------------------------------------------------------ the same in 64 bits
# Fields here are [n][spin][colour][T][Z][Y][X] complex128, links as _links() makes them.
def _gamma_tables():
    return [([3, 2, 1, 0], [-1j, -1j, 1j, 1j]), ([3, 2, 1, 0], [-1, 1, 1, -1]),
            ([2, 3, 0, 1], [-1j, 1j, 1j, -1j]), ([0, 1, 2, 3], [1, 1, -1, -1])]


def _gamma_matrices():
    out = []
    for idx, fac in _gamma_tables():
        m = np.zeros((4, 4), complex)
        for s in range(4):
            m[s, idx[s]] = fac[s]
        out.append(m)
    return out


def _spin(f, mu):
    """gamma_mu f."""
    idx, fac = _gamma_tables()[mu]
    return torch.stack([f[:, i] * c for i, c in zip(idx, fac)], 1)


def _colour(u, f, dag):
    """u f (or u^dag f) at every site."""
    m = u.transpose(0, 1).conj().resolve_conj() if dag else u
    return torch.stack([m[a, 0] * f[:, :, 0] + m[a, 1] * f[:, :, 1] + m[a, 2] * f[:, :, 2]
                        for a in range(3)], 2)


def _move(u, f, mu, forward):
    """U_mu(x) f(x + mu), or U_mu(x - mu)^dag f(x - mu)."""
    axis = -1 - mu
    if forward:
        return _colour(u[mu], torch.roll(f, -1, axis), False)
    return torch.roll(_colour(u[mu], f, True), 1, axis)


def _hop(u, f):
    out = None
    for mu in range(4):
        a, b = _move(u, f, mu, True), _move(u, f, mu, False)
        t = a + b - _spin(a - b, mu)
        out = t if out is None else out + t
    return out


def _g5(f):
    return torch.roll(f, 2, 1)


def _dhat(u, k, f, dag=False):
    """On fields that vanish on odd sites."""
    if dag:
        return _g5(_dhat(u, k, _g5(f)))
    return f - k * k * _hop(u, _hop(u, f))


def _from_half(dims, b):
    Lx, Ly, Lz, Lt = dims
    f = torch.zeros((Lt, Lz, Ly, Lx, 4, 3), dtype=torch.complex128, device=_device())
    f[_even(dims)] = torch.view_as_complex(
        torch.as_tensor(b, device=_device()).reshape(-1, 4, 3, 2).contiguous())
    return f.permute(4, 5, 0, 1, 2, 3)[None].contiguous()


def _to_host(f, keep=None):
    v = f[0].permute(2, 3, 4, 5, 0, 1).contiguous()
    v = v[keep] if keep is not None else v
    return torch.view_as_real(v.contiguous()).reshape(-1).cpu().numpy()


def _norms(f):
    return f.abs().square().flatten(1).sum(1)


def _cg(op, b, tol=1e-14):
    """Conjugate gradients for each of n systems at once."""
    x, r, p = torch.zeros_like(b), b.clone(), b.clone()
    rr = _norms(r)
    stop = tol * tol * rr
    view = (-1,) + (1,) * (b.dim() - 1)
    for _ in range(2000):
        if bool((rr <= stop).all()):
            break
        ap = op(p)
        alpha = rr / (p.conj() * ap).real.flatten(1).sum(1)
        alpha = torch.where(rr <= stop, torch.zeros_like(alpha), alpha)
        x += alpha.view(view) * p
        r -= alpha.view(view) * ap
        new = _norms(r)
        p = r + (new / rr).view(view) * p
        rr = new
    return x


def _traceless_antihermitian(m):
    """On [mu][row][col][...]."""
    a = (m - m.transpose(1, 2).conj()) / 2
    tr = (a[:, 0, 0] + a[:, 1, 1] + a[:, 2, 2]) / 3
    for k in range(3):
        a[:, k, k] -= tr
    return a


def _propagator(u, dims, kappa, site):
    b = torch.zeros((12, 4, 3, dims[3], dims[2], dims[1], dims[0]), dtype=torch.complex128,
                    device=_device())
    x, y, z, t = site
    for s in range(4):
        for c in range(3):
            b[3 * s + c, s, c, t, z, y, x] = 1

    def d(f, dag):
        if dag:
            return _g5(d(_g5(f), False))
        return f - kappa * _hop(u, f)
    return _cg(lambda f: d(d(f, False), True), d(b, True))


#: the two gamma structures of each of the 18 channels: per spin its partner and the factor
_UNIT, _G5 = ([0, 1, 2, 3], [1, 1, 1, 1]), ([2, 3, 0, 1], [1, 1, 1, 1])
_GM = [([3, 2, 1, 0], [-1j, -1j, 1j, 1j]), ([3, 2, 1, 0], [-1, 1, 1, -1]),
       ([2, 3, 0, 1], [-1j, 1j, 1j, -1j]), ([0, 1, 2, 3], [1, 1, -1, -1])]
_GM5 = [([1, 0, 3, 2], [-1j, -1j, 1j, 1j]), ([1, 0, 3, 2], [-1, 1, 1, -1]),
        ([0, 1, 2, 3], [-1j, 1j, 1j, -1j]), ([2, 3, 0, 1], [1, 1, -1, -1])]
_SG5 = [([2, 3, 0, 1], [1j, -1j, 1j, -1j]), ([3, 2, 1, 0], [1, -1, 1, -1]),
        ([1, 0, 2, 3], [1, 1, 1, 1]), ([3, 2, 1, 0], [1j, 1j, 1j, 1j]),
        ([1, 0, 3, 2], [1, -1, 1, -1]), ([0, 1, 2, 3], [1j, -1j, 1j, -1j])]
_CHANNELS = ([(_UNIT, _UNIT), (_G5, _G5)] + [(g, g) for g in _GM5] + [(g, g) for g in _GM] +
             [(g, g) for g in _SG5] + [(_GM[3], _UNIT), (_UNIT, _GM[3])])


def _correlators(q, dims, mode, mom):
    q = q.reshape((4, 3) + q.shape[1:])  # [source spin][source colour][spin][colour][T][Z][Y][X]
    pair = {}

    def prod(s1, s2, s4, s3):
        if (s1, s2, s4, s3) not in pair:
            pair[s1, s2, s4, s3] = (q[s1, :, s2].conj() * q[s4, :, s3]).sum((0, 1))
        return pair[s1, s2, s4, s3]
    z, y, x = (torch.arange(n, device=q.device, dtype=torch.float64) for n in dims[2::-1])
    ph = mom[0] * x + (mom[1] * y)[:, None] + (mom[2] * z)[:, None, None]
    cs = torch.cos(mom[0] * x) * torch.cos(mom[1] * y)[:, None] * torch.cos(mom[2] * z)[:, None, None]
    out = []
    for (i1, f1), (i2, f2) in _CHANNELS:
        v = torch.zeros(q.shape[4:], dtype=torch.complex128, device=q.device)
        for s4 in range(4):
            for s2 in range(4):
                gf = (f2[s4] * f1[s2])
                gf = gf.real if isinstance(gf, complex) else gf
                if gf:
                    v += gf * prod(i2[s4], s2, s4, i1[s2])
        if mode == 0:
            c = v.real.sum((1, 2, 3))
        elif mode == 1:
            c = torch.view_as_real((v * torch.polar(torch.ones_like(ph), ph)).sum((1, 2, 3))).reshape(-1)
        else:
            c = (v.real * cs).sum((1, 2, 3))
        out.append(c.cpu().numpy())
    return np.stack(out)


def _loss_grad(u, dims, ws, bs, ys):
    w = [torch.as_tensor(x.astype(np.complex128), device=_device()).requires_grad_() for x in ws]
    even, total = _even(dims), 0.0

    def layer(f, wl):
        cout, cin = wl.shape[1], wl.shape[2]
        out = None
        for d in range(9):
            t = f if d == 0 else _move(u, f, (d - 1) // 2, (d - 1) % 2 == 0)
            m = wl[d].permute(0, 2, 1, 3).reshape(4 * cout, 4 * cin)
            o = m @ t.reshape(4 * cin, -1)
            out = o if out is None else out + o
        return out.reshape((cout, 4) + tuple(f.shape[2:]))
    for b, y in zip(bs, ys):
        f, want = _from_half(dims, b), _from_half(dims, y)
        for wl in w:
            f = torch.utils.checkpoint.checkpoint(layer, f, wl, use_reentrant=False)
        loss = ((f - want).abs().square() * even).sum() / want.abs().square().sum()
        loss.backward()
        total += float(loss.detach())
    return {"loss": total, "grads": [x.grad.cpu().numpy() for x in w]}


def exact(case, seed):
    dims, kind, k = _dims(case), case["kind"], case["kappa"]
    v = dims[0] * dims[1] * dims[2] * dims[3]
    if kind in ("qprop", "mesons") and v > 700000:
        return None
    u = _links(dims, seed)
    even = _even(dims)
    if kind in ("qprop", "mesons"):
        q = _propagator(u, dims, k, _site(dims, seed))
        if kind == "qprop":
            return [_to_host(q[c:c + 1]) for c in range(12)]
        return _correlators(q, dims, case["mode"], _mom(case))
    if kind == "net_grad":
        return _loss_grad(u, dims, _weights(k, seed), *_pairs(case, seed))
    if kind == "invert":
        b = torch.as_tensor(_gauss(dims, seed, 0, "full"), device=_device())
        b = torch.view_as_complex(b.reshape(dims[3], dims[2], dims[1], dims[0], 4, 3, 2))
        b = b.permute(4, 5, 0, 1, 2, 3)[None].contiguous()
        be, bo = b * even, b * ~even
        xe = _cg(lambda f: _dhat(u, k, _dhat(u, k, f), True),
                 _dhat(u, k, be + k * _hop(u, bo), True))
        return _to_host(xe + bo + k * _hop(u, xe))
    b = _from_half(dims, _gauss(dims, seed, 0, "even"))
    if kind == "dhat":
        return _to_host(_dhat(u, k, b), even)

    def op(f):
        return _dhat(u, k, _dhat(u, k, f), True)
    if kind == "ddagd":
        return _to_host(op(b), even)
    if kind == "cg":
        return _to_host(_cg(op, b), even)
    if kind == "rational":
        ra = _approx(case["degree"])
        x = b * ra.InvConst()
        for res, pole in zip(ra.InvResiduals(), ra.InvPoles()):
            x += float(res) * _cg(lambda f: op(f) + float(pole) * f, b)
        return _to_host(x, even)
    # two-flavour force: the derivative of Re <zeta, Dhat eta> along U -> (1 + eps X) U
    # is Re tr(X F), with eta = (Dhat^dag Dhat)^-1 phi and zeta = Dhat eta
    eta = _cg(op, b)
    zeta = _dhat(u, k, eta)
    uu = u.clone().requires_grad_()
    s = (zeta.conj() * _dhat(uu, k, eta)).real.sum()
    g, = torch.autograd.grad(s, uu)
    with torch.no_grad():
        f = torch.stack([torch.stack([
            sum(u[:, a, c] * g[:, b2, c].conj() for c in range(3)) for b2 in range(3)], 1)
            for a in range(3)], 1)
        f = _traceless_antihermitian(f)
    return torch.view_as_real(f.permute(0, 3, 4, 5, 6, 1, 2).contiguous()).reshape(-1).cpu().numpy()
