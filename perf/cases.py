"""The work that programs built on yahmc_amd have it do, as cases that can be
timed and checked: solves of the even/odd Wilson-clover operator, rational
functions of it, molecular dynamics of the gauge field, HMC steps and
trajectories, meson correlators, and the learned preconditioner.

A case is a dict of plain values.  listed() names the ones to follow over
time, draw() gives more of the same ranges, prepare() makes what a program
holds before the call (a lattice context with links near those of a
thermalised field, plaquette about 0.6, sources, page-locked host buffers),
run() is one pass, and exact() restates the pass in 64-bit torch."""
import ctypes
import math

import numpy as np
import torch

import yahmc_amd as yh
from yahmc_amd import hmc, md, spectrum

DEV = "cuda"
CSW = 1.0
BETA = 5.6
# algebra width of the links: the mean plaquette comes out at 0.55 to 0.65
EPS = {2: 0.27, 3: 0.21, 4: 0.18}
# model -> (nc, representation, D_R, mass)
MODELS = {
    "su3": (3, "fundamental", 3, -0.2),
    "su2": (2, "fundamental", 2, -0.1),
    "su4": (4, "fundamental", 4, -0.2),
    "su2_adj": (2, "adjoint", 3, -0.5),
    "su3_sym": (3, "symmetric", 6, -0.4),
}


def _case(name, kind, model, dims, **more):
    c = {"kind": kind, "model": model, "T": dims[0], "X": dims[1], "Y": dims[2], "Z": dims[3], **more}
    return {"name": name, **c} if name else c


def listed():
    return [
        # the smallest call: a solve on a test lattice, where launches and waits count
        _case("solve_f64_8x4", "solve", "su3", (8, 4, 4, 4), solver="f64", bc="antiperiodic"),
        # the reference's own solver, double precision throughout, on the bench lattice
        _case("solve_f64_32x32", "solve", "su3", (32, 32, 32, 32), solver="f64", bc="antiperiodic"),
        # the production solve: 16-bit inner operator under FP64 reliable updates
        _case("solve_mixed16_32x32", "solve", "su3", (32, 32, 32, 32), solver="f16", bc="antiperiodic"),
        # FP32 inner operator, two colours, extents that divide nothing, open time boundary
        _case("solve_mixed32_ragged", "solve", "su2", (26, 14, 10, 18), solver="f32", bc="open"),
        # RHMC: x^(-1/2) of the operator by a 12-pole multishift solve, SU(2) adjoint
        _case("rational_su2adj_48x24", "rational", "su2_adj", (48, 24, 24, 24), poles=12),
        # spectroscopy: 12 point-source propagators and their 16 meson channels
        _case("mesons_32x16", "mesons", "su3", (32, 16, 16, 16), tau=3),
        # pure-gauge trajectories: the MD of a quenched run and of every thermalisation
        _case("md_wilson_32x16", "md", "su3", (32, 16, 16, 16), c0=1.0, steps=10),
        # the same with the Symanzik-improved action
        _case("md_improved_16x12", "md", "su3", (16, 12, 12, 12), c0=5.0 / 3.0, steps=4),
        # leapfrog steps of two-flavour HMC apart from their solves: fermion, clover, log-det and gauge
        # forces, link update, new represented links and clover term
        _case("step_su3_32x32", "step", "su3", (32, 32, 32, 32), steps=4),
        # the same for two-index symmetric quarks
        _case("step_sextet_32x24", "step", "su3_sym", (32, 24, 24, 24), steps=2),
        # a whole two-flavour HMC trajectory on a small lattice, from a given configuration
        _case("hmc_16x8", "hmc", "su3", (16, 8, 8, 8), steps=4, sloppy="f16"),
        # one training evaluation of the learned preconditioner, 1-8-8-1 channels: loss and weight gradients
        _case("net_train_16x16", "train", "su3", (16, 16, 16, 16), width=8, pairs=2),
    ]


def _dims_for(rng, lo, hi):
    """Even extents with a volume spread over [lo, hi] by its logarithm."""
    while True:
        v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
        side = v ** 0.25
        d = [max(4, 2 * round(side * math.exp(rng.uniform(-0.4, 0.4)) / 2)) for _ in range(4)]
        if lo <= math.prod(d) <= hi:
            return tuple(sorted(d, reverse=True)) if rng.random() < 0.5 else tuple(d)


def draw(rng):
    kind = rng.choice(["solve", "solve", "rational", "mesons", "md", "md", "step", "step", "hmc", "train"])
    if kind == "solve":
        return _case(None, kind, rng.choice(["su3", "su3", "su2", "su4", "su2_adj", "su3_sym"]),
                     _dims_for(rng, 512, 400000), solver=rng.choice(["f64", "f32", "f16"]),
                     bc=rng.choice(["antiperiodic", "periodic", "open"]))
    if kind == "rational":
        return _case(None, kind, rng.choice(["su2_adj", "su3", "su2"]), _dims_for(rng, 512, 400000),
                     poles=rng.choice([8, 10, 12]))
    if kind == "mesons":
        dims = _dims_for(rng, 512, 60000)
        return _case(None, kind, rng.choice(["su3", "su2"]), dims, tau=rng.randrange(dims[0]))
    if kind == "md":
        return _case(None, kind, rng.choice(["su3", "su3", "su2", "su4"]), _dims_for(rng, 512, 200000),
                     c0=rng.choice([1.0, 1.0, 5.0 / 3.0]), steps=rng.choice([2, 4, 8]))
    if kind == "step":
        return _case(None, kind, rng.choice(["su3", "su2", "su2_adj", "su3_sym"]), _dims_for(rng, 512, 400000),
                     steps=rng.choice([1, 2, 4]))
    if kind == "hmc":
        return _case(None, kind, rng.choice(["su3", "su2"]), _dims_for(rng, 512, 8192), steps=rng.choice([2, 4]),
                     sloppy=rng.choice(["f32", "f16"]))
    # activations are tiled by 32 sites
    while True:
        dims = _dims_for(rng, 512, 70000)
        if math.prod(dims) % 32 == 0:
            return _case(None, kind, "su3", dims, width=rng.choice([4, 8]), pairs=rng.choice([1, 2]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _geom(case):
    dims = (case["T"], case["X"], case["Y"], case["Z"])
    nc, rep, dr, mass = MODELS[case["model"]]
    return dims, math.prod(dims), nc, rep, dr, mass


def _gen(seed, what):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + what)
    return g


def _links(case, seed):
    """(4V, N, N) complex128 SU(N) links exp(i eps A), A Gaussian, traceless Hermitian."""
    _, V, nc, _, _, _ = _geom(case)
    a = torch.randn(4 * V, nc, nc, dtype=torch.complex128, device=DEV, generator=_gen(seed, 1))
    a = a - a.mH
    a = EPS[nc] * (a - torch.diag_embed((torch.diagonal(a, dim1=-2, dim2=-1).sum(-1, keepdim=True) / nc).expand(-1, nc)))
    u = torch.eye(nc, dtype=a.dtype, device=DEV).expand_as(a)
    for k in range(24, 0, -1):  # Taylor series by Horner's rule
        u = torch.eye(nc, dtype=a.dtype, device=DEV) + _mm(a, u) / k
    return u


def _split(z):
    """complex (..., n, m) -> (rows, 2 n m) doubles, all real parts then all imaginary parts"""
    z = z.reshape(z.shape[0], -1)
    return torch.cat([z.real, z.imag], 1).cpu().numpy()


def _spinor(case, seed, what, even_only=True):
    """(V, 4, D) complex128 Gaussian source, zero on the odd half"""
    dims, V, _, _, dr, _ = _geom(case)
    s = torch.randn(V, 4, dr, dtype=torch.complex128, device=DEV, generator=_gen(seed, what))
    if even_only:
        s[V // 2:] = 0
    if case.get("bc") == "open":
        s = s * _bc_mask(case)[_lex_of(dims)].reshape(V, 1, 1)
    return s


def _spinor_host(s):
    return _split(s.transpose(1, 2))  # re[D][4], im[D][4]


def _pinned(*shape):
    return torch.zeros(*shape, dtype=torch.float64, pin_memory=True).numpy()


def _momenta(case, seed):
    _, V, nc, _, _, _ = _geom(case)
    return math.sqrt(0.5) * torch.randn(4 * V, nc * nc - 1, dtype=torch.float64, device=DEV, generator=_gen(seed, 5))


def _weights(case, seed):
    """weights (9, out, in, 4, 4) per layer: small random plus the identity on path 0"""
    g = np.random.default_rng(7 + int(seed))
    ch = (1, case["width"], case["width"], 1)
    out = []
    for ci, co in zip(ch[:-1], ch[1:]):
        w = 0.1 * (g.normal(size=(9, co, ci, 4, 4)) + 1j * g.normal(size=(9, co, ci, 4, 4))) / np.sqrt(36 * ci)
        for k in range(min(ci, co)):
            w[0, k, k] += 0.5 * np.eye(4)
        out.append(w)
    return out


def prepare(case, seed):
    dims, V, nc, rep, dr, mass = _geom(case)
    lat = yh.Lattice(dims, nc=nc, repr=rep, bc=case.get("bc", "antiperiodic"), csw=CSW)
    lat.set_gauge(_split(_links(case, seed)))
    if lat.bc == yh.BC["open"]:
        lat.apply_bcs_on_gauge_field()
        lat.represent_gauge_field()
    s = {"case": case, "lat": lat, "mass": mass}
    kind = case["kind"]
    if kind in ("solve", "rational"):
        s["b"] = lat.field("f64").upload(_spinor_host(_spinor(case, seed, 2)))
        s["x"] = lat.field("f64")
        s["out"] = _pinned(V, 8 * dr)
        if kind == "rational":
            s["rat"] = yh.rational_zolotarev(case["poles"], -1, 2, 1e-2, 64.0)
    elif kind in ("md", "step"):
        lat.set_momenta(_momenta(case, seed).cpu().numpy())
        s["links"], s["mom"] = _pinned(4 * V, 2 * nc * nc), _pinned(4 * V, nc * nc - 1)
        s["gauge"] = hmc.GaugeMonomial(BETA, c0=case.get("c0", 1.0))
        if kind == "step":
            s["x"] = lat.field("f64").upload(_spinor_host(_spinor(case, seed, 2)))
    elif kind == "hmc":
        s["links"] = _pinned(4 * V, 2 * nc * nc)
        s["start"] = lat.get_gauge()
        s["fermion"] = hmc.FermionMonomial(mass, prec=1e-26, sloppy=case["sloppy"])
        s["hmc"] = hmc.HMC(lat, [hmc.GaugeMonomial(BETA), s["fermion"]], [("o2mn", 2), ("o2mn", case["steps"])])
        s["rng"] = np.random.default_rng(int(seed))
    elif kind == "train":
        s["net"] = yh.Net(lat, (1, case["width"], case["width"], 1))
        s["net"].set_weights(_weights(case, seed))
        # (H^2 v, v) pairs
        s["xs"] = [lat.field("f64").upload(_spinor_host(_spinor(case, seed, 20 + k))) for k in range(case["pairs"])]
        s["bs"] = [lat.field("f64") for _ in s["xs"]]
        for b, x in zip(s["bs"], s["xs"]):
            lat.Hphi_sq(mass, b, x)
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _ptr(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def _ok(rc):
    if rc != yh.YH_OK:
        raise yh.YahmcError(rc, yh.lib().yh_last_error().decode())


def _even(s, field):
    """the even half of a field, in the program's page-locked buffer"""
    lat, out = s["lat"], s["out"]
    _ok(yh.lib().yh_field_download(lat.ctx, field.h, _ptr(out), yh.EVEN))
    return out[: lat.VH]


def _gauge_out(s):
    _ok(yh.lib().yh_get_gauge(s["lat"].ctx, _ptr(s["links"])))
    return s["links"]


def _momenta_out(s):
    _ok(yh.lib().yh_get_momenta(s["lat"].ctx, _ptr(s["mom"])))
    return s["mom"]


def _solve(s):
    lat, x, b = s["lat"], s["x"], s["b"]
    solver = s["case"]["solver"]
    x.zero(yh.EVEN)
    if solver == "f64":
        lat.cg_inverter(lat.inv_par(s["mass"], 1e-20, max_iter=5000), x, b)
    else:
        lat.cg_mixed(lat.inv_par(s["mass"], 1e-20, sloppy=solver, reliable_every=50, max_iter=5000), x, b)
    return _even(s, x)


def _rational(s):
    lat = s["lat"]
    lat.rational_calc(s["rat"], lat.inv_par(s["mass"], 1e-20), s["x"], s["b"])
    return _even(s, s["x"])


def _mesons(s):
    got = spectrum.meson_measure(s["lat"], s["mass"], 1e-20, 1, spectrum.POINT, np.random.default_rng(0),
                                 taus=[s["case"]["tau"]])
    return {k: got[k] for k in spectrum.CHANNELS}


def _md(s):
    """a trajectory of o2mn from the current links and momenta"""
    lat, g, steps = s["lat"], s["gauge"], s["case"]["steps"]
    a, dt = md.O2MN_LAMBDA, 0.1
    for n in range(steps):
        g.update(lat, (a if n == 0 else 2 * a) * dt)
        lat.update_links(dt / 2)
        g.update(lat, (1 - 2 * a) * dt)
        lat.update_links(dt / 2)
    g.update(lat, a * dt)
    return [_gauge_out(s), _momenta_out(s)]


STEP_DT = 0.01


def _step(s):
    """leapfrog steps with a given solution of the fermions' system"""
    lat = s["lat"]
    for _ in range(s["case"]["steps"]):
        lat.begin_fermion_force()
        lat.wilson_fermion_force_q(STEP_DT, s["mass"], 1.0, s["x"])
        lat.clover_logdet_force(s["mass"], 2.0)
        lat.end_fermion_force(STEP_DT)
        s["gauge"].update(lat, STEP_DT)
        lat.update_links(STEP_DT)
        lat.represent_gauge_field()
    return [_gauge_out(s), _momenta_out(s)]


def _hmc(s):
    s["lat"].set_gauge(s["start"])
    rec = s["hmc"].trajectory(s["rng"], length=0.4, metropolis=False)
    return {"dH": rec["dH"], "plaquette": rec["plaquette"], "links": _gauge_out(s)}


def _train(s):
    loss, grads = s["net"].loss_grad(s["bs"], s["xs"])
    return {"loss": loss, "grads": grads}


RUN = {"solve": _solve, "rational": _rational, "mesons": _mesons, "md": _md, "step": _step, "hmc": _hmc,
       "train": _train}


def run(state):
    return RUN[state["case"]["kind"]](state)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
# iterations that the solves take at the masses above (they grow slowly with
# the lattice); a solver's start and its reliable updates are left out
SOLVE_ITERS = {"su3": 130, "su2": 100, "su4": 115, "su2_adj": 85, "su3_sym": 70}


def _op_cost(case, prec):
    """(bytes, flops) of one H^2 over the lattice: four hops of V/2 output sites, each reading its links, one
    spinor (two with the clover term), a clover block and writing one spinor"""
    _, V, _, _, d, _ = _geom(case)
    sb = {"f64": 64, "f32": 32, "f16": 16}[prec] * d + (4 if prec == "f16" else 0)
    rows = 2 if case["model"] == "su3" and prec != "f64" else d
    lb = {"f64": 16, "f32": 8, "f16": 4}[prec] * rows * d
    cb = {"f64": 64, "f32": 32, "f16": 16}[prec] * d * d + (8 if prec == "f16" else 0)
    flops = 8 * (2 * d * (8 * d - 2) + 12 * d) + 2 * 8 * (2 * d) ** 2
    return V // 2 * (4 * (8 * lb + cb) + 10 * sb), V // 2 * 4 * flops


def _cg_cost(case, prec, iters):
    """H^2 and the two vector updates of a CG iteration"""
    _, V, _, _, d, _ = _geom(case)
    b, f = _op_cost(case, prec)
    xr = 64 if prec == "f64" else 32
    pq = {"f64": 64, "f32": 32, "f16": 16}[prec]
    return iters * (b + V // 2 * d * (5 * xr + 4 * pq)), iters * (f + V // 2 * d * 100)


def work(case):
    _, V, nc, _, d, _ = _geom(case)
    kind = case["kind"]
    ng, lk = nc * nc - 1, 16 * nc * nc
    if kind == "solve":
        b, f = _cg_cost(case, case["solver"], SOLVE_ITERS[case["model"]])
    elif kind == "rational":
        n, it = case["poles"], SOLVE_ITERS[case["model"]]
        b, f = _op_cost(case, "f64")
        b, f = it * (b + V // 2 * d * 64 * (4 * n + 6)), it * (f + V // 2 * d * 64 * n)
    elif kind == "mesons":
        b, f = _cg_cost(case, "f32", SOLVE_ITERS[case["model"]])
        b, f = 4 * d * (b + 3 * V * 64 * d), 4 * d * f + V * 16 * 16 * d * d * 8
    elif kind == "md":
        # force: links read, momenta read and written; update: links read and written, momenta read
        k = case["steps"]
        mm = 8 * nc ** 3
        loops = 3 * 5 if case["c0"] == 1.0 else 3 * 5 + 3 * 14
        b = V * 4 * ((2 * k + 1) * (lk + 16 * ng) + 2 * k * (2 * lk + 8 * ng))
        f = V * 4 * ((2 * k + 1) * mm * loops + 2 * k * mm * 14)
    elif kind == "step":
        rl, cl, cf = 16 * d * d, 64 * d * d, 96 * d * d
        mm, mr = 8 * nc ** 3, 8 * d ** 3
        k = case["steps"]
        b = k * V * (3 * 4 * lk + 4 * 16 * ng + 2 * 4 * rl + 2 * cl + 2 * cf + 6 * 64 * d)
        f = k * V * (4 * mr * 43 + 24 * 3 * mm + 4 * mm * 29 + 4 * mr)
    elif kind == "hmc":
        solves = 2 * case["steps"] + 2
        b, f = _cg_cost(case, case["sloppy"], SOLVE_ITERS[case["model"]])
        b, f = solves * b, solves * f
    else:
        # forward, adjoint and backward layers, and the weight gradients, per pair: activations in FP32
        w = case["width"]
        act = 96 * V
        b = case["pairs"] * 6 * (act * (4 * w + 2) + 3 * V * 4 * 72)
        f = case["pairs"] * V * 3 * 8 * 9 * 16 * (w * w + 2 * w) * 6
    return {"bytes": b, "flops": f}


def tolerance(case):
    # about four times what is seen between precisions of the inner operator, orders of sums, and exact()
    return {
        "solve": {"rel": 4e-9, "max": 1e-6},      # a residual of 1e-10 over the spread of H^2's spectrum
        "rational": {"rel": 4e-9, "max": 1e-6},
        "mesons": {"rel": 5e-10, "max": 1e-7},    # traces of products of two such solutions
        "md": {"rel": 2e-12, "max": 1e-9},        # 64-bit sums, amplified along the trajectory
        "step": {"rel": 5e-14, "max": 1e-10},
        "hmc": {"rel": 1e-6, "max": 1e-4},        # dH is a small difference of large sums
        "train": {"rel": 1e-2, "max": 0.2},       # bf16 products
    }[case["kind"]]


# ---------------------------------------------------------------------------
# the same in 64-bit torch, on the lattice as a grid (T, X, Y, Z, ...)
# ---------------------------------------------------------------------------
def _lex_of(dims):
    """the grid's flat index of each site in even/odd order"""
    t, x, y, z = torch.meshgrid(*[torch.arange(n, device=DEV) for n in dims], indexing="ij")
    lex = torch.arange(math.prod(dims), device=DEV)
    eo = ((t + x + y + z) % 2).reshape(-1) * (math.prod(dims) // 2) + lex // 2
    return torch.empty_like(lex).scatter_(0, eo, lex)


def _grid(dims, a):
    """even/odd order -> grid"""
    out = torch.empty_like(a)
    out[_lex_of(dims)] = a
    return out.reshape(*dims, *a.shape[1:])


def _flat(dims, a):
    return a.reshape(math.prod(dims), *a.shape[4:])[_lex_of(dims)]


def _bc_mask(case):
    """one on the time slices that the open boundary leaves free, in grid order"""
    dims = (case["T"], case["X"], case["Y"], case["Z"])
    m = torch.ones(dims, dtype=torch.float64, device=DEV)
    if case.get("bc") == "open":
        m[0] = m[-1] = 0
    return m.reshape(-1)


def _mm(a, b):
    return sum(a[..., :, k : k + 1] * b[..., k : k + 1, :] for k in range(b.shape[-2]))


# the chiral basis: gamma_mu psi = PHASE[mu] * psi[PERM[mu]]
PERM = ((2, 3, 0, 1), (3, 2, 1, 0), (3, 2, 1, 0), (2, 3, 0, 1))
PHASE = ((-1, -1, -1, -1), (-1j, -1j, 1j, 1j), (-1, 1, 1, -1), (-1j, 1j, 1j, -1j))
G5 = (1, 1, -1, -1)


def _c(v):
    return torch.tensor(v, dtype=torch.complex128, device=DEV)


def _gamma(mu):
    g = torch.zeros(4, 4, dtype=torch.complex128, device=DEV)
    for a in range(4):
        g[a, PERM[mu][a]] = PHASE[mu][a]
    return g


def _generators(nc):
    """iT_a in the reference's order: below the diagonal symmetric imaginary, above it antisymmetric real"""
    out = []
    for i in range(nc):
        for j in range(nc):
            m = np.zeros((nc, nc), dtype=complex)
            if i > j:
                m[i, j] = m[j, i] = 1j
            elif i < j:
                m[i, j], m[j, i] = 1, -1
            elif i > 0:
                m[range(i), range(i)] = 1j * math.sqrt(2 / (i * (i + 1)))
                m[i, i] = -1j * i * math.sqrt(2 / (i * (i + 1)))
            else:
                continue
            out.append(m)
    return _c(np.array(out))


def _represent(case, u):
    _, _, nc, rep, dr, _ = _geom(case)
    if rep == "fundamental":
        return u
    if rep == "adjoint":
        b = -1j / math.sqrt(2) * _generators(nc)
    else:
        b = torch.zeros(dr, nc, nc, dtype=torch.complex128, device=DEV)
        n = 0
        for i in range(nc):
            for j in range(i + 1):
                b[n, i, j] = b[n, j, i] = 1 if i == j else math.sqrt(0.5)
                n += 1
    right = u.mH if rep == "adjoint" else u.mT
    cols = [_mm(_mm(u, b[m]), right) for m in range(dr)]
    return torch.stack([torch.stack([(b[n].conj() * x).sum((-2, -1)) for x in cols], -1) for n in range(dr)], -2)


class _Inverse(torch.autograd.Function):
    """inverse and log det of positive Hermitian blocks, by elimination without pivots"""

    @staticmethod
    def forward(ctx, a):
        a = a.clone()
        ld = torch.zeros(a.shape[:-2], dtype=torch.float64, device=a.device)
        for k in range(a.shape[-1]):
            p = a[..., k, k].clone()
            ld += p.abs().log()
            row = a[..., k, :] / p[..., None]
            col = a[..., :, k].clone()
            col[..., k] = 0
            a -= col[..., :, None] * row[..., None, :]
            a[..., :, k] = -col / p[..., None]
            a[..., k, :] = row
            a[..., k, k] = 1 / p
        ctx.save_for_backward(a)
        return a, ld

    @staticmethod
    def backward(ctx, g, gl):
        (b,) = ctx.saved_tensors
        return -_mm(_mm(b.mH, g), b.mH) + gl[..., None, None] * b.mH


class _Ref:
    """Operators over the fundamental links u: four grids (T, X, Y, Z, N, N)."""

    def __init__(self, case, u):
        self.case, self.u = case, u
        self.dims, self.V, self.nc, _, self.d, self.mass = _geom(case)
        t, x, y, z = torch.meshgrid(*[torch.arange(n, device=DEV) for n in self.dims], indexing="ij")
        self.even = ((t + x + y + z) % 2 == 0).to(torch.float64)[..., None, None]
        self.free = _bc_mask(case).reshape(self.dims)[..., None, None]
        r = [_represent(case, v) for v in u]
        blocks = self.clover(r)
        if case.get("bc", "antiperiodic") == "antiperiodic":
            sign = torch.ones(self.dims[0], 1, 1, 1, 1, 1, dtype=torch.float64, device=DEV)
            sign[0] = -1
            r = [r[0] * sign] + r[1:]
        self.r = r
        one = torch.eye(2 * self.d, dtype=torch.complex128, device=DEV)
        self.dd = [b + (4 + self.mass) * one for b in blocks]
        inv = [_Inverse.apply(b) for b in self.dd]
        self.inv = [b for b, _ in inv]
        self.logdet = sum((ld * (1 - self.even[..., 0, 0])).sum() for _, ld in inv)

    def clover(self, u):
        """the two chiral blocks of -(c_sw / 16) sum_{mu < nu} [g_mu, g_nu] / 2 (x) (Q - Q^+)"""
        out = [0, 0]
        for mu in range(4):
            for nu in range(mu + 1, 4):
                um, un = u[mu], u[nu]
                um_n, un_m = um.roll(-1, nu), un.roll(-1, mu)                   # at x + nu, x + mu
                um_b, un_b, un_d, um_d = um.roll(1, mu), un.roll(1, mu), un.roll(1, nu), um.roll(1, nu)  # x - mu, x - nu
                q = _mm(_mm(um, un_m), _mm(un, um_n).mH)
                q = q + _mm(_mm(un, um_n.roll(1, mu).mH), _mm(un_b.mH, um_b))
                q = q + _mm(_mm(un_b.roll(1, nu), um_b).mH, _mm(um_b.roll(1, nu), un_d))
                q = q + _mm(_mm(un_d.mH, um_d), _mm(un_d.roll(-1, mu), um.mH))
                f = (q - q.mH) * self.free
                s = (_gamma(mu) @ _gamma(nu) - _gamma(nu) @ _gamma(mu)) / 2
                for b in range(2):
                    out[b] = out[b] + torch.cat([torch.cat([s[2 * b + i, 2 * b + j] * f for j in range(2)], -1)
                                                 for i in range(2)], -2)
        return [-CSW / 16 * b for b in out]

    def hop(self, psi):
        """-1/2 sum_mu [(1 - g_mu) U psi(x + mu) + (1 + g_mu) U^+ psi(x - mu)]"""
        out = 0
        for mu in range(4):
            ph, perm, u = _c(PHASE[mu])[:, None], list(PERM[mu]), self.r[mu]
            up = psi.roll(-1, mu)
            out = out + _mm(up - ph * up[..., perm, :], u.mT)
            out = out + _mm(psi + ph * psi[..., perm, :], u.conj()).roll(1, mu)
        return -0.5 * out * self.free

    def blocks(self, m, psi):
        v = psi.reshape(*self.dims, 2, 2 * self.d, 1)
        return torch.stack([_mm(m[b], v[..., b, :, :]) for b in range(2)], -3).reshape(psi.shape)

    def D(self, psi):
        """the even/odd operator D_ee - D_eo D_oo^-1 D_oe on even fields"""
        odd = self.blocks(self.inv, self.hop(psi) * (1 - self.even))
        return (self.blocks(self.dd, psi) * self.free - self.hop(odd)) * self.even

    def H(self, psi):
        return self.D(psi) * _c(G5)[:, None]

    def solve(self, b, shifts=(0.0,), prec=1e-28):
        """(H^2 + s) x = b for each shift, by conjugate gradients"""
        out = []
        for s in shifts:
            x, r = torch.zeros_like(b), b.clone()
            p, rr, stop = r.clone(), float(_dot(r, r)), prec * float(_dot(b, b))
            while rr > stop:
                q = self.H(self.H(p)) + s * p
                a = rr / float(_dot(p, q))
                x += a * p
                r -= a * q
                old, rr = rr, float(_dot(r, r))
                p = r + (rr / old) * p
            out.append(x)
        return out

    def multishift(self, b, shifts, prec=1e-26):
        """the same on one Krylov space"""
        x = [torch.zeros_like(b) for _ in shifts]
        k = [b.clone() for _ in shifts]
        p, r = b.clone(), b.clone()
        beta, alpha, rr = 1.0, 0.0, float(_dot(b, b))
        stop = prec * rr
        z0, z1 = [1.0] * len(x), [1.0] * len(x)
        while rr * max(z * z for z in z1) > stop:
            q = self.H(self.H(p))
            old, beta = beta, -rr / float(_dot(p, q))
            z2 = [b1 * b0 * old / (beta * alpha * (b0 - b1) + b0 * old * (1 - s * beta))
                  for b0, b1, s in zip(z0, z1, shifts)]
            r += beta * q
            last, rr = rr, float(_dot(r, r))
            alpha = rr / last
            for n in range(len(x)):
                if last * z1[n] ** 2 < 1e-8 * stop:  # converged long ago: its factor would underflow
                    z2[n] = z1[n]
                    continue
                x[n] -= (beta * z2[n] / z1[n]) * k[n]
                k[n] = (alpha * (z2[n] / z1[n]) ** 2) * k[n] + z2[n] * r
            p = alpha * p + r
            z0, z1 = z1, z2
        return x


def _dot(a, b):
    return (a.conj() * b).real.sum()


def _wilson_sum(u, h, w, mu, nu):
    """sum of Re Tr of the h x w loops, h links along mu, w along nu"""
    def line(d, n):
        out = u[d]
        for k in range(1, n):
            out = _mm(out, u[d].roll(-k, d))
        return out
    a, b = line(mu, h), line(nu, w)
    return (_mm(a, b.roll(-h, mu)) * _mm(b, a.roll(-w, nu)).conj()).real.sum()


def _gauge_action(u, c0, nc):
    s = 0
    for mu in range(1, 4):
        for nu in range(mu):
            s = s + c0 * _wilson_sum(u, 1, 1, mu, nu)
            if c0 != 1.0:
                s = s + (1 - c0) / 8 * (_wilson_sum(u, 2, 1, mu, nu) + _wilson_sum(u, 1, 2, mu, nu))
    return -BETA / nc * s


def _kick(u, mom, dt, action, nc):
    """mom -= dt / 2 dS/domega; mom: grids (T, X, Y, Z, 4, NG)"""
    v = [m.detach().requires_grad_() for m in u]
    grads = torch.autograd.grad(action(v), v)
    t = _generators(nc)
    with torch.no_grad():
        for mu in range(4):
            m = _mm(v[mu], grads[mu].mH)
            for a in range(nc * nc - 1):
                mom[..., mu, a] -= dt / 2 * (t[a].mT * m).sum((-2, -1)).real


def _move(u, mom, dt, nc):
    """U <- exp(dt P) U"""
    t, one = _generators(nc), torch.eye(nc, dtype=torch.complex128, device=DEV)
    for mu in range(4):
        x = dt * sum(mom[..., mu, a, None, None] * t[a] for a in range(nc * nc - 1))
        e = one
        for k in range(20, 0, -1):
            e = one + _mm(x, e) / k
        u[mu] = _mm(e, u[mu])


def _o2mn(steps, dt, kick, move):
    a = md.O2MN_LAMBDA
    for n in range(steps):
        kick((a if n == 0 else 2 * a) * dt)
        move(dt / 2)
        kick((1 - 2 * a) * dt)
        move(dt / 2)
    kick(a * dt)


def _links_out(dims, u):
    return torch.from_numpy(_split(_flat(dims, torch.stack(u, -3)).reshape(-1, *u[0].shape[-2:])))


def _exact_md(case, u, mom):
    dims, _, nc, _, _, _ = _geom(case)
    _o2mn(case["steps"], 0.1, lambda dt: _kick(u, mom, dt, lambda v: _gauge_action(v, case["c0"], nc), nc),
          lambda dt: _move(u, mom, dt, nc))


def _fermion_action(case, x):
    """what the force of a solution x of H^2 x = phi derives from, at fixed x: -|H x|^2 - 2 log det D_oo"""
    def action(v):
        op = _Ref(case, v)
        h = op.H(x)
        return -_dot(h, h) - 2 * op.logdet
    return action


def _exact_hmc(case, u, seed):
    dims, V, nc, _, d, _ = _geom(case)
    rng = np.random.default_rng(int(seed))
    mom = _grid(dims, torch.from_numpy(rng.normal(0.0, np.sqrt(0.5), size=(4 * V, nc * nc - 1))).to(DEV)
                .reshape(V, 4, -1))
    eta = np.zeros((V, 8 * d))
    eta[: V // 2] = rng.normal(0.0, np.sqrt(0.5), size=(V // 2, 8 * d))
    eta = _grid(dims, torch.complex(*torch.from_numpy(eta).to(DEV).reshape(V, 2, d, 4).unbind(1)).mT.contiguous())
    op = _Ref(case, u)
    phi = op.H(eta)

    def total(s):
        return float((mom * mom).sum()) + float(_gauge_action(u, 1.0, nc)) + s

    h0 = total(float(_dot(eta, eta)) - 2 * float(op.logdet))

    def gauge_kick(dt):
        _kick(u, mom, dt, lambda v: _gauge_action(v, 1.0, nc), nc)

    def kick(dt):
        x = _Ref(case, u).solve(phi, prec=1e-29)[0]
        _kick(u, mom, dt, _fermion_action(case, x), nc)

    def move(dt):
        _o2mn(2, dt / 2, gauge_kick, lambda e: _move(u, mom, e, nc))

    _o2mn(case["steps"], 0.4 / case["steps"], kick, move)
    op = _Ref(case, u)
    x = op.solve(phi, prec=1e-29)[0]
    dh = total(float(_dot(phi, x)) - 2 * float(op.logdet)) - h0
    plaq = float(_gauge_action(u, 1.0, nc)) / (-BETA * 6 * V)
    return {"dH": dh, "plaquette": plaq, "links": _links_out(dims, u)}


def _exact_mesons(case, u):
    dims, V, _, _, d, mass = _geom(case)
    op = _Ref(case, u)
    S = []
    for n in range(4 * d):
        b = torch.zeros(*dims, 4, d, dtype=torch.complex128, device=DEV)
        b[case["tau"], 0, 0, 0, n // d, n % d] = 1
        odd = op.blocks(op.inv, b * (1 - op.even))
        s = (b - op.hop(odd)) * op.even
        x = op.solve(op.H(s * _c(G5)[:, None]))[0]
        S.append(x + op.blocks(op.inv, (b - op.hop(x)) * (1 - op.even)))
    # rows (source spin, sink spin), columns (source colour, sink colour, space) of each time slice
    S = torch.stack(S).reshape(4, d, dims[0], -1, 4, d).permute(2, 0, 4, 1, 5, 3).reshape(dims[0], 16, -1)
    M = torch.stack([s @ s.mH for s in S]).reshape(dims[0], 4, 4, 4, 4)  # t, c, b, d, a
    g5 = torch.diag(_c(G5))
    one = torch.eye(4, dtype=torch.complex128, device=DEV)
    named = {"g%d" % mu: _gamma(mu) for mu in range(4)} | {"g5": g5, "id": one}

    def table(name):
        g = one
        for part in (name[i : i + 2] for i in range(0, len(name), 2)):
            g = g @ named[part]
        return g5 @ g

    out = {}
    for name, sign in zip(spectrum.CHANNELS, spectrum.SIGNS):
        g1, g2 = (table("g0g5"), table("g5")) if name == "g5_g0g5" else (table(name), table(name))
        c = (M * g1.mT[None, None, :, None, :] * g2[None, :, None, :, None]).sum((1, 2, 3, 4)).real
        out[name] = sign * c.roll(-case["tau"])
    return out


def _exact_train(case, op, seed):
    W = [_c(w).requires_grad_() for w in _weights(case, seed)]

    def layer(w, h):  # h: (T, X, Y, Z, channels, 4, 3)
        flat = (*op.dims, -1, 3)
        out = 0
        for q in range(9):
            mu = (q - 1) % 4
            if q == 0:
                t = h
            elif q <= 4:
                t = _mm(h.roll(-1, mu), op.r[mu].mT[..., None, :, :])
            else:
                t = _mm(h, op.r[mu].conj()[..., None, :, :]).roll(1, mu)
            m = w[q].permute(0, 2, 1, 3).reshape(w.shape[1] * 4, -1)
            out = out + (m @ t.reshape(flat).permute(4, 5, 0, 1, 2, 3).reshape(m.shape[1], -1)).reshape(
                m.shape[0], 3, *op.dims).permute(2, 3, 4, 5, 0, 1).reshape(*op.dims, -1, 4, 3)
        return out

    bar = [0, 5, 6, 7, 8, 1, 2, 3, 4]
    adj = [w[bar].permute(0, 2, 1, 4, 3).conj() for w in W]
    loss = 0
    for k in range(case["pairs"]):
        x = _grid(op.dims, _spinor(case, seed, 20 + k))
        h = op.H(op.H(x))[..., None, :, :]
        for w in adj[::-1]:
            h = layer(w, h)
        h = h * op.even[..., None]
        for w in W:
            h = layer(w, h)
        e = h[..., 0, :, :] * op.even - x
        loss = loss + _dot(e, e) / _dot(x, x)
    return {"loss": float(loss.detach()), "grads": list(torch.autograd.grad(loss, W))}


def exact(case, seed):
    dims, V, nc, _, d, _ = _geom(case)
    kind = case["kind"]
    u = [m.contiguous() for m in _grid(dims, _links(case, seed).reshape(V, 4, nc, nc)).unbind(4)]
    if case.get("bc") == "open":
        u[0][-1] = 0
    if kind == "mesons":
        return _exact_mesons(case, u)
    if kind == "hmc":
        return _exact_hmc(case, u, seed)
    if kind == "train":
        return _exact_train(case, _Ref(case, u), seed)
    if kind in ("solve", "rational"):
        op, b = _Ref(case, u), _grid(dims, _spinor(case, seed, 2))
        if kind == "solve":
            x = op.solve(b)[0]
        else:
            rat = yh.rational_zolotarev(case["poles"], -1, 2, 1e-2, 64.0)
            x = rat.a0 * b
            for r, y in zip(rat.residue, op.multishift(b, rat.pole[: rat.order])):
                x = x + r * y
        return torch.from_numpy(_spinor_host(_flat(dims, x)[: V // 2]))
    mom = _grid(dims, _momenta(case, seed).reshape(V, 4, -1))
    if kind == "md":
        _exact_md(case, u, mom)
    else:
        x = _grid(dims, _spinor(case, seed, 2))
        for _ in range(case["steps"]):
            _kick(u, mom, STEP_DT, _fermion_action(case, x), nc)
            _kick(u, mom, STEP_DT, lambda v: _gauge_action(v, 1.0, nc), nc)
            _move(u, mom, STEP_DT, nc)
    return [_links_out(dims, u), _flat(dims, mom).reshape(4 * V, -1)]
