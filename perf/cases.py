"""Workloads of the radiation solver whose time is watched: one pass of each
through the public entry points, the inputs a program holds before it, and the
value of its outputs in 64 bits.

A radiation step is what the channel DNS asks for every few time steps: the
temperature field in (host memory), the solve, Q_rad and its standard error
out (host memory).  The spectral table is the synthetic 100 x 16 x 69
correlated-k table and the grids are those of the channel workloads
(dnsmc_amd/workloads.py, bench.py): periodic x and z, black walls in y.
"""
import math

import numpy as np
import torch

import dnsmc_amd
from dnsmc_amd import learned
from dnsmc_amd.solver import config_from_dict

SIGMA = 5.670373e-08
SEED = 20240601                      # of the solver's own ray draws
LENGTHS = (2.0 * math.pi, 2.0, math.pi)
BETA = 1.5                           # tanh stretching of the wall-normal axis
NB, NQ = 100, 16                     # bands, quadrature points
DEV = "cuda" if torch.cuda.is_available() else "cpu"
EXACT_MOST = 4e9                     # cell crossings that exact() follows
SLAB_ROWS = 2                        # ranks of the coupled DNS along y


# ------------------------------------------------------------------ cases ----
def _step(name, n, rays, gas="ck", levels=1, snaps=1, tally=0):
    return dict(name=name, kind="step", gas=gas, n0=n[0], n1=n[1], n2=n[2], rays=rays, levels=levels, snaps=snaps,
                tally=tally)


def listed():
    return [
        # the smallest call: a coarse grey box, as a unit test or a first try of the coupling runs it
        _step("grey_16", (16, 24, 16), 32, gas="grey"),
        # the grey 32^3 channel at its usual ray count
        _step("grey_32", (32, 32, 32), 100, gas="grey"),
        # the small correlated-k channel at its usual ray count
        _step("ck_64", (64, 96, 64), 500),
        # a grid of odd sizes with run-to-run identical sums (deterministic FP64 tally)
        _step("ck_odd_fixed_sums", (45, 61, 37), 100, tally=1),
        # two snapshots of the middle channel in one call, the reference's five coarsening levels
        _step("ck_256_coarsened", (256, 128, 128), 100, levels=5, snaps=2),
        # the production channel, fine grid only: the largest call
        _step("ck_384", (384, 256, 256), 100),
        # the middle channel with a learned proposal, coarsened, as the time-to-accuracy runs solve it
        dict(name="learned_256", kind="learned", n0=256, n1=128, n2=128, rays=100, levels=5),
        # one step of the coupled DNS: slabs of eight ranks in, solve with four levels, slabs out
        dict(name="coupled_192", kind="coupled", n0=192, n1=128, n2=128, rays=20, levels=4, ranks=4),
        # the reference's own sampling (XORWOW and Sobol, sorted bands) at its shipped 3 x 20000 bundles per cell
        dict(name="reference_sampling", kind="sampled", n0=16, n1=24, n2=16, photmax=20000, levels=3, srt=1),
        # the FP64 traversal on sampled cells: the converged values that errors are measured against
        dict(name="fp64_cells", kind="fp64", n0=64, n1=96, n2=64, cells=1024, rays=8192),
        # one optimiser step of the proposal at the trainer's minibatch
        dict(name="train_16384", kind="train", rows=16384, nbin=NB * NQ),
        # training data from one recorded run of the trainer's grid at its 8 rays per cell
        dict(name="collect_64", kind="collect", n0=64, n1=96, n2=64, rays=8),
    ]


def _loguniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sizes(rng, cells, multiple=1):
    """Grid sizes near the channel's proportions with about `cells` cells, multiples of `multiple`, odd ones among them."""
    a = (cells / 1.2) ** (1.0 / 3.0)
    out = []
    for ratio in (1.2, 1.3, 0.9):
        v = a * ratio * rng.uniform(0.8, 1.2)
        out.append(max(4 * multiple, min(384, int(round(v / multiple)) * multiple)))
    return tuple(out)


def draw(rng):
    kind = rng.choice(("step", "step", "step", "step", "learned", "coupled", "sampled", "fp64", "train", "collect"))
    if kind == "train":
        return dict(kind=kind, rows=_loguniform(rng, 1000, 16384), nbin=rng.choice((121, 400, 1000, 1600)))
    if kind == "collect":
        n = _sizes(rng, _loguniform(rng, 20000, 400000))
        most = (1 << 22) // (n[0] * n[1] * n[2])                 # a recorded run holds 2^22 rays
        return dict(kind=kind, n0=n[0], n1=n[1], n2=n[2], rays=min(rng.randint(4, 8), most))
    if kind == "fp64":
        n = _sizes(rng, _loguniform(rng, 10000, 400000))
        return dict(kind=kind, n0=n[0], n1=n[1], n2=n[2], cells=rng.randint(100, 1024), rays=_loguniform(rng, 500, 8192))
    if kind == "sampled":
        return dict(kind=kind, n0=16, n1=4 * rng.randint(2, 6), n2=4 * rng.randint(2, 5),
                    photmax=_loguniform(rng, 500, 20000), levels=rng.choice((1, 3)), srt=rng.choice((0, 1)))
    levels = rng.choice((1, 4, 5)) if kind == "step" else 4
    n = _sizes(rng, _loguniform(rng, 8000, 4000000), 1 << (levels - 1))
    cells = n[0] * n[1] * n[2]
    if kind == "coupled":
        n = (n[0], n[1] // 16 * 16 + 16, n[2] // 16 * 16 + 16)
        return dict(kind=kind, n0=n[0], n1=n[1], n2=n[2], rays=rng.randint(10, 40), levels=4, ranks=rng.choice((2, 4)))
    rays = _loguniform(rng, 20, max(21, min(500, int(4e8 / cells))))
    if kind == "learned":
        return dict(kind=kind, n0=n[0], n1=n[1], n2=n[2], rays=min(rays, 200), levels=levels)
    gas = rng.choice(("grey", "ck", "ck"))
    return dict(kind=kind, gas=gas, n0=n[0], n1=n[1], n2=n[2], rays=rays, levels=levels, snaps=rng.choice((1, 1, 2)),
                tally=rng.choice((0, 0, 0, 1)))


# ----------------------------------------------------------------- inputs ----
def _rng(case, seed, salt=0):
    return np.random.Generator(np.random.Philox(key=[int(seed), salt]))


def _grid(case):
    return (case["n0"], case["n1"], case["n2"])


def _faces(n):
    """Face coordinates of the finest level, FP32 (uniform, tanh-stretched, uniform)."""
    out = []
    for a in range(3):
        if a == 1:
            e = 2.0 * np.arange(n[1] + 1) / n[1] - 1.0
            f = (0.5 * LENGTHS[1] * (1.0 + np.tanh(BETA * e) / math.tanh(BETA))).astype(np.float32)
            f[0], f[-1] = 0.0, LENGTHS[1]
        else:
            f = np.arange(n[a] + 1, dtype=np.float32) * (np.float32(LENGTHS[a]) / np.float32(n[a]))
        out.append(f)
    return out


def _fields(case, seed, snaps=1):
    """Interior temperatures (n0, n1, n2): the channel's parabolic profile with a few random modes and cell noise."""
    n = _grid(case)
    y = _faces(n)[1].astype(np.float64)
    yc = torch.tensor(0.5 * (y[1:] + y[:-1]), device=DEV)
    x, z = (torch.arange(m, device=DEV, dtype=torch.float64) * (2.0 * math.pi / m) for m in (n[0], n[2]))
    out = []
    for s in range(snaps):
        g = _rng(case, seed, 1 + s)
        if case.get("gas") == "grey":
            T = torch.full(n, 1000.0, device=DEV, dtype=torch.float64)
            amp = 5.0
        else:
            T = (573.0 + 382.0 * (1.0 - (yc - 1.0) ** 2))[None, :, None].expand(n).clone()
            amp = 10.0
            for _ in range(6):
                kx, ky, kz = g.integers(0, 9), g.integers(1, 9), g.integers(0, 9)
                px, pz = g.uniform(0.0, 2.0 * math.pi, 2)
                T += 10.0 * (torch.cos(kx * x + px)[:, None, None] * torch.sin(math.pi * ky * yc / 2.0)[None, :, None]
                             * torch.cos(kz * z + pz)[None, None, :])
        gen = torch.Generator(device="cpu").manual_seed(int(g.integers(1 << 31)))
        noise = torch.randn(1 << 16, generator=gen).to(DEV)
        reps = -(-T.numel() // noise.numel())
        T += amp * noise.repeat(reps)[:T.numel()].reshape(n).clamp(-4.0, 4.0)
        out.append(T.float().cpu().numpy())
    return out


def _ghosted(T):
    """Interior field -> T(0:n0+1, 0:n1+1, 0:n2+1), i fastest, as the DNS holds it."""
    return np.asfortranarray(np.pad(T, 1, mode="edge"))


def _planck(T, nu):
    nu_m = nu * 100.0
    return 3.741771790075259e-16 / math.pi * nu_m ** 3 / np.expm1(0.014387741858429 * nu_m / T)


def _table():
    """Log-normal correlated-k table (100 bands, 16 points, 300-2000 K), FP32 arrays in the reference's layouts."""
    g = np.random.Generator(np.random.Philox(key=11))
    Tnb = np.arange(300.0, 2012.5, 25.0)
    dnu = (7500.0 - 150.0) / NB
    wvl = 150.0 + dnu * np.arange(NB)
    wvc = wvl + 0.5 * dnu
    xq, wq = np.polynomial.legendre.leggauss(NQ)
    ndtri = torch.special.ndtri(torch.tensor(0.5 * (xq + 1.0))).numpy()
    m = g.uniform(math.log(0.01), math.log(10.0), NB)
    c = g.uniform(-1.0, 0.5, NB)
    mu = m[:, None] + c[:, None] * np.log(Tnb[None, :] / 1000.0)
    kq = np.exp(mu[:, :, None] + 2.0 * ndtri[None, None, :])                    # [band][T][g]
    e = kq * (0.5 * wq)[None, None, :] * (_planck(Tnb[None, :], wvc[:, None]) * dnu * 100.0)[:, :, None]
    kP = math.pi * e.sum(axis=(0, 2)) / (SIGMA * Tnb ** 4)
    eb = e.sum(axis=2)
    probg = np.cumsum(kq * (0.5 * wq), axis=2)
    t = dict(Tnb=Tnb, kP=kP, wvl=wvl, wvr=wvl + dnu, wvc=wvc, kq=kq, prob=(np.cumsum(eb, axis=0) / eb.sum(axis=0)).T,
             probg=(probg / probg[:, :, -1:]).transpose(1, 0, 2), kavg=(kq * (0.5 * wq)).sum(axis=2)[:, -1])
    return {k: np.ascontiguousarray(v, np.float32) for k, v in t.items()}


def _config(case):
    grey = case.get("gas") == "grey"
    kind, levels = case["kind"], case.get("levels", 1)
    maxs = [5] * (levels - 1) + [100000] * (7 - levels)
    Tw = 300.0 if grey else 573.0
    d = dict(n=_grid(case), L=LENGTHS, stretch=(0, 2, 0), stretch_beta=(BETA,) * 3, bc=((1, 1), (2, 2), (1, 1)),
             Tw=((0.0, 0.0), (Tw, Tw), (0.0, 0.0)), polar_axis=1, rays_per_cell=case.get("rays", 2), grid_num=levels,
             maxs=maxs[:6], toll=1.0e-3, spectral=3 if grey else 0, kappa_grey=1.0, mode=0, num_streams=16, num_gpu=1,
             gpu=0, p_row=1, seed=SEED, nsnap=case.get("snaps", 1), precision=0, tally=case.get("tally", 0), srt=0,
             batch_rays=1 << 31, table_dir="")
    if kind == "sampled":
        d.update(mode=1, nvar=3, photmax=case["photmax"], sobol=1, srt=case["srt"])
    elif kind == "learned":
        d.update(mode=2)
    elif kind == "fp64":
        d.update(precision=1, tally=1)
    return d


def _emitters(case, seed):
    n = _grid(case)
    cells = _rng(case, seed, 50).choice(n[0] * n[1] * n[2], size=case["cells"], replace=False)
    return np.sort(cells).astype(np.int32)


def _network(seed):
    """A proposal as training leaves it: bins that are emitted from and seen far away, directions towards the walls."""
    g = np.random.default_rng(int(seed))
    t = _table()
    L = learned.layout(NB * NQ)
    node = 26                                                                    # 950 K
    _, wq = np.polynomial.legendre.leggauss(NQ)
    kappa = t["kq"][:, node, :].astype(np.float64)
    p = kappa * (0.5 * wq) * _planck(950.0, t["wvc"].astype(np.float64))[:, None]
    far = p * np.sqrt((1.0 - np.exp(-kappa)) / kappa * np.exp(-0.05 * kappa) + 1e-4)
    b3 = np.full(L["noutp"], 0.0)
    cosine = np.abs(np.arange(8) - 3.5) / 3.5
    b3[:64] = np.repeat(0.5 * cosine, 8)
    b3[64:64 + NB * NQ] = np.log(far / far.sum() + 1e-9).ravel()
    W = [g.uniform(-1, 1, s) * a for s, a in ((6 * 64, 0.29), (64 * 64, 0.21), (64 * L["noutp"], 0.03))]
    b = [g.uniform(-0.1, 0.1, 64), g.uniform(-0.1, 0.1, 64), b3]
    return [x for w, c in zip(W, b) for x in (_bf16(w), c.astype(np.float32))]


def _bf16(x):
    return torch.tensor(np.asarray(x), dtype=torch.float32).bfloat16().view(torch.int16).numpy().view(np.uint16)


def _slabs(case):
    """(start, end) of the ranks' slabs, 1-based inclusive, ranks along z times SLAB_ROWS along y."""
    n, out = _grid(case), []
    for rz in range(case["ranks"]):
        for ry in range(SLAB_ROWS):
            j, k = n[1] // SLAB_ROWS, n[2] // case["ranks"]
            out.append(((1, 1 + ry * j, 1 + rz * k), (n[0], (ry + 1) * j, (rz + 1) * k)))
    return out


T_REF, T_PLUS = 573.0, 2.0           # the coupled DNS's reference temperature and scale


def _nondimensional(case, seed):
    """cnew of every rank: (T - T_REF) T_PLUS / T_REF on its slab, FP64, x with ghosts."""
    T = _fields(case, seed)[0].astype(np.float64)
    c = np.pad((T - T_REF) * T_PLUS / T_REF, ((1, 1), (0, 0), (0, 0)), mode="edge")
    return [np.asfortranarray(c[:, s[1] - 1:e[1], s[2] - 1:e[2]]) for s, e in _slabs(case)]


def _train_inputs(case, seed):
    g = _rng(case, seed, 90)
    n, nbin = case["rows"], case["nbin"]
    L = learned.layout(nbin)
    th = np.zeros(L["P"], np.float32)
    for key, end, a in (("W1", "b1", 0.29), ("b1", "W2", 0.1), ("W2", "b2", 0.21), ("b2", "W3", 0.1), ("W3", "b3", 0.1),
                        ("b3", "P", 1.0)):
        th[L[key]:L[end]] = g.uniform(-a, a, L[end] - L[key])
    X = g.uniform(-1.0, 1.0, (n, 6))
    X[:, 1] = 0.6 + 0.4 * np.abs(X[:, 1])
    X[:, 5] = 0.58
    wt = g.lognormal(0.0, 1.5, n)
    m = g.normal(0.0, 1e-4, L["P"])
    v = g.uniform(1e-8, 2e-8, L["P"])
    return dict(theta=th, X=X.astype(np.float32), td=g.integers(0, 64, n).astype(np.int32),
                tb=(nbin * g.beta(1.0, 2.0, n)).astype(np.int32), wt=wt.astype(np.float32), m=m.astype(np.float32),
                v=v.astype(np.float32))


TRAIN_STEP, TRAIN_RATE, COST0 = 200, 2e-3, 16.0


# ---------------------------------------------------------- prepare and run ----
class _View:
    """A device array of the library, for torch (no copy; keeps the array alive)."""

    def __init__(self, a):
        self.a = a
        self.__cuda_array_interface__ = dict(shape=a.shape, typestr=a.dtype.str, data=(a.ptr, False), version=3, strides=None)


def _view(a):
    return torch.as_tensor(_View(a), device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        i = _train_inputs(case, seed)
        net = learned.ProposalNet(case["nbin"], theta=i["theta"])
        net.m, net.v = learned.DeviceArray.from_numpy(i["m"]), learned.DeviceArray.from_numpy(i["v"])
        net.step_count = TRAIN_STEP
        return dict(kind=kind, net=net, data=[learned.DeviceArray.from_numpy(i[k]) for k in ("X", "td", "tb", "wt")])
    S = dnsmc_amd.Solver(config_from_dict(_config(case)))
    if case.get("gas") == "grey":
        S.load_tables()
    else:
        S.set_tables(_table())
    state = dict(kind=kind, S=S)
    if kind == "coupled":
        n = _grid(case)
        k = n[2] // case["ranks"]
        state.update(cnew=_nondimensional(case, seed), slabs=_slabs(case),
                     out=[((1, 1, 1 + r * k), (n[0], n[1], (r + 1) * k)) for r in range(case["ranks"])])
        return state
    if kind == "learned":
        S.set_mlp(*_network(seed))
    if kind == "fp64":
        S.set_emitters(_emitters(case, seed))
    if kind == "collect":
        S.set_record(True)
    state["T"] = [_ghosted(T) for T in _fields(case, seed, case.get("snaps", 1))]
    if kind in ("fp64", "collect"):
        S.set_field(0, state["T"][0])
    return state


def run(state):
    kind = state["kind"]
    if kind == "train":
        net = state["net"]
        loss = net.loss_grad(*state["data"])
        net.adam(TRAIN_RATE)
        return dict(loss=loss, grad=_view(net.grad), theta=_view(net.theta), m=_view(net.m), v=_view(net.v))
    S = state["S"]
    if kind == "coupled":
        for c, (start, end) in zip(state["cnew"], state["slabs"]):
            S.fix_temp_slab(0, c, start, end, T_REF, T_PLUS)
        S.commit_field(0)
        S.run()
        return [S.fix_rad_slab(0, start, end, T_REF) for start, end in state["out"]]
    if kind == "fp64":
        S.run()
        return S.results(0)
    if kind == "collect":
        S.run()
        S.wait()
        samples = learned.SampleSet()
        samples.add_run(S, cost0=COST0)
        return [_view(a) for a in samples.parts[0]]
    for s, T in enumerate(state["T"]):
        S.set_field(s, T)
    S.run()
    if kind == "learned":
        return S.results(0)
    return [S.results_fortran(s) for s in range(len(state["T"]))]


# -------------------------------------------------------------------- work ----
def _crossings(case):
    """About how many cells a ray of this case crosses (measured on the channel workloads)."""
    n = _grid(case)
    per_metre = sum(m / l for m, l in zip(n, LENGTHS)) / 3.0
    if case.get("gas") == "grey":
        fine = 3.5 * per_metre
    else:
        fine = 1.0 + 0.4 * per_metre
    if case.get("levels", 1) > 1:
        fine = min(fine, 10.0)
    return fine * (2.5 if case["kind"] == "learned" else 1.0)


def _rays(case):
    n = _grid(case)
    cells = case.get("cells", n[0] * n[1] * n[2])
    if case["kind"] == "sampled":
        return cells * 3 * case["photmax"]
    return cells * case["rays"] * case.get("snaps", 1)


def work(case):
    """The inputs and outputs once; about 40 operations per cell crossing and 150 per ray, the products of the network."""
    if case["kind"] == "train":
        P, rows = learned.layout(case["nbin"])["P"], case["rows"]
        return dict(bytes=rows * 36 + 30 * P, flops=6.0 * P * rows)
    n = _grid(case)
    cells, rays = n[0] * n[1] * n[2], _rays(case)
    flops = rays * (40.0 * _crossings(case) + 150.0)
    kind = case["kind"]
    if kind == "coupled":
        moved = cells * (8 + 16)
    elif kind == "fp64":
        moved = cells * 4 + case["cells"] * 32
    elif kind == "collect":
        moved = cells * 4 + rays * 36
    elif kind == "learned":
        moved = cells * (4 + 32)
        flops += cells * 222000.0
    else:
        moved = cells * case.get("snaps", 1) * (4 + 8)
    return dict(bytes=float(moved), flops=float(flops))


# --------------------------------------------- the same estimator in 64 bits ----
def _philox(c, key):
    """Philox4x32-10 (Salmon et al. 2011) on int64 tensors holding 32-bit words."""
    M = 0xFFFFFFFF

    def mul(k, x):
        p, q = k * (x >> 16), k * (x & 0xFFFF)
        return (p + (q >> 16)) >> 16, ((p << 16) + q) & M

    k0, k1 = key & M, key >> 32
    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c[0])
        h1, l1 = mul(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
        k0, k1 = (k0 + 0x9E3779B9) & M, (k1 + 0xBB67AE85) & M
    return c


def _spline(x, xc):
    """Matrix of the natural cubic spline through nodes x, evaluated at xc."""
    n, h = len(x), np.diff(x)
    A, B = np.eye(n), np.zeros((n, n))
    for i in range(1, n - 1):
        A[i, i - 1:i + 2] = h[i - 1] / 6.0, (h[i - 1] + h[i]) / 3.0, h[i] / 6.0
        B[i, i - 1:i + 2] = 1.0 / h[i - 1], -1.0 / h[i - 1] - 1.0 / h[i], 1.0 / h[i]
    C = np.linalg.solve(A, B)
    k = np.clip(np.searchsorted(x, xc, side="right") - 1, 0, n - 2)
    q, r = np.arange(len(xc)), h[k]
    a = (x[k + 1] - xc) / r
    b = 1.0 - a
    W = np.zeros((len(xc), n))
    W[q, k] += a
    W[q, k + 1] += b
    return W + ((a ** 3 - a) * r * r / 6.0)[:, None] * C[k] + ((b ** 3 - b) * r * r / 6.0)[:, None] * C[k + 1]


class _Exact:
    """The plain estimator's rays of one temperature field, followed in FP64."""

    def __init__(self, case, T, Tmax=0.0):
        self.case, self.cfg = case, _config(case)
        n0, levels = _grid(case), case.get("levels", 1)
        fine = _faces(n0)
        self.centre = [(0.5 * (f[1:] + f[:-1])).astype(np.float64) for f in fine]
        T = torch.tensor(T, dtype=torch.float64)
        faces, fields, self.n, self.fo, self.to = [], [], [], [], []
        nf = nt = 0
        for g in range(levels):
            f = [a[::1 << g] for a in fine]
            W = [torch.tensor(_spline(self.centre[a], (0.5 * (f[a][1:] + f[a][:-1])).astype(np.float64)))
                 for a in range(3)] if g else None
            t = T
            for a in range(3 if g else 0):                       # axis by axis, as FP32 fields
                t = torch.tensordot(W[a], t, dims=([1], [a])).movedim(0, a).float().double()
            self.n.append(t.shape)
            self.to.append(nt)
            self.fo.append([nf, nf + len(f[0]), nf + len(f[0]) + len(f[1])])
            faces += [a.astype(np.float64) for a in f]
            fields.append(t.permute(2, 1, 0).reshape(-1))
            nf += sum(len(a) for a in f)
            nt += t.numel()
        Tmax = max(float(T.max()), Tmax, max(max(w) for w in self.cfg["Tw"]))
        arrays = dict(face=np.concatenate(faces), T=torch.cat(fields).numpy(), n=np.array([list(s) for s in self.n]).T,
                      fo=np.array(self.fo).T, to=np.array(self.to), maxs=np.array(self.cfg["maxs"][:levels]))
        self.grey = case.get("gas") == "grey"
        R = self.cfg["rays_per_cell"]
        if self.grey:
            self.total = 4.0 * SIGMA * Tmax ** 4 / R
            self.scale = self.total / Tmax ** 4
            arrays["wall"] = np.array([w ** 4 for w in (300.0, 300.0)])
        else:
            t = _table()
            kq = t["kq"].transpose(0, 2, 1).reshape(NB * NQ, -1).astype(np.float64)
            Ib = _planck(t["Tnb"].astype(np.float64)[None, :], t["wvc"].astype(np.float64)[:, None])
            pos = (Tmax - 300.0) / 25.0
            k = int(pos)
            at = lambda a: a[:, k] + (pos - k) * (a[:, k + 1] - a[:, k])  # noqa: E731
            em = at(kq).reshape(NB, NQ) * at(Ib)[:, None]
            _, wq = np.polynomial.legendre.leggauss(NQ)
            dnu = (t["wvr"].astype(np.float64) - t["wvl"]) * 100.0
            e = 4.0 * math.pi * em * (0.5 * wq) * dnu[:, None]
            cb = np.cumsum(e.sum(axis=1)) / e.sum()
            cg = np.cumsum(e, axis=1) / e.sum(axis=1, keepdims=True)
            cb[-1], cg[:, -1] = 1.0, 1.0
            self.total = e.sum() / R
            arrays.update(kq=kq.ravel(), Ib=Ib.ravel(), iem=1.0 / em.ravel(), cb=cb.astype(np.float32).astype(np.float64),
                          cg=(cg.astype(np.float32).astype(np.float64) + np.arange(NB)[:, None]).ravel(),
                          wall=_planck(573.0, t["wvc"].astype(np.float64)))
            self.nT = Ib.shape[1]
        self.on = {"torch": {k: torch.tensor(v, device=DEV) for k, v in arrays.items()}, "numpy": arrays}

    def table(self, A, xp, T, row, band):
        if self.grey:
            return 1.0, T * T * T * T
        pos = xp.clip((T - 300.0) / 25.0, 0.0, self.nT - 1.0)
        k = xp.clip(pos.long() if xp is torch else pos.astype(np.int64), 0, self.nT - 2)
        fr = pos - k
        q, i = row * self.nT + k, band * self.nT + k
        return A["kq"][q] + fr * (A["kq"][q + 1] - A["kq"][q]), A["Ib"][i] + fr * (A["Ib"][i + 1] - A["Ib"][i])

    def start(self, cell, r, snap):
        """State of rays r of cells `cell` (int64 tensors, 0-based, i fastest)."""
        A, n = self.on["torch"], self.n[0]
        x = _philox([r, cell, torch.full_like(r, snap), torch.zeros_like(r)], SEED)
        u = [((w >> 9).double() + 0.5) * 2.0 ** -23 for w in x[:2]]
        ut, up = [((w >> 8).double() + 0.5) * 2.0 ** -24 for w in x[2:]]
        ijk = torch.stack([cell % n[0], cell // n[0] % n[1], cell // (n[0] * n[1])])
        if self.grey:
            band = row = torch.zeros_like(cell)
        else:
            band = torch.searchsorted(A["cb"], u[0], right=True).clamp(max=NB - 1)
            g = (torch.searchsorted(A["cg"], band + u[1], right=True) - band * NQ).clamp(0, NQ - 1)
            row = band * NQ + g
        cth, sth, ph = 1.0 - 2.0 * ut, 2.0 * torch.sqrt(ut * (1.0 - ut)), 2.0 * math.pi * up
        s = torch.stack([sth * torch.sin(ph), cth, sth * torch.cos(ph)])
        s = torch.where(s == 0.0, torch.full_like(s, 1e-10), s)
        p = torch.stack([torch.tensor(self.centre[a], device=DEV)[ijk[a]] for a in range(3)])
        T = A["T"][cell]
        kap, ib = self.table(A, torch, T, row, band)
        w = self.scale * ib if self.grey else self.total * kap * ib * A["iem"][row]
        z = torch.zeros_like(cell)
        return dict(p=p, s=s, c=ijk + 1, lev=z, cnt=z.clone(), steps=z.clone(), row=row, band=band, tau=torch.zeros_like(T),
                    tra=torch.ones_like(T), G=torch.zeros_like(T), w=w, wi=w / ib, id=torch.arange(len(cell), device=DEV))

    def step(self, st, A, xp):
        """One cell crossing of every ray; returns (ended, the emission factor of those)."""
        lev, c, p = st["lev"], st["c"], st["p"]
        neg = st["s"] < 0.0
        n, fo = A["n"][:, lev], A["fo"][:, lev]
        fx = A["face"][fo + c - neg * 1]
        d = (fx - p) / st["s"]
        ds = xp.minimum(xp.minimum(d[0], d[1]), d[2])
        p = xp.where(d == ds, fx, p + ds * st["s"])
        T = A["T"][A["to"][lev] + (c[0] - 1) + n[0] * ((c[1] - 1) + n[1] * (c[2] - 1))]
        kap, ib = self.table(A, xp, T, st["row"], st["band"])
        tau = st["tau"] + kap * ds
        cut = tau >= -math.log(1.0e-3)
        tra = xp.exp(-tau)
        G = st["G"] + xp.where(cut, st["tra"], st["tra"] - tra) * ib
        ax = xp.where(d[0] < d[1], xp.where(d[0] < d[2], 0, 2), xp.where(d[1] < d[2], 1, 2))
        axes = xp.stack([ax == 0, ax == 1, ax == 2])
        c = c + axes * (1 - 2 * neg * 1)
        low, high = c == 0, c == n + 1
        hit = ~cut & (low[1] | high[1])
        G = xp.where(hit, G + tra * (A["wall"][st["band"]] if not self.grey else A["wall"][0]), G)
        out = (low | high) & (xp.stack([xp.ones_like(cut), xp.zeros_like(cut), xp.ones_like(cut)]) > 0)
        c = xp.where(out & low, n, xp.where(out & high, 1, c))
        p = xp.where(out, A["face"][fo + xp.where(low, n, 0)], p)
        cnt = st["cnt"] + 1
        cap = ~cut & ~hit & (cnt >= A["maxs"][lev])
        last = cap & (lev + 1 >= len(self.n))
        down = cap & ~last
        st.update(p=p, c=xp.where(down, (c + 1) // 2, c), lev=lev + down * 1, cnt=xp.where(down, 0, cnt),
                  steps=st["steps"] + 1, tau=tau, tra=xp.where(cut, st["tra"], tra), G=G)
        return cut | hit | last, xp.where(last, 1.0 - tra, xp.ones_like(tra))

    def follow(self, st, done):
        """Rays of one chunk until few are left; the finished ones go to done(id, e, a, steps)."""
        A, k, count = self.on["torch"], 0, st["w"].shape[0]
        few = max(2000, count // 50)
        while st["w"].shape[0] > few:
            ended, D = self.step(st, A, torch)
            done(st["id"][ended], (st["w"] * D)[ended], (st["wi"] * st["G"])[ended], st["steps"][ended])
            left = ~ended
            st = {q: v[..., left] for q, v in st.items()}
            k += 1
        return st

    def finish(self, st, done):
        st = self.follow(st, done)
        A = self.on["numpy"]
        st = {q: v.cpu().numpy() for q, v in st.items()}
        while st["w"].size:
            ended, D = self.step(st, A, np)
            if ended.any():
                put = [torch.tensor(x, device=DEV) for x in (st["id"][ended], (st["w"] * D)[ended],
                                                             (st["wi"] * st["G"])[ended], st["steps"][ended])]
                done(*put)
                st = {q: v[..., ~ended] for q, v in st.items()}

    def all_rays(self, cells, R, snap, done, chunk=1 << 22):
        """Follows rays 0..R-1 of `cells` (int64 tensor); done() gets the ray's index cell position * R + r."""
        left = []
        for b in range(0, len(cells) * R, chunk):
            q = torch.arange(b, min(b + chunk, len(cells) * R), device=DEV)
            st = self.start(cells[q // R], q % R, snap)
            st["id"] = q
            left.append(self.follow(st, done))
        self.finish({k: torch.cat([s[k] for s in left], dim=-1) for k in left[0]}, done)

    def sums(self, cells, R, snap):
        """E, A, Q and its standard error of every cell."""
        E, Ab, X2 = (torch.zeros(len(cells), dtype=torch.float64, device=DEV) for _ in range(3))

        def done(i, e, a, steps):
            for s, v in ((E, e), (Ab, a), (X2, (e - a) ** 2)):
                s.index_add_(0, i // R, v)

        self.all_rays(cells, R, snap, done)
        Q = E - Ab
        return E.cpu().numpy(), Ab.cpu().numpy(), Q.cpu().numpy(), torch.sqrt(((R * X2 - Q * Q) / (R - 1)).clamp(min=0)).cpu().numpy()


def _exact_train(case, seed):
    i, nbin, L = _train_inputs(case, seed), case["nbin"], learned.layout(case["nbin"])
    theta = torch.tensor(i["theta"], dtype=torch.float64, device=DEV)
    used = theta.clone()
    for a, b in (("W1", "b1"), ("W2", "b2"), ("W3", "b3")):                      # the products take BF16 weights
        used[L[a]:L[b]] = theta[L[a]:L[b]].float().bfloat16().double()
    used.requires_grad_(True)
    part = lambda a, b, s: used[L[a]:L[b]].reshape(s)  # noqa: E731
    X, wt = (torch.tensor(i[k], dtype=torch.float64, device=DEV) for k in ("X", "wt"))
    td, tb = (torch.tensor(i[k], dtype=torch.int64, device=DEV) for k in ("td", "tb"))
    h = torch.tanh(X @ part("W1", "b1", (6, 64)) + part("b1", "W2", (64,)))
    h = torch.tanh(h @ part("W2", "b2", (64, 64)) + part("b2", "W3", (64,)))
    Z = h @ part("W3", "b3", (64, L["noutp"])) + part("b3", "P", (L["noutp"],))
    ce = torch.nn.functional.cross_entropy
    loss = (wt * (ce(Z[:, :64], td, reduction="none") + ce(Z[:, 64:64 + nbin], tb, reduction="none"))).sum() / wt.sum()
    g, = torch.autograd.grad(loss, used)
    m, v = (torch.tensor(i[k], dtype=torch.float64, device=DEV) for k in ("m", "v"))
    m, v, t = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g, TRAIN_STEP + 1
    theta = theta - TRAIN_RATE * (m / (1 - 0.9 ** t)) / (torch.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
    return dict(loss=loss.detach(), grad=g, theta=theta, m=m, v=v)


def _exact_collect(case, seed):
    """Samples in the solver's order: 8^3 blocks of cells, x fastest among the blocks and inside them."""
    n, R = _grid(case), case["rays"]
    T = _fields(case, seed)[0]
    k, j, i = (a.ravel() for a in np.meshgrid(*(np.arange(m) for m in n[::-1]), indexing="ij"))
    cells = np.lexsort((i, j, k, i // 8, j // 8, k // 8))
    ex, N = _Exact(case, T), len(cells) * R
    wt = torch.zeros(N, dtype=torch.float64, device=DEV)

    def done(q, e, a, steps):
        wt[q] = (e - a).abs() / torch.sqrt(steps + COST0)

    ex.all_rays(torch.tensor(cells, device=DEV), R, 0, done)
    Td, Tmax, c = T.astype(np.float64), max(float(T.max()), 573.0), ex.centre
    X = np.zeros(n + (6,))
    X[..., 0] = (2.0 * c[1] / 2.0 - 1.0)[None, :, None]
    X[..., 1], X[..., 5] = Td / Tmax, 573.0 / Tmax
    for a in range(3):
        up, dn = np.roll(Td, -1, a), np.roll(Td, 1, a)
        x = c[a]
        if a == 1:
            up[:, -1], dn[:, 0] = Td[:, -1], Td[:, 0]
            span = np.append(x[1:], x[-1]) - np.append(x[0], x[:-1])
        else:
            span = np.full(n[a], 2.0 * LENGTHS[a] / n[a])
        X[..., 2 + a] = (up - dn) / span.reshape([-1 if b == a else 1 for b in range(3)]) / Tmax
    X = X.transpose(2, 1, 0, 3).reshape(-1, 6)[cells]
    return [np.repeat(X, R, axis=0), None, None, wt]


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    # the reference's sampling and the learned proposal draw from the library's own streams and rows: no other value
    # of the same draws exists; the largest cases take too long
    if kind in ("sampled", "learned") or _rays(case) * _crossings(case) > EXACT_MOST:
        return None
    if kind == "collect":
        return _exact_collect(case, seed)
    n, R = _grid(case), case["rays"]
    if kind == "fp64":
        cells = torch.tensor(_emitters(case, seed).astype(np.int64), device=DEV)
        E, A, Q, sd = _Exact(case, _fields(case, seed)[0]).sums(cells, R, 0)
        return dict(Q=Q, E=E, A=A, sdev=sd)
    cells = torch.arange(n[0] * n[1] * n[2], device=DEV)
    cube = lambda v: v.reshape(n[::-1]).transpose(2, 1, 0)  # noqa: E731
    if kind == "coupled":
        T = np.zeros(n, np.float32)
        for c, (s, e) in zip(_nondimensional(case, seed), _slabs(case)):
            T[:, s[1] - 1:e[1], s[2] - 1:e[2]] = (c[1:-1] * T_REF / T_PLUS + T_REF).astype(np.float32)
        _, _, Q, sd = _Exact(case, T).sums(cells, R, 0)
        k = n[2] // case["ranks"]
        full = [np.pad(cube(v) / SIGMA / T_REF ** 4, ((1, 1), (0, 0), (0, 0))) for v in (Q, sd)]
        return [tuple(v[:, :, r * k:(r + 1) * k] for v in full) for r in range(case["ranks"])]
    out = []
    fields = _fields(case, seed, case["snaps"])
    Tmax = max(float(T.max()) for T in fields)
    for s, T in enumerate(fields):
        _, _, Q, sd = _Exact(case, T, Tmax).sums(cells, R, s)
        out.append(tuple(np.pad(cube(v), 1) for v in (Q, sd)))
    return out
