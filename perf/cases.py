"""The performance cases of the framework: the calls that a Wigner-ensemble program makes, over the sizes it makes them at.

listed() names twelve of them, draw() gives more of the same ranges, prepare() makes what the program has in hand
before the call, run() is one pass through the public entry points, work() is what a pass cannot do without, and
exact() gives the pass's results in 64 bits from plain torch.

Results that were computed in single precision are returned as single precision (the binding widens them).
"""
import ctypes
import math

import numpy as np
import torch

import bec_amd as B
from bec_amd import fno as F
from bec_amd import surrogate as S

# the Rb-87 Ramsey cloud of the examples: 30000 atoms, losses on, vacuum noise in both components
CLOUD = dict(N=30000, a11=100.4, a12=97.66, a22=95.0, fx=97.6, fz=11.96, detuning=0.0, gamma111=5.4e-30,
             gamma12=0.78e-13, gamma22=1.5e-14)


def listed():
    return [
        # a small ensemble, where a step is two short launches; its state is saved at the end
        dict(name="evolve-8", kind="evolve", precision=0, nz=128, n=16, ne=8, nz_b=0, n_b=0, ne_b=0, steps=50, every=25, save=1),
        # the ordinary run: 64 trajectories, sampled
        dict(name="evolve-64", kind="evolve", precision=0, nz=128, n=16, ne=64, nz_b=0, n_b=0, ne_b=0, steps=100, every=50, save=0),
        # the largest ensemble of the benchmark
        dict(name="evolve-2048", kind="evolve", precision=0, nz=128, n=16, ne=2048, nz_b=0, n_b=0, ne_b=0, steps=20, every=10, save=0),
        # two uneven grids stepped together
        dict(name="evolve-uneven", kind="evolve", precision=0, nz=128, n=16, ne=256, nz_b=256, n_b=32, ne_b=128, steps=10, every=5, save=0),
        # the all-double run that the single-precision results are checked against
        dict(name="evolve-double", kind="evolve", precision=1, nz=128, n=32, ne=16, nz_b=0, n_b=0, ne_b=0, steps=20, every=10, save=0),
        # one displayed frame: a step, the observables and the density projections
        dict(name="frame-64", kind="frame", precision=0, nz=128, n=16, ne=64),
        # the ground state that every run starts from, by the default rule
        dict(name="ground-1", kind="ground", method="split", nz=128, n=16, sets=1),
        # two-component ground states of a block of parameter sets (training data of the learned start)
        dict(name="pair-16", kind="pair", nz=128, n=16, sets=16),
        # the learned start of one parameter set: input features and forward pass
        dict(name="guess-1", kind="guess", nz=128, n=16, modes=16, width=32, layers=4, hidden=64, batch=1),
        # training of the learned start: eight batches, then the checkpoint
        dict(name="train-16", kind="train", nz=128, n=16, modes=16, width=32, layers=4, hidden=64, batch=16, steps=8),
        # the 2D program with its own constants (half its equilibration: rounding differences grow by e every 15 steps)
        dict(name="plane-32", kind="plane", rule=0, nvx=64, nvy=64, ne=32, equil=100, meas=1),
        # the 1D program on its own lattice, the first steps of its run (e every 40 steps)
        dict(name="line-20", kind="line", dz=1.0, ne=20, steps=101),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["evolve", "evolve", "evolve", "frame", "ground", "pair", "guess", "train", "plane", "line"])
    if kind == "evolve":
        prec = rng.choice([0, 0, 0, 1])
        c = dict(kind=kind, precision=prec, nz=rng.choice([64, 128, 256]), n=rng.choice([16, 16, 32]), nz_b=0, n_b=0, ne_b=0)
        most = 2048 * 32768 // (c["nz"] * c["n"] ** 2) // (8 if prec else 1)
        c["ne"] = _log(rng, 1, most)
        if not prec and rng.random() < 0.25:
            c["nz_b"], c["n_b"] = rng.choice([64, 128, 256]), rng.choice([16, 32])
            c["ne"] = max(1, c["ne"] // 2)
            c["ne_b"] = _log(rng, 1, 1024 * 32768 // (c["nz_b"] * c["n_b"] ** 2))
        cells = c["ne"] * c["nz"] * c["n"] ** 2 + c["ne_b"] * c["nz_b"] * c["n_b"] ** 2
        c["save"] = int(cells <= 1 << 19 and rng.random() < 0.5)
        c["every"] = rng.randint(4, 10 if cells > 1 << 24 else 25 if c["save"] else 50)
        return dict(c, steps=c["every"] * rng.randint(1, 2))
    if kind == "frame":
        c = dict(kind=kind, precision=rng.choice([0, 0, 1]), nz=rng.choice([64, 128, 256]), n=rng.choice([16, 16, 32]))
        return dict(c, ne=_log(rng, 1, 512 * 32768 // (c["nz"] * c["n"] ** 2)))
    if kind == "ground":
        return dict(kind=kind, method=rng.choice(["split", "flow"]), nz=rng.choice([64, 128, 128, 256]), n=rng.choice([16, 16, 32]), sets=_log(rng, 1, 12))
    if kind == "pair":
        return dict(kind=kind, nz=rng.choice([64, 128, 128]), n=16, sets=_log(rng, 1, 24))
    if kind in ("guess", "train"):
        c = dict(kind=kind, nz=rng.choice([32, 64, 128]), n=rng.choice([8, 16]), modes=rng.choice([4, 8, 16]), width=rng.choice([8, 16, 32]), layers=rng.randint(1, 4),
                 hidden=rng.choice([16, 24, 32, 64]), batch=rng.randint(1, 16))
        c["modes"] = min(c["modes"], c["n"])
        return dict(c, steps=rng.randint(2, 8)) if kind == "train" else c
    if kind == "plane":
        return dict(kind=kind, rule=rng.choice([0, 2]), nvx=rng.choice([16, 32, 64]), nvy=rng.choice([16, 32, 64]), ne=_log(rng, 1, 256),
                    equil=rng.randint(1, 60), meas=rng.randint(1, 40))
    dz = rng.uniform(0.12, 2.0)   # 21 to 333 cells
    return dict(kind=kind, dz=dz, ne=_log(rng, 2, 1024), steps=rng.randint(10, 101 if dz > 0.6 else 30))


# ------------------------------------------------------------------ parameters

def _derived(nz, n, **kw):
    """The cloud in natural units (the trap's radial length and time), as plain numbers."""
    m = dict(CLOUD, **kw)
    hbar, a0, mass = 1.054571628e-34, 5.2917720859e-11, 1.443160648e-25
    w = 2 * math.pi * m["fx"]
    l = math.sqrt(hbar / (mass * w))
    lam = m["fx"] / m["fz"]
    c = dict(nz=nz, n=n, N=m["N"], lam=lam, det=2 * math.pi * m["detuning"] / w, l111=m["gamma111"] / 1e12 / (l ** 6 * w),
             l12=m["gamma12"] / 1e6 / (l ** 3 * w), l22=m["gamma22"] / 1e6 / (l ** 3 * w))
    for k in ("11", "12", "22"):
        c["g" + k] = 4 * math.pi * m["a" + k] * a0 / l
    c["mu"] = (15 * m["N"] * c["g11"] / (16 * math.pi * lam * math.sqrt(2))) ** 0.4
    c["xm"] = 1.2 * math.sqrt(2 * c["mu"])
    c["zm"] = lam * c["xm"]
    c["dx"], c["dz"] = 2 * c["xm"] / (n - 1), 2 * c["zm"] / (nz - 1)
    c["dV"] = c["dx"] ** 2 * c["dz"]
    c["dt_evo"], c["dt_steady"] = _step(n) * w, 1e-5 * w
    return c


def _step(n):
    """The time step that is stable on the lattice, in seconds."""
    return 4e-5 if n == 16 else 2e-5


def _calc(nz, n, ne, dt, **kw):
    m = {**CLOUD, "nvx": n, "nvy": n, "nvz": nz, "ne": ne, "fy": kw.get("fx", CLOUD["fx"]), "Va": 1.0, "Vb": 1.0,
         "t_equilib": 0.0, "itmax": 1, "dt_evo": dt, "dt_steady": 1e-5, **kw}
    return B.derive(B.default_model(**m))


def _grid(c, dev="cpu"):
    """x, y, z coordinates of the lattice, broadcastable over [z][y][x]."""
    t = lambda m, d, n: -m + d * torch.arange(n, dtype=torch.float64, device=dev)  # noqa: E731
    x = t(c["xm"], c["dx"], c["n"])
    return x[None, None, :], x[None, :, None], t(c["zm"], c["dz"], c["nz"])[:, None, None]


def _potential(c, dev="cpu"):
    x, y, z = _grid(c, dev)
    return 0.5 * (x ** 2 + y ** 2 + z ** 2 / c["lam"] ** 2)


def _kinetic(c, dev="cpu"):
    k = lambda n, m: (math.pi / m * torch.tensor([i - n if 2 * i > n else i for i in range(n)], dtype=torch.float64, device=dev)) ** 2 / 2  # noqa: E731
    kx = k(c["n"], c["xm"])
    return kx[None, None, :] + kx[None, :, None] + k(c["nz"], c["zm"])[:, None, None]


def _thomas_fermi(c, dev="cpu"):
    return torch.sqrt(torch.clamp(c["mu"] - _potential(c, dev), min=0) / c["g11"])


def _sets(case, seed):
    """Parameter sets (atoms, axial and radial trap frequency, a12) over the learned start's ranges."""
    rng = np.random.default_rng(seed)
    lo, hi = np.array([5e3, 5.0, 50.0, 95.0]), np.array([1e5, 20.0, 150.0, 100.0])
    th = lo + (hi - lo) * rng.random((case.get("sets") or case["batch"] * case.get("steps", 1), 4))
    return th, 2 * (th - lo) / (hi - lo) - 1


def _of_set(t):
    return dict(N=int(round(t[0])), fz=float(t[1]), fx=float(t[2]), a12=float(t[3]))


class _At:
    """A device address, as the binding takes one."""

    def __init__(self, address):
        self.ptr = ctypes.c_void_p(address)


# --------------------------------------------------------------------- prepare

def _groups(case):
    g = [(case["nz"], case["n"], case["ne"])]
    return g + [(case["nz_b"], case["n_b"], case["ne_b"])] if case.get("ne_b") else g


def _net(case, seed):
    m = case["modes"]
    cfg = dict(nz=case["nz"], ny=case["n"], nx=case["n"], mz=m, my=m, mx=m, width=case["width"], layers=case["layers"], c_in=16,
               c_out=2, hidden=case["hidden"], max_batch=case["batch"])
    net = F.FNO(seed=seed, **cfg)
    net.set_params(_weights(case, seed))
    return net


def _shapes(case):
    W, H, m = case["width"], case["hidden"], case["modes"]
    s = [("P", (16, W), 0.25), ("p", (W,), 0.25)]
    for _ in range(case["layers"]):
        s += [("W", (W, W), W ** -0.5), ("b", (W,), W ** -0.5), ("R", (m, m, m, W, W, 2), 1 / W)]
    return s + [("Q1", (W, H), W ** -0.5), ("q1", (H,), W ** -0.5), ("Q2", (H, 2), H ** -0.5), ("q2", (2,), H ** -0.5)]


def _weights(case, seed):
    rng = np.random.default_rng([seed, 1])
    return np.concatenate([(2 * rng.random(math.prod(s), dtype=np.float32) - 1) * np.float32(a) for _, s, a in _shapes(case)])


def _features(case, seed, dev="cuda"):
    """The network's input channels and smooth targets of every set: [set][cells][16], [set][cells][2], float32."""
    th, sc = _sets(case, seed)
    X = torch.zeros((len(th), case["nz"], case["n"], case["n"], 16), dtype=torch.float32, device=dev)
    Y = torch.empty((len(th), case["nz"], case["n"], case["n"], 2), dtype=torch.float32, device=dev)
    for i, t in enumerate(th):
        c = _derived(case["nz"], case["n"], **_of_set(t))
        x, y, z = _grid(c, dev)
        V = _potential(c, dev)
        tf = torch.sqrt(torch.clamp(c["mu"] - V, min=0) / c["mu"])
        for k, v in enumerate((tf, V / c["mu"], x / c["xm"], y / c["xm"], z / c["zm"], *sc[i])):
            X[i, ..., k] = v
        Y[i, ..., 0] = torch.exp(-V / c["mu"]) * (1 + 0.1 * sc[i][0])
        Y[i, ..., 1] = 0.3 * tf * sc[i][3] * torch.cos(z / c["zm"])
    return X.reshape(len(th), -1, 16), Y.reshape(len(th), -1, 2)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("evolve", "frame"):
        g = _groups(case)
        dt = min(_step(n) for _, n, _ in g)
        s = B.Solver(None, precision=case["precision"], groups=[_calc(nz, n, ne, dt) for nz, n, ne in g])
        for i, (nz, n, _) in enumerate(g):
            s.init_evolution(_thomas_fermi(_derived(nz, n)).numpy(), seed + 7 * i, group=i)
        return case, s
    if kind in ("ground", "pair"):
        th, _ = _sets(case, seed)
        return case, [_calc(case["nz"], case["n"], 1, _step(case["n"]), **_of_set(t)) for t in th]
    if kind == "guess":
        th, sc = _sets(case, seed)
        calcs = [_calc(case["nz"], case["n"], 1, 4e-5, **_of_set(t)) for t in th]
        cells = case["nz"] * case["n"] ** 2
        y = torch.empty((case["batch"], cells, 2), dtype=torch.float32, device="cuda")
        return case, _net(case, seed), calcs, sc, F.DeviceArray((case["batch"], cells, 16), np.float32), y
    if kind == "train":
        return case, _net(case, seed), *_features(case, seed)
    if kind == "plane":
        if case["rule"] == 0:
            return case, B.params2d(nvx=case["nvx"], nvy=case["nvy"], ne=case["ne"], ntW=case["equil"], n_meas=case["meas"], seed=seed)
        m = B.default_model(**dict(CLOUD, fy=CLOUD["fx"], nvx=case["nvx"], nvy=case["nvy"], nvz=2, ne=case["ne"], Va=1.0, Vb=1.0, dt_evo=1e-5))
        return case, B.params2d_from_model(m, ntW=case["equil"], n_meas=case["meas"], seed=seed)
    return case, B.params1d(dz=case["dz"], ne=case["ne"], ntW=case["steps"], seed=seed)


# ------------------------------------------------------------------------- run

def run(state):
    case, kind = state[0], state[0]["kind"]
    if kind == "evolve":
        s, num = state[1], (np.float64, np.complex128) if case["precision"] else (np.float32, np.complex64)
        out = [s.propagate(case["steps"], sample_every=case["every"]).astype(num[0], copy=False)]
        if case["save"]:
            out += [v.astype(num[1], copy=False) for v in s.get_state(B.SPACE_X)]
        return out
    if kind == "frame":
        o = state[1].calculate_evolution()[0]
        p = state[1].projections()
        num = np.float64 if case["precision"] else np.float32
        return dict(atoms=np.array([o[k] for k in ("Na", "Nb", "N_total", "N1", "N2", "Na_stderr", "Nb_stderr")], dtype=num),
                    fringe=np.array([o[k] for k in ("visibility_grid", "visibility", "phase")], dtype=num),
                    **{k: v.astype(num) for k, v in p.items()})
    if kind == "ground":
        o = {} if case["method"] == "split" else dict(method=B.GS_GRADIENT, rule=B.GS_RULE_RESIDUAL, tol=1e-6)
        out, reps, _ = B.ground_states_batched(state[1], **o)
        return _reported(out, reps, ("E_ref", "mu_ref", "E", "mu", "N"))
    if kind == "pair":
        out, reps, _ = B.ground_states_two_component(state[1], tol=1e-6)
        return _reported(out, reps, ("E", "mu_a", "mu_b", "N_a", "N_b"))
    if kind == "guess":
        _, net, calcs, sc, x, y = state
        for j, c in enumerate(calcs):
            F.gs2_features(c, sc[j], F.DeviceView(x, j * c.cells * 64))
        net.forward(x, _At(y.data_ptr()), case["batch"])
        return y
    if kind == "train":
        _, net, X, Y = state
        loss = []
        for j in range(0, len(X), case["batch"]):
            loss.append(net.loss_backward(_At(X[j].data_ptr()), _At(Y[j].data_ptr()), case["batch"]))
            net.adam_step(1e-3)
        return dict(loss=np.array(loss, dtype=np.float32), params=net.get_params())
    r = B.run_2d(state[1]) if kind == "plane" else B.run_1d(state[1])
    rep = r.pop("report")
    r["ground"] = np.array([rep["N0"], rep["gs_mu"]])
    r["residual"] = rep["gs_residual"]
    return r


def _reported(out, reps, keys):
    return dict(states=out, report=np.array([[r[k] for k in keys] for r in reps]), residual=np.array([r["residual"] for r in reps], dtype=np.float32),
                iterations=np.array([r["iterations"] for r in reps]))


# ------------------------------------------------------------------------ work

def work(case):
    """Bytes: states, weights, inputs and outputs once (for a real-time step: the state read and written, since a step
    needs all of it). Flops: radix-2 transforms and the products of the network."""
    kind = case["kind"]
    if kind in ("evolve", "frame"):
        by = fl = 0
        for nz, n, ne in _groups(case):
            cells = ne * nz * n * n
            by += cells * 32 * (2 if case["precision"] else 1)
            fl += cells * 2 * (2 * 5 * math.log2(nz * n * n) + 60)
        if kind == "frame":   # the step, then the observables and the projections read the state again
            return dict(bytes=2 * by, flops=2 * fl)
        return dict(bytes=by * (case["steps"] + case["save"]), flops=fl * case["steps"])
    if kind in ("ground", "pair"):
        cells = case["nz"] * case["n"] ** 2 * case["sets"] * (2 if kind == "pair" else 1)
        iters = 150 if kind == "pair" else 380 if case["method"] == "split" else 50
        return dict(bytes=cells * 16, flops=iters * cells * (4 if kind == "pair" or case["method"] == "flow" else 3) * 5 * math.log2(case["nz"] * case["n"] ** 2))
    if kind in ("guess", "train"):
        cells, b, W, H, L = case["nz"] * case["n"] ** 2, case["batch"], case["width"], case["hidden"], case["layers"]
        par = sum(math.prod(s) for _, s, _ in _shapes(case))
        one = b * cells * (2 * (16 * W + W * H + 2 * H) + L * (2 * W * W + W * 5 * math.log2(cells))) + b * L * case["modes"] ** 3 * 8 * W * W
        if kind == "guess":
            return dict(bytes=par * 2 + b * cells * 72, flops=one)
        return dict(bytes=case["steps"] * (par * 28 + b * cells * 72) + par * 4, flops=case["steps"] * 3 * one)
    if kind == "plane":
        n = case["nvx"] * case["nvy"]
        return dict(bytes=n * 8 * (2 + case["ne"]) + 40 * case["meas"], flops=case["ne"] * n * (case["equil"] + case["meas"]) * (20 * math.log2(n) + 120))
    n = 1 + 2 * int(20.0 / case["dz"])
    return dict(bytes=40 * case["steps"] + 24 * n, flops=case["ne"] * 2 * case["steps"] * n * (20 * math.log2(n) + 120))


# ----------------------------------------------------------------------- exact

_X, _K = torch.fft.fftn, torch.fft.ifftn   # to x-space (unnormalised, -i), to k-space (normalised, +i)
ZYX = (-3, -2, -1)


def _philox(cells, first, ntraj, seed):
    """The four noise deviates (deviation 0.5) of every cell of trajectories first .. first + ntraj: Philox4x32-10, Box-Muller."""
    m = 0xFFFFFFFF
    cell = torch.arange(cells, dtype=torch.int64, device="cuda").repeat(ntraj)
    c = [cell, torch.arange(first, first + ntraj, dtype=torch.int64, device="cuda").repeat_interleave(cells), torch.zeros_like(cell), torch.zeros_like(cell)]
    k0, k1 = seed & m, (seed >> 32) & m
    for _ in range(10):
        p0, p1 = c[0] * 0xD2511F53, c[2] * 0xCD9E8D57
        c = [((p1 >> 32) & m) ^ c[1] ^ k0, p1 & m, ((p0 >> 32) & m) ^ c[3] ^ k1, p0 & m]
        k0, k1 = (k0 + 0x9E3779B9) & m, (k1 + 0xBB67AE85) & m
    out = []
    for p in (0, 2):
        r = 0.5 * torch.sqrt(-2 * torch.log((c[p].double() + 1) / 2.0 ** 32))
        a = 2 * math.pi * ((c[p + 1].double() + 1) / 2.0 ** 32)
        out += [r * torch.cos(a), r * torch.sin(a)]
    return [v.reshape(ntraj, cells) for v in out]


def _start(gs, first, ntraj, seed, da, db):
    e = _philox(gs.numel(), first, ntraj, seed)
    shape = (ntraj, *gs.shape)
    return gs + da * torch.complex(e[0], e[1]).reshape(shape), db * torch.complex(e[2], e[3]).reshape(shape)


def _half_pi(a, b):
    return (a - 1j * b) / math.sqrt(2), (b - 1j * a) / math.sqrt(2)


def _real_time(c, dt, n, a, b, V, K):
    """n split steps of x-space fields."""
    half = torch.exp(0.5j * dt * K)
    for _ in range(n):
        a, b = _X(half * _K(a, dim=ZYX), dim=ZYX), _X(half * _K(b, dim=ZYX), dim=ZYX)
        na, nb = a.abs() ** 2, b.abs() ** 2
        a = a * torch.exp(dt * torch.complex(-(c["l111"] * na * na + c["l12"] * nb) / 2, V + c["g11"] * na + c["g12"] * nb))
        b = b * torch.exp(dt * torch.complex(-(c["l22"] * nb + c["l12"] * na) / 2, V + c["g22"] * nb + c["g12"] * na - c["det"]))
        a, b = _X(half * _K(a, dim=ZYX), dim=ZYX), _X(half * _K(b, dim=ZYX), dim=ZYX)
    return a, b


def _ensembles(case, seed):
    """(group index, parameters, step, a, b) of chunks of trajectories as init_evolution leaves them."""
    g = _groups(case)
    for i, (nz, n, ne) in enumerate(g):
        c = _derived(nz, n)
        dt = c["dt_evo"] * min(_step(m) for _, m, _ in g) / _step(n)
        V, K, gs = _potential(c, "cuda"), _kinetic(c, "cuda"), _thomas_fermi(c, "cuda").to(torch.complex128)
        chunk = max(1, (1 << 22) // (nz * n * n))
        for first in range(0, ne, chunk):
            a, b = _start(gs, first, min(chunk, ne - first), seed + 7 * i, c["dV"] ** -0.5, c["dV"] ** -0.5)
            a, b = _half_pi(*_real_time(c, dt, 1, a, b, V, K))
            yield i, c, dt, V, K, a, b


def _sums(a, b):
    ab = (a.conj() * b).sum(ZYX)
    return torch.stack([(a.abs() ** 2).sum(ZYX), (b.abs() ** 2).sum(ZYX), ab.real, ab.imag], -1)


def _exact_evolve(case, seed):
    rows, kept = [], []
    for i, c, dt, V, K, a, b in _ensembles(case, seed):
        got = []
        for _ in range(case["steps"] // case["every"]):
            a, b = _real_time(c, dt, case["every"], a, b, V, K)
            got.append(_sums(a, b))
        rows.append(torch.stack(got))
        if case["save"] and i == 0:
            kept.append((a, b))
    return [torch.cat(rows, 1), *(torch.cat(v) for v in zip(*kept))]


def _exact_frame(case, seed):
    sums, da, db = [], 0, 0
    for _, c, dt, V, K, a, b in _ensembles(case, seed):
        a, b = _real_time(c, dt, 1, a, b, V, K)
        sums.append(_sums(a, b))
        # the virtual pulse before the densities, alpha = 0
        da = da + (((a - 1j * b).abs() ** 2) / 2 - 0.5 / c["dV"]).sum(0)
        db = db + (((b - 1j * a).abs() ** 2) / 2 - 0.5 / c["dV"]).sum(0)
    s = torch.cat(sums).cpu().numpy()
    ne, dV = case["ne"], c["dV"]
    saa, sbb, sre, sim = s.sum(0)
    vac = case["nz"] * case["n"] ** 2 / (2 * dV)

    def rotated(al):
        x = math.sin(al) * sre + math.cos(al) * sim
        return (saa + sbb) / 2 + x - ne * vac, (saa + sbb) / 2 - x - ne * vac

    n1, n2 = rotated(0.0)
    grid = max(abs((abs(p) - abs(q)) / (abs(p) + abs(q))) for p, q in (rotated(0.5 * i) for i in range(13)))
    pop = [(0.5 * (s[:, 0] + s[:, 1]) + sg * s[:, 3] - vac) * dV for sg in (1, -1)]
    err = [float(np.std(p) / math.sqrt(ne - 1)) if ne > 1 else 0.0 for p in pop]
    N1, N2 = saa - ne * vac, sbb - ne * vac
    r = dict(atoms=np.array([n1 * dV, n2 * dV, (n1 + n2) * dV / ne, N1 * dV, N2 * dV, *err]),
             fringe=np.array([grid, 2 * math.hypot(sre, sim) / (N1 + N2), math.atan2(sim, sre)]))
    for k, d in (("a", da), ("b", db)):
        r.update({"xy_" + k: d.sum(0), "zy_" + k: d.sum(2).T.contiguous(), "axial_" + k: d.sum((1, 2))})
    return r


def _exact_split(c):
    V, K, N, hdt = _potential(c, "cuda"), _kinetic(c, "cuda"), c["N"], 0.5 * c["dt_steady"]
    x = _thomas_fermi(c, "cuda").to(torch.complex128)
    s, prev, half = math.sqrt(N / (c["dV"] * float((x.abs() ** 2).sum()))), 0.0, torch.exp(-hdt * K)
    it = 0
    while True:
        a = _X(half * _K(x * s))
        x = a * torch.exp(2 * hdt * (-V - c["g11"] * a.abs() ** 2))
        k = half * _K(x)
        x, it = _X(k), it + 1
        n = x.abs() ** 2
        s2 = N / (c["dV"] * float(n.sum()))
        e1 = float((n * V).sum() + ((x * k).real * K).sum())
        E = c["dV"] * (s2 * e1 + c["g11"] * s2 * s2 * float((n * n).sum()) / 2)
        s = math.sqrt(s2)
        if abs((E - prev) / E) < 1e-6:
            return x * s, it
        prev = E


def _exact_flow(c, V, K, g, g12, target, tau, beta):
    """The preconditioned gradient flow of one (g = [g11]) or two coupled components to residual 1e-6."""
    x = [_thomas_fermi(c, "cuda").to(torch.complex128) for _ in g]
    scale = lambda v, n: v * math.sqrt(n / (c["dV"] * float((v.abs() ** 2).sum())))  # noqa: E731
    x = [scale(v, n) for v, n in zip(x, target)]
    prev, it = list(x), 0
    while True:
        h = [_X(K * _K(v)) + (V + g[i] * v.abs() ** 2 + (g12 * x[1 - i].abs() ** 2 if len(g) > 1 else 0)) * v for i, v in enumerate(x)]
        mu = [float((v.conj() * u).real.sum() / (v.abs() ** 2).sum()) for v, u in zip(x, h)]
        r = [u - m * v for v, u, m in zip(x, h, mu)]
        res = max(math.sqrt(float((q.abs() ** 2).sum() / (v.abs() ** 2).sum())) / abs(m) for v, q, m in zip(x, r, mu))
        if res < 1e-6 or it > 20000:
            return x, it
        d = [_X(_K(q) / (c["mu"] + K)) for q in r]
        x, prev = [scale(v - tau * p + beta * (v - o), n) for v, p, o, n in zip(x, d, prev, target)], x
        it += 1


def _exact_ground(case, seed):
    pair = case["kind"] == "pair"
    if (1 if pair else 4) * case["sets"] > 16:
        return None
    states, rows, res = [], [], []
    for t in _sets(case, seed)[0]:
        c = _derived(case["nz"], case["n"], **_of_set(t))
        V, K, dV = _potential(c, "cuda"), _kinetic(c, "cuda"), c["dV"]
        if pair:
            x, _ = _exact_flow(c, V, K, [c["g11"], c["g22"]], c["g12"], [c["N"] / 2] * 2, 1.0, 0.85)
        elif case["method"] == "flow":
            x, _ = _exact_flow(c, V, K, [c["g11"]], 0.0, [c["N"]], 0.5, 0.6)
        else:
            x = [_exact_split(c)[0]]
        n = [v.abs() ** 2 for v in x]
        kin = [_X(K * _K(v)) for v in x]
        g = [c["g11"], c["g22"]]
        h = [k + (V + g[i] * n[i] + (c["g12"] * n[1 - i] if pair else 0)) * v for i, (v, k) in enumerate(zip(x, kin))]
        mu = [float((v.conj() * u).real.sum() / m.sum()) for v, u, m in zip(x, h, n)]
        res.append(max(math.sqrt(float(((u - m * v).abs() ** 2).sum() / q.sum())) / abs(m) for v, u, m, q in zip(x, h, mu, n)))
        atoms = [float(m.sum()) * dV for m in n]
        kp = sum(float((v.conj() * k).real.sum() + (V * m).sum()) for v, k, m in zip(x, kin, n)) * dV
        if pair:
            rows.append([(kp + atoms[0] * mu[0] + atoms[1] * mu[1]) / 2 / sum(atoms), *mu, *atoms])
            states.append(torch.stack(x))
        else:
            q = float((n[0] ** 2).sum()) * dV * c["g11"]
            ref = float((n[0] * V).sum() + ((x[0] * _K(x[0])).real * K).sum()) * dV
            rows.append([(ref + q / 2) / c["N"], (ref + q) / c["N"], (kp + q / 2) / atoms[0], mu[0], atoms[0]])
            states.append(x[0])
    return dict(states=torch.stack(states), report=np.array(rows), residual=np.array(res), iterations=None)


def _unpacked(case, seed, grad=False):
    flat, at, out = torch.from_numpy(_weights(case, seed)).double().cuda(), 0, []
    for name, s, _ in _shapes(case):
        out.append((name, flat[at:at + math.prod(s)].reshape(s).clone().requires_grad_(grad)))
        at += math.prod(s)
    return out


def _network(case, p, x):
    p, m, n, nz = iter(t for _, t in p), case["modes"], case["n"], case["nz"]
    kz = [i if i < m // 2 else nz + i - m for i in range(m)]
    kx = [i if i < (m + 1) // 2 else n + i - m for i in range(m)]
    at = torch.tensor([(z * n + y) * n + x_ for z in kz for y in kx for x_ in kx], device=x.device)
    b, W = x.shape[0], case["width"]
    h = x @ next(p) + next(p)
    for l in range(case["layers"]):
        w, bias, R = next(p), next(p), torch.view_as_complex(next(p)).reshape(-1, W, W)
        sp = torch.fft.fftn(h.reshape(b, nz, n, n, W), dim=(1, 2, 3), norm="ortho").reshape(b, -1, W)[:, at]
        t = torch.matmul(sp.transpose(0, 1), R).transpose(0, 1)
        full = torch.zeros((b, nz * n * n, W), dtype=torch.complex128, device=x.device).index_copy(1, at, t)
        u = torch.fft.ifftn(full.reshape(b, nz, n, n, W), dim=(1, 2, 3), norm="ortho").real.reshape(b, -1, W) + h @ w + bias
        h = torch.nn.functional.gelu(u) if l < case["layers"] - 1 else u
    return torch.nn.functional.gelu(h @ next(p) + next(p)) @ next(p) + next(p)


def _exact_train(case, seed):
    p = _unpacked(case, seed, True)
    X, Y = _features(case, seed)
    m, v, loss = [0.0] * len(p), [0.0] * len(p), []
    for k in range(case["steps"]):
        at = slice(k * case["batch"], (k + 1) * case["batch"])
        e = ((_network(case, p, X[at].double()) - Y[at].double()) ** 2).mean()
        loss.append(float(e.detach()))
        g = torch.autograd.grad(e, [t for _, t in p])
        with torch.no_grad():
            for i, (_, t) in enumerate(p):
                m[i], v[i] = 0.9 * m[i] + 0.1 * g[i], 0.999 * v[i] + 0.001 * g[i] ** 2
                t -= 1e-3 * (m[i] / (1 - 0.9 ** (k + 1))) / (torch.sqrt(v[i] / (1 - 0.999 ** (k + 1))) + 1e-8)
    return dict(loss=np.array(loss), params=torch.cat([t.detach().reshape(-1) for _, t in p]))


def _spread(q, ne):
    """Ensemble mean and standard error over the first axis."""
    return q.mean(0), torch.sqrt(torch.abs((q * q).mean(0) - q.mean(0) ** 2) / (ne - 1)) if ne > 1 else torch.zeros_like(q[0])


def _exact_program(case, seed):
    """The 2D and the 1D program: imaginary-time ground state, noisy ensemble, pulse, sampled steps."""
    line = case["kind"] == "line"
    k2_of = lambda n, m: (math.pi / m * torch.tensor([i - n if 2 * i > n else i for i in range(n)], dtype=torch.float64, device="cuda")) ** 2  # noqa: E731
    at = lambda n, m, d: (-m + d * torch.arange(n, dtype=torch.float64, device="cuda")) ** 2  # noqa: E731
    q = dict(g11=6.18, g12=6.03, g22=5.88, E=2.5, mu=26.8, Va=0.2, Vb=0.5, dtG=1 / 31, steps=31, itmax=3, dt=0.01, rule=0)
    if line:
        n, dz = 1 + 2 * int(20.0 / case["dz"]), case["dz"]
        q.update(Va=0.5, Vb=1.0, dtG=0.01, steps=100)
        r2, k2, dv, dim, dev = at(n, 20.0, dz), k2_of(n, 20.0), dz, (-1,), math.sqrt(1 / dz) / 2
        equil, meas = case["steps"], case["steps"]
    else:
        nx, ny, xm = case["nvx"], case["nvy"], 20.0
        if case["rule"] == 2:
            hbar, mass, w = 1.054571628e-34, 1.443160648e-25, 2 * math.pi * CLOUD["fx"]
            k = 4 * math.sqrt(2 * math.pi) * 5.2917720859e-11 / math.sqrt(hbar / (mass * 2 * math.pi * CLOUD["fz"]))
            q.update({"g" + s: k * CLOUD["a" + s] for s in ("11", "12", "22")}, E=0.0, Va=1.0, Vb=1.0, dt=1e-5 * w, rule=2)
            q["mu"] = math.sqrt(q["g11"] * CLOUD["N"] / (2 * math.pi))
            xm = 2.4 * math.sqrt(q["mu"])
        n, dx, dy = nx * ny, 2 * xm / (nx - 1), 2 * xm / (ny - 1)
        r2, k2 = at(ny, xm, dy)[:, None] + at(nx, xm, dx)[None], k2_of(ny, xm)[:, None] + k2_of(nx, xm)[None]
        dv, dim, dev = dx * dy, (-2, -1), (1.0 if case["rule"] == 0 else 0.5) / math.sqrt(dx * dy)
        equil, meas = case["equil"], case["meas"]
    to_x, to_k = lambda v: _X(v, dim=dim), lambda v: _K(v, dim=dim)  # noqa: E731
    ham = lambda v: to_x(k2 * to_k(v)) + (r2 / 4 + q["g11"] * v.abs() ** 2) * v  # noqa: E731
    ray = lambda v: float((v.conj() * ham(v)).real.sum() / (v.abs() ** 2).sum())  # noqa: E731
    resid = lambda v, m: float(torch.sqrt(((ham(v) - m * v).abs() ** 2).sum() / (v.abs() ** 2).sum())) / abs(m)  # noqa: E731
    ntot = []
    if q["rule"] == 2:
        scale = lambda v: v * math.sqrt(CLOUD["N"] / (dv * float((v.abs() ** 2).sum())))  # noqa: E731
        x = scale(torch.sqrt(torch.clamp(q["mu"] - r2 / 4, min=0) / q["g11"]).to(torch.complex128))
        prev = x
        while True:
            m = ray(x)
            if resid(x, m) < 1e-8:
                break
            d = to_x(to_k(ham(x) - m * x) / (q["mu"] + k2))
            x, prev = scale(x - 0.5 * d + 0.6 * (x - prev)), x
    else:
        k, half = to_k(torch.ones_like(r2).to(torch.complex128)), torch.exp(-k2 * q["dtG"] / 2)
        ntot.append(float((k.abs() ** 2).sum()) * dv * n)
        for _ in range(q["steps"]):
            a1 = to_x(half * k)
            a = a1
            for _ in range(q["itmax"]):
                f = torch.exp(q["dtG"] / 2 * (q["mu"] - r2 / 4 - q["g11"] * a.abs() ** 2))
                a = a1 * f
            k = half * to_k(a * f)
            ntot.append(float((k.abs() ** 2).sum()) * dv * n)
        x = to_x(k)
    N0, mu = float((x.abs() ** 2).sum()) * dv, ray(x)
    ne, V = case["ne"], (q["Va"] + q["Vb"]) / 2
    a, b = _start(x, 0, ne, seed, q["Va"] * dev / 0.5, q["Vb"] * dev / 0.5)
    a, b = to_k(a), to_k(b)
    kin, got = torch.exp(0.5j * q["dt"] * k2), []
    for t in range(-equil, meas):
        if t > -equil:
            if t == 0:
                a, b = _half_pi(a, b)
            a, b = to_x(kin * a), to_x(kin * b)
            na, nb = a.abs() ** 2, b.abs() ** 2
            a = a * torch.exp(-1j * q["dt"] * (q["mu"] - r2 / 4 - q["g11"] * na - q["g12"] * nb + q["E"] / 2))
            b = b * torch.exp(-1j * q["dt"] * (q["mu"] - r2 / 4 - q["g22"] * nb - q["g12"] * na - q["E"] / 2))
            a, b = kin * to_k(a), kin * to_k(b)
        if t >= 0:
            ab = (a.conj() * b).sum(dim).abs()
            got.append(torch.stack([n * (((a + 1j * b).abs() ** 2).sum(dim) / 2 * dv - V / 2), n * (((b + 1j * a).abs() ** 2).sum(dim) / 2 * dv - V / 2),
                                    2 * ab / ((a.abs() ** 2).sum(dim) + (b.abs() ** 2).sum(dim))], -1))
    got = torch.stack(got, 1)   # [trajectory][sample][N1, N2, visibility]
    mean, err = _spread(got[..., :2], ne)
    r = dict(m=mean.T.contiguous(), var=err.T.contiguous(), vis=got[..., 2].mean(0), gs=x, avn=(to_x(a).abs() ** 2 - V / 2 / dv).mean(0),
             ground=np.array([N0, mu]), residual=resid(x, mu))
    return dict(r, ntot=np.array(ntot)) if line else r


def exact(case, seed):
    kind = case["kind"]
    if kind == "evolve":
        return _exact_evolve(case, seed)
    if kind == "frame":
        return _exact_frame(case, seed)
    if kind in ("ground", "pair"):
        return _exact_ground(case, seed)
    if kind == "guess":
        with torch.no_grad():
            return _network(case, _unpacked(case, seed), _features(case, seed)[0].double())
    if kind == "train":
        return _exact_train(case, seed)
    return _exact_program(case, seed)
