"""Performance cases of the channel-flow library: what its users run.

A case is a dict of plain values.  Five kinds:

  run       one channel marched `steps` RK3 steps (compute_dt +
            compute_time_step_RK3 without a host round trip), with the
            monitoring of the reference's loop (divergence, plane statistics,
            wall shear) every `monitor` steps when that is not 0, then the
            velocity read back, as a run does between two snapshots;
  coupled   the reference's loop with a host wall-stress hook: alpha_x
            uploaded, compute_dt read, one RK3 step, `steps` times, then the
            whole state with the true pressure;
  agents    the RL loop on the device: observe, act, one step, `steps` times;
  ensemble  many channels of uneven size and Re_tau in one launch per stage;
  train     the learned wall model: one epoch of Adam on a sample set, then
            inference on a validation set.

Grids are given by their face counts (nx ny nz faces: nx-2, ny-1, nz-2 unique
cells).  `run` returns the whole resulting fields.  Those of an FP32-bulk
channel come back as float32, which is what the device holds.
"""
import math

import numpy as np
import torch

import channel_rl_amd as cr
from channel_rl_amd import cases as C
from channel_rl_amd.ensemble import make_channel

# the units of the reference's shipped parameters: u_tau = 0.0413, U ~ 1
UTAU = math.sqrt(0.001705857682121)
KAPPA, B = 0.41, 5.2


def _run(name, nx, ny, nz, precision="fp64", les="dsm", wall="equilibrium", mass=1, re_tau=2000.0, h_wm=0.1,
         lx=2.0 * math.pi, steps=50, monitor=0, tune=False):
    return dict(name=name, kind="run", nx=nx, ny=ny, nz=nz, precision=precision, les=les, wall=wall, mass=mass,
                re_tau=re_tau, h_wm=h_wm, lx=lx, steps=steps, monitor=monitor, tune=tune)


def listed():
    return [
        # the smallest configuration, 32x33x32 cells: launches and latency count
        _run("small", 34, 33, 34, re_tau=180.0, mass=2, h_wm=0.0, steps=100),
        # a ragged mid-size grid (radix 3 and 5 lengths, rows that fill no tile)
        # of the FP32 bulk with the default tile shapes, as the driver program runs it
        _run("ragged_fp32", 122, 59, 92, "fp32", mass=2, steps=150),
        # a mid-size FP64 run with the reference's monitoring in the loop
        _run("monitored", 98, 65, 98, mass=2, steps=120, monitor=20),
        # the WMLES configuration, FP64 (the headline) and FP32 bulk, tuned once
        _run("wmles", 194, 97, 194, tune=True, steps=150),
        _run("wmles_fp32", 194, 97, 194, "fp32", tune=True, steps=150),
        # the same channel with the AMD model the shipped case uses, and with
        # the learned wall model
        _run("wmles_amd", 194, 97, 194, les="amd", steps=150),
        _run("wmles_network", 194, 97, 194, "fp32", wall="network", tune=True, steps=150),
        # the large single channel, FP32 bulk
        _run("large_fp32", 386, 193, 386, "fp32", re_tau=5200.0, lx=4.0 * math.pi, tune=True, steps=80),
        # the shipped production grid (fixed dt, AMD) with the wall stress from the host
        dict(name="coupled", kind="coupled", nx=130, ny=41, nz=66, precision="fp64", les="amd", re_tau=2003.0, steps=60),
        # the same grid with the RL coupling on the device
        dict(name="agents", kind="agents", nx=130, ny=41, nz=66, precision="fp64", les="amd", re_tau=2003.0, agents=16,
             steps=60),
        # the batched ensemble: FP32 bulk, learned wall model in the loop
        dict(name="ensemble", kind="ensemble", members=64, precision="fp32", wall="network", steps=100),
        # training the wall model at its default batch
        dict(name="train", kind="train", samples=131072, batch=1024),
    ]


_SMOOTH = sorted(n for n in (2 ** a * 3 ** b * 5 ** c for a in range(1, 9) for b in range(4) for c in range(3))
                 if 16 <= n <= 384)


def draw(rng):
    kind = rng.choices(("run", "coupled", "agents", "ensemble", "train"), (8, 1, 1, 1, 1))[0]
    if kind == "train":
        return dict(kind=kind, samples=int(math.exp(rng.uniform(math.log(3000), math.log(131072)))),
                    batch=rng.choice((256, 512, 1024, 2048)))
    if kind == "ensemble":
        precision = rng.choice(("fp32", "fp64"))
        return dict(kind=kind, members=rng.randint(5, 64), precision=precision,
                    wall="network" if precision == "fp32" and rng.random() < 0.6 else "equilibrium",
                    steps=rng.randint(20, 60))

    def periodic(top):
        # an even number of cells of the lengths the FFTs take, log-uniform
        want = math.exp(rng.uniform(math.log(16), math.log(top)))
        return min(_SMOOTH, key=lambda n: abs(n - want) + rng.random()) + 2

    if kind in ("coupled", "agents"):
        nx, ny, nz = periodic(160), rng.randint(17, 65), periodic(160)
        c = dict(kind=kind, nx=nx, ny=ny, nz=nz, precision="fp64", les=rng.choice(("amd", "dsm")), re_tau=2003.0,
                 steps=rng.randint(10, 60))
        if kind == "agents":
            c["agents"] = rng.choice([a for a in (4, 8, 10, 12, 16, 20, 24, 32) if (nx - 2) % a == 0] or [nx - 2])
        return c
    nx, ny, nz = periodic(384), int(math.exp(rng.uniform(math.log(17), math.log(193)))), periodic(384)
    precision = rng.choice(("fp64", "fp32"))
    # the length of a run such that it costs at most half the large channel's
    most = 0.5 * 80 * 384 * 192 * 384 / ((nx - 2) * (ny - 1) * (nz - 2)) * (0.6 if precision == "fp64" else 1.0)
    steps = max(1, min(rng.randint(20, 150), int(most)))
    wall = "network" if precision == "fp32" and rng.random() < 0.3 else "equilibrium"
    c = _run("", nx, ny, nz, precision, rng.choice(("dsm", "dsm", "amd")), wall, rng.choice((0, 1, 2)),
             round(math.exp(rng.uniform(math.log(500), math.log(5200))), 1), rng.choice((0.05, 0.1, 0.2)),
             (4.0 if nx > 200 else 2.0) * math.pi, steps, rng.choice((0, 0, 10)), rng.random() < 0.4)
    del c["name"]
    return c


# ------------------------------------------------------------------ inputs

def _field(case, profile, amp, seed):
    """A raw initial field: the mean profile on U plus uniform noise of
    amp times the local mean on every component (drawn on the GPU)."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)
    yg = C.centres_with_ghosts(case.y)
    centre = profile(np.minimum(yg, 2.0 - yg))
    face = profile(np.maximum(np.minimum(case.y, 2.0 - case.y), 0.0))
    out = []
    for q, (n1, n2, n3) in enumerate(case.field_shapes()):
        m = torch.from_numpy(np.ascontiguousarray(face if q == 1 else centre)).cuda()
        r = torch.rand((n3, n2, n1), generator=g, device="cuda", dtype=torch.float64).mul_(2.0).sub_(1.0)
        f = r.mul_((amp * m)[None, :, None])
        if q == 0:
            f += m[None, :, None]
        out.append(f.cpu().numpy().transpose(2, 1, 0))
    return tuple(out)


def _case(c, cfl=0.5):
    nu = UTAU / c["re_tau"]
    case = C.Case("case", c["nx"], c["ny"], c["nz"], c.get("lx", 2.0 * math.pi), c.get("lx", 2.0 * math.pi) / 2.0,
                  C.tanh_y(c["ny"], 1.5), nu=nu, dPdx=UTAU ** 2, CFL=cfl, x_mass_cte=c.get("mass", 1),
                  LES_model={"dsm": 2, "amd": 3}[c["les"]], h_wm=c.get("h_wm", 0.1))
    if case.x_mass_cte == 2:
        case.wm_nu_limit = 0.25
    return case


def _loglaw(nu, utau):
    return lambda d: utau * C.loglaw_plus(d * utau / nu)


def _precision(c):
    return {"fp64": cr.FP64, "fp32": cr.FP32_BULK}[c["precision"]]


def _round_bf16(a):
    return torch.from_numpy(np.asarray(a, np.float32)).bfloat16().double().numpy()


def _network(seed):
    """A wall network as a program has it in hand after training: it carries
    the log law o0(f0) to about 1% (random hidden layers, the last one fitted
    by least squares) and ignores the other features."""
    rng = np.random.default_rng(seed)
    yp = np.exp(rng.uniform(math.log(4.0), math.log(2500.0), 8192))
    f0, o0 = np.arcsinh(yp * C.loglaw_plus(yp, KAPPA, B) / 10.0), np.log1p(yp * yp)
    xm, xs, ym, ys = f0.mean(), f0.std(), o0.mean(), o0.std()
    W1 = np.zeros((4, 64))
    W1[0] = rng.choice([-3.0, 3.0], 64) * rng.uniform(0.7, 1.3, 64)
    b1 = -W1[0] * rng.uniform(-2.0, 2.0, 64)
    W2, W3 = (rng.uniform(-1.0, 1.0, (64, 64)) * math.sqrt(6.0 / 64.0) for _ in range(2))
    h = _round_bf16(_silu(((f0 - xm) / xs)[:, None] * _round_bf16(W1[0]) + b1))
    h = _round_bf16(_silu(h @ _round_bf16(W2)))
    h = np.c_[_round_bf16(_silu(h @ _round_bf16(W3))), np.ones(len(f0))]
    w = np.linalg.solve(h.T @ h + 1e-5 * len(f0) * np.eye(65), h.T @ ((o0 - ym) / ys))
    W4 = np.zeros((64, 2))
    W4[:, 0] = w[:64]
    z = np.zeros(64)
    params = np.concatenate([W1.ravel(), b1, W2.ravel(), z, W3.ravel(), z, W4.ravel(), [w[64], 0.0]])
    norm = np.array([xm, 0, 0, 0, xs, 8.0, 4.0, 15.0, ym, 0.0, ys, 1.0])
    net = cr.WallNetwork(seed=int(seed) & 0xFFFF)
    net.set_params(params.astype(np.float32), norm.astype(np.float32))
    return net


def _silu(z):
    return z / (1.0 + np.exp(-z))


def _channel(c, seed, net=None):
    case = _case(c)
    ch = make_channel(case, _field(case, _loglaw(case.nu, UTAU), 0.1, seed), precision=_precision(c),
                      wall=cr.WALL_MLP if net is not None else cr.WALL_EQUILIBRIUM, net=net)
    if c.get("tune"):
        ch.autotune(reps=5)
    return ch


def _samples(rng, n):
    """Raw features over the training ranges with the log law's targets."""
    yp = np.exp(rng.uniform(math.log(0.5), math.log(3000.0), n))
    X = np.empty((n, 4), np.float32)
    X[:, 0] = np.arcsinh(yp * C.loglaw_plus(yp, KAPPA, B) / 10.0)
    X[:, 1] = rng.uniform(-12.0, 12.0, n)
    X[:, 2] = rng.uniform(0.0, 10.0, n)
    X[:, 3] = rng.uniform(-25.0, 25.0, n)
    Y = np.zeros((n, 2), np.float32)
    Y[:, 0] = np.log1p(yp * yp)
    return X, Y


def _training_set(rng, n):
    """Samples, validation features, He-uniform parameters and the samples'
    standardisation."""
    X, Y = _samples(rng, n)
    Xv = _samples(rng, max(1024, n // 8))[0]
    p = [rng.uniform(-1.0, 1.0, a * b) * math.sqrt(6.0 / a) if b else np.zeros(a)
         for a, b in ((4, 64), (64, 0), (64, 64), (64, 0), (64, 64), (64, 0), (64, 2), (2, 0))]
    ys = Y.std(axis=0, dtype=np.float64)
    ys[1] = 1.0
    norm = np.concatenate([X.mean(axis=0, dtype=np.float64), X.std(axis=0, dtype=np.float64),
                           Y.mean(axis=0, dtype=np.float64), ys])
    return X, Y, Xv, np.concatenate(p).astype(np.float32), norm.astype(np.float32)


def _grids(n):
    """The grids of an ensemble of n members, the same for every seed."""
    rng = np.random.default_rng(42)
    return [C.ENSEMBLE_GRIDS[int(rng.integers(len(C.ENSEMBLE_GRIDS)))] for _ in range(n)]


def prepare(case, seed):
    c = dict(case)
    kind = c["kind"]
    rng = np.random.default_rng(seed)
    if kind == "run":
        net = _network(seed) if c["wall"] == "network" else None
        return dict(c=c, ch=_channel(c, seed, net), net=net)
    if kind in ("coupled", "agents"):
        cc = _case(c, cfl=-1e-2)
        ch = make_channel(cc, _field(cc, _loglaw(cc.nu, UTAU), 0.05, seed), wall=cr.WALL_GIVEN)
        ch.compute_equilibrium_wall_stress(h_wm=0.1)
        s = dict(c=c, ch=ch)
        if kind == "coupled":
            alpha = ch.get_field(cr.ALPHA_X)
            s["alpha"] = [np.asfortranarray(alpha * rng.uniform(0.95, 1.05, alpha.shape)) for _ in range(c["steps"])]
        else:
            # the agents' factors: the second half takes the first half back,
            # so that a long run's wall stress does not wander off
            n, na = c["steps"], c["agents"]
            f = rng.uniform(0.97, 1.03, (n, 2, na))
            for q in range(n // 2):
                f[n - 1 - q] = 1.0 / f[q]
            s["factors"], s["draws"] = f, rng.uniform(0.0, 1.0, (n, 2, na, 2))
        return s
    if kind == "ensemble":
        net = _network(seed) if c["wall"] == "network" else None
        chans = []
        for q, (nx, ny, nz) in enumerate(_grids(c["members"])):
            re_tau = float(np.exp(rng.uniform(math.log(180.0), math.log(5200.0))))
            m = C.Case(f"member{q}", nx, ny, nz, 2 * math.pi, math.pi, C.tanh_y(ny, 1.5), nu=1.0 / re_tau, dPdx=1.0,
                       CFL=0.5, x_mass_cte=2, h_wm=0.1)
            m.wm_nu_limit = 0.25
            chans.append(make_channel(m, _field(m, _loglaw(m.nu, 1.0), 0.1, seed + 1 + q), precision=_precision(c),
                                      wall=cr.WALL_MLP if net is not None else cr.WALL_EQUILIBRIUM, net=net))
        return dict(c=c, chans=chans, ens=cr.Ensemble(chans), net=net)
    if kind == "train":
        X, Y, Xv, p0, norm = _training_set(rng, c["samples"])
        net = cr.WallNetwork(seed=1)
        net.set_params(p0, norm)
        return dict(c=c, net=net, X=X, Y=Y, Xv=Xv, p0=p0, seed=int(seed) & 0xFFFF)
    raise KeyError(kind)


# -------------------------------------------------------------------- a pass

def _fields(c, *a):
    return [np.asarray(x, np.float32) for x in a] if c["precision"] == "fp32" else list(a)


def run(s):
    c, ch = s["c"], s.get("ch")
    kind = c["kind"]
    if kind == "run":
        out = {}
        if c["monitor"]:
            seen = []
            for q in range(0, c["steps"], c["monitor"]):
                ch.run_steps(min(c["monitor"], c["steps"] - q))
                ch.check_divergence()
                ch.wall_shear()
                seen.append(ch.plane_statistics())
            # round-off of sums over a plane is not a field's: float32 for either precision
            out["profiles"] = np.stack(seen).astype(np.float32)
        else:
            ch.run_steps(c["steps"])
        out["U"], out["V"], out["W"] = _fields(c, *ch.state())
        return out
    if kind == "coupled":
        dts = []
        for a in s["alpha"]:
            ch.set_field(cr.ALPHA_X, a)
            dts.append(ch.compute_dt())
            ch.compute_time_step_RK3()
        U, V, W = ch.state()
        nu_t = ch.get_field(cr.NU_T)
        return dict(dt=np.array(dts), U=U, V=V, W=W, nu_t=nu_t, P=ch.compute_pressure())
    if kind == "agents":
        states, rewards = [], []
        for d, f in zip(s["draws"], s["factors"]):
            st, rw = ch.rl_observe(c["agents"], UTAU ** 2, d)
            states.append(st)
            rewards.append(rw)
            ch.rl_act(c["agents"], f)
            ch.run_steps(1)
        U, V, W = ch.state()
        return dict(states=np.stack(states), rewards=np.stack(rewards), U=U, V=V, W=W)
    if kind == "ensemble":
        s["ens"].run_steps(c["steps"])
        # one array a member, as a checkpoint packs it
        t = np.float32 if c["precision"] == "fp32" else np.float64
        return [np.concatenate([f.ravel(order="K") for f in m.state()], dtype=t, casting="same_kind") for m in s["chans"]]
    net = s["net"]
    net.set_params(s["p0"])
    loss = net.train(s["X"], s["Y"], epochs=1, batch=c["batch"], lr=1e-3, seed=s["seed"])
    return dict(loss=loss, params=net.params()[0], Y=net.forward(s["Xv"]))


# ---------------------------------------------------------- what it must cost

def _step_values(les):
    """(bulk, FP64) values a cell of one RK3 step must move: per substep the
    eddy viscosity reads U, V, W and writes one field (a plane mean separates
    it from its use), the RHS reads four fields and writes three (and F1 or
    Uo and F1), the divergence reads three, the half-size spectra cross
    memory between the x, z and y solves (1 + 2 + 2 + 2 + 1 + 1), the
    projection reads p and reads and writes U, V, W."""
    eddy = 4 * 3 + (2 if les == "dsm" else 0)
    return eddy + (10 + 13 + 13) + 3 * 3 + 6 * 3, 3 * (1 + 2 + 2 + 2 + 2 + 1)


def work(case):
    c = dict(case)
    if c["kind"] == "train":
        n, nv = c["samples"], max(1024, c["samples"] // 8)
        mac = 4 * 64 + 2 * 64 * 64 + 64 * 2
        return {"bytes": 24.0 * (n + nv), "flops": 2.0 * mac * (3 * n + nv)}
    bulk = 8 if c["precision"] == "fp64" else 4
    if c["kind"] == "ensemble":
        cells = sum((a - 2) * (b - 1) * (d - 2) for a, b, d in _grids(c["members"]))
        les = "dsm"
    else:
        cells, les = (c["nx"] - 2) * (c["ny"] - 1) * (c["nz"] - 2), c["les"]
    b, p = _step_values(les)
    flops = (3 * 519 if les == "dsm" else 3 * 200) + 3 * 330 + 3 * 200 + 60
    out = (5 if c["kind"] == "coupled" else 3) * cells * 8
    return {"bytes": float(cells * (b * bulk + p * 8) * c["steps"] + out), "flops": float(cells * flops * c["steps"])}


# ------------------------------------------------------------- in 64 bits

_M64 = (1 << 64) - 1


def _shuffled(n, seed):
    """Fisher-Yates with splitmix64, the order the training visits its samples in."""
    perm, st = list(range(n)), seed
    for q in range(n - 1, 0, -1):
        st = (st + 0x9E3779B97F4A7C15) & _M64
        z = ((st ^ (st >> 30)) * 0xBF58476D1CE4E5B9) & _M64
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _M64
        r = (z ^ (z >> 31)) % (q + 1)
        perm[q], perm[r] = perm[r], perm[q]
    return np.array(perm)


def exact(case, seed):
    """The trained network in 64-bit arithmetic throughout (no rounding of
    weights or activations); a run's fields are the end of a chain of whole
    time steps, for which there is no value here."""
    c = dict(case)
    if c["kind"] != "train":
        return None
    n, batch = c["samples"], c["batch"]
    X, Y, Xv, p0, norm = _training_set(np.random.default_rng(seed), n)
    norm = norm.astype(np.float64)
    x, t, xv = ((a.astype(np.float64) - m) / s for a, m, s in
                ((X, norm[:4], norm[4:8]), (Y, norm[8:10], norm[10:12]), (Xv, norm[:4], norm[4:8])))
    shapes = ((4, 64), (64,), (64, 64), (64,), (64, 64), (64,), (64, 2), (2,))
    at = np.cumsum([0] + [int(np.prod(q)) for q in shapes])
    p = p0.astype(np.float64)

    def forward(p, x):
        w = [p[at[q]:at[q + 1]].reshape(shapes[q]) for q in range(8)]
        h, z = [x], []
        for q in range(3):
            z.append(h[-1] @ w[2 * q] + w[2 * q + 1])
            h.append(_silu(z[-1]))
        return w, h, z, h[-1] @ w[6] + w[7]

    m, v, lr, b1, b2 = np.zeros_like(p), np.zeros_like(p), 1e-3, 0.9, 0.999
    order, loss = _shuffled(n, int(seed) & 0xFFFF), 0.0
    for k, a in enumerate(range(0, n, batch)):
        idx = order[a:a + batch]
        w, h, z, y = forward(p, x[idx])
        e = y - t[idx]
        loss += 0.5 * float(np.sum(e * e))
        d, g = e / len(idx), [None] * 8
        for q in (3, 2, 1, 0):
            g[2 * q], g[2 * q + 1] = h[q].T @ d, d.sum(axis=0)
            if q:
                s = 1.0 / (1.0 + np.exp(-z[q - 1]))
                d = (d @ w[2 * q].T) * (s * (1.0 + z[q - 1] * (1.0 - s)))
        g = np.concatenate([q.ravel() for q in g])
        m, v = b1 * m + (1 - b1) * g, b2 * v + (1 - b2) * g * g
        p = p - lr * (m / (1 - b1 ** (k + 1))) / (np.sqrt(v / (1 - b2 ** (k + 1))) + 1e-8)
    return dict(loss=np.array([loss / n]), params=p, Y=forward(p, xv)[3] * norm[10:12] + norm[8:10])
