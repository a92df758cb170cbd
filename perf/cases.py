"""Measured workloads of the batched integrator, through its public entry points.

Every case is one call a user's program makes, at sizes from a single condition to the large ensembles of the
benchmark:

* ``integrate`` (host arrays, the reference library's own call): a scalar caller and small ensembles, where latency,
  launches and copies count;
* ``integrate_device`` (states resident in device memory): the reaction step of an operator-splitting flow solver,
  one or a few global steps on many conditions, FP64 and mixed precision, with and without the learned Newton start,
  analytic and finite-difference Jacobians;
* ``integrate_device_hetero3``: several networks in one launch;
* ``mlp_train_host``: training the start network on logged samples.

Two kinds of chemistry states occur in use.  ``ignition``: random mixtures at t = 0, as an ignition study reads them
from its initial-condition file; the first global steps resolve a violent transient.  ``burning``: states some
microseconds into that transient, with a little mixing between neighbours, as a flow solver hands them over after its
transport step.
"""
import functools
import math

import numpy as np
import torch

import accelerint_amd as acc
from accelerint_amd import mechanism as M

RTOL, ATOL = 1e-6, 1e-10  # the library's defaults
DT_CHEM, DT_VDP = 1e-6, 1e-3  # global steps of the kinetics networks and of the van der Pol oscillator


def listed():
    return [
        # a scalar caller: one oscillator, ten global steps, host arrays
        {"name": "vdp_one", "path": "host", "n": 2, "num": 1, "steps": 10, "precision": "fp64"},
        # a large parameter study of the oscillator, states on the device
        {"name": "vdp_study", "path": "device", "n": 2, "num": 262144, "steps": 5, "precision": "fp64"},
        # a small ignition ensemble of a hydrogen-sized network from an initial-condition file
        {"name": "k14_few", "path": "host", "n": 14, "num": 100, "steps": 5, "precision": "fp64", "state": "ignition"},
        # the reaction step of a flow solver, hydrogen-sized network, default precision
        {"name": "k14_flow_fp64", "path": "device", "n": 14, "num": 262144, "steps": 2, "precision": "fp64", "state": "burning"},
        # the same with FP32 factors on a ragged sub-domain, from host arrays
        {"name": "k14_ragged_mixed", "path": "host", "n": 14, "num": 30011, "steps": 4, "precision": "mixed", "state": "burning"},
        # a handful of ignition cases of a hydrocarbon-sized network, host arrays, default precision
        {"name": "k54_few", "path": "host", "n": 54, "num": 33, "steps": 2, "precision": "fp64", "state": "ignition"},
        # the reaction step of a flow solver, hydrocarbon-sized network, default precision
        {"name": "k54_flow_fp64", "path": "device", "n": 54, "num": 32768, "steps": 1, "precision": "fp64", "state": "burning"},
        # the same with FP32 factors on twice the cells
        {"name": "k54_flow_mixed", "path": "device", "n": 54, "num": 65536, "steps": 1, "precision": "mixed", "state": "burning"},
        # FP32 factors with the learned Newton start, a ragged sub-domain over a few global steps
        {"name": "k54_learned", "path": "device", "n": 54, "num": 8191, "steps": 4, "precision": "mixed", "state": "burning", "learned": True},
        # callbacks without an analytic Jacobian: finite differences, an ordinary ensemble
        {"name": "k14_fd", "path": "device", "n": 14, "num": 8191, "steps": 2, "precision": "fp64", "state": "burning", "jacobian": "fd"},
        # zones of three chemistry sizes in one launch
        {"name": "zones", "path": "zones", "n": 112, "num": 24, "num54": 2049, "num14": 8190, "steps": 1, "precision": "fp64", "state": "burning"},
        # training the start network on logged samples, forward and backward passes
        {"name": "start_training", "path": "train", "n": 54, "num": 32768, "steps": 2, "batch": 512},
    ]


def _log_int(rng, lo, hi):
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, min(hi, v + rng.randrange(2)))


def draw(rng):
    kind = rng.choice(["vdp", "k14", "k14", "k54", "k54", "k54", "fd", "zones", "train"])
    if kind == "vdp":
        path = rng.choice(["host", "device"])
        return {"path": path, "n": 2, "num": _log_int(rng, 1, 200000), "steps": rng.randint(1, 10), "precision": rng.choice(["fp64", "fp64", "mixed"])}
    if kind == "k14":
        state = rng.choice(["ignition", "burning", "burning"])
        path = rng.choice(["host", "device"])
        num = _log_int(rng, 1, 20000 if state == "ignition" else 200000)
        return {"path": path, "n": 14, "num": num, "steps": rng.randint(1, 3), "precision": rng.choice(["fp64", "mixed"]), "state": state}
    if kind == "k54":
        state = rng.choice(["ignition", "burning", "burning"])
        path = rng.choice(["host", "device"])
        steps = rng.randint(1, 3)
        num = _log_int(rng, 1, 1000 if state == "ignition" else 30000 // steps)
        c = {"path": path, "n": 54, "num": num, "steps": steps, "precision": rng.choice(["fp64", "mixed"]), "state": state}
        if c["precision"] == "mixed" and rng.random() < 0.3:
            c["learned"] = True
        return c
    if kind == "fd":
        return {"path": "device", "n": 14, "num": _log_int(rng, 1, 20000), "steps": rng.randint(1, 2), "precision": rng.choice(["fp64", "mixed"]), "state": "burning", "jacobian": "fd"}
    if kind == "zones":
        # FP32 factors without the largest network: a single one of its conditions can need thousands of small steps
        large = rng.random() < 0.5
        num = _log_int(rng, 1, 24) if large else 0
        return {"path": "zones", "n": 112, "num": num, "num54": _log_int(rng, 1, 2000), "num14": _log_int(rng, 1, 16000), "steps": 1, "precision": "fp64" if large else "mixed", "state": "burning"}
    n = rng.choice([14, 54])
    batch = rng.choice([64, 128, 256, 512])
    return {"path": "train", "n": n, "num": batch * _log_int(rng, 8, 50) + rng.randrange(batch), "steps": rng.randint(1, 2), "batch": batch}


# ---- inputs -------------------------------------------------------------------------------------------------------

DEV = "cuda"


@functools.lru_cache(maxsize=None)
def _stream():
    """The program's one stream: the library's queues and work buffers belong to the process, so calls follow each other."""
    return torch.cuda.Stream()


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


@functools.lru_cache(maxsize=None)
def _net(n):
    """The network and its tables as tensors: slot species (absent ones point at a column of ones), nu, rates."""
    m = M.network(n)
    t = functools.partial(torch.tensor, dtype=torch.float64, device=DEV)
    sp = torch.tensor(np.where(m.slots < 0, m.ns, m.slots), dtype=torch.int64, device=DEV)
    sign = np.array([-1, -1, -1, 1, 1, 1.0])
    nu = np.zeros((m.nr, m.ns + 1))
    for a in range(6):
        np.add.at(nu, (np.arange(m.nr), np.where(m.slots[:, a] < 0, m.ns, m.slots[:, a])), sign[a] * (m.slots[:, a] >= 0))
    return m, {"sp": sp, "nu": t(nu[:, :m.ns]), "W": t(m.W), "th": t(m.thermo), "lnA": t(m.lnA), "beta": t(m.beta), "EaR": t(m.EaR)}


def _thermo(k, T):
    """cp/R, h/R and s/R (pressure-free) of every species at temperatures T (..., 1)."""
    a0, a1, a2, bh, bs = k["th"].T
    cp = a0 + a1 * T + a2 * T * T
    h = a0 * T + a1 * T * T / 2 + a2 * T ** 3 / 3 + bh
    s = a0 * torch.log(T) + a1 * T + a2 * T * T / 2 + bs
    return cp, h, s


def _rates(k, T, P, x):
    """Forward and reverse rate constants, the slots' concentrations and the density (mol/cm3 per mol/kg)."""
    T = T[..., None]
    cp, h, s = _thermo(k, T)
    lnkc = -((h / T - s) @ k["nu"].T) + k["nu"].sum(1) * torch.log(1e-6 * M.P_ATM / (M.R_GAS * T))
    lnkf = k["lnA"] + k["beta"] * torch.log(T / 1000.0) - k["EaR"] / T
    rho = (1e-6 * P / (M.R_GAS * T[..., 0]) / x.sum(-1))[..., None]
    c = torch.cat([rho * x, torch.ones_like(rho)], -1)[..., k["sp"]]
    return torch.exp(lnkf), torch.exp(lnkf - lnkc), c, rho, cp, h


def _relax(n, T, P, x, t_end):
    """Mixtures after about t_end: linearly implicit Euler on growing steps, enthalpy kept."""
    _, k = _net(n)
    ar = torch.arange(k["nu"].shape[0], device=DEV)
    eye = torch.eye(n - 1, dtype=torch.float64, device=DEV)
    H = (x * _thermo(k, T[:, None])[1]).sum(1)
    mass = (x * k["W"]).sum(1)
    h, t = 1e-13, 0.0
    while t < t_end:
        kf, kr, c, rho, _, _ = _rates(k, T, P, x)
        d = torch.zeros(x.shape[0], k["nu"].shape[0], n, dtype=torch.float64, device=DEV)
        for b in range(6):
            lo = 3 * (b // 3)
            o = [a for a in range(lo, lo + 3) if a != b]
            part = (kf if lo == 0 else -kr) * c[:, :, o[0]] * c[:, :, o[1]]
            d[:, ar, k["sp"][:, b]] = d[:, ar, k["sp"][:, b]] + part
        q = kf * c[..., 0] * c[..., 1] * c[..., 2] - kr * c[..., 3] * c[..., 4] * c[..., 5]
        f = (q @ k["nu"]) / rho
        J = torch.matmul(k["nu"].T.contiguous(), d[:, :, :n - 1].contiguous())
        x = (x + torch.linalg.solve(eye - h * J, h * f)).clamp(min=0.0)
        x = x * (mass / (x * k["W"]).sum(1))[:, None]
        for _ in range(4):
            cp, hh, _ = _thermo(k, T[:, None])
            T = (T - ((x * hh).sum(1) - H) / (x * cp).sum(1)).clamp(300.0, 5000.0)
        t += h
        h *= 1.4
    return T, x


def _chemistry(n, num, state, seed):
    """States y (num, n) and pressures (num,) on the device, condition-major."""
    m, k = _net(n)
    if state == "ignition":
        y, P = M.initial_conditions(m, num, seed)
        return torch.from_numpy(np.ascontiguousarray(y.T)).to(DEV), torch.from_numpy(P).to(DEV)
    g = _gen(seed)
    rand = lambda *s: torch.rand(*s, generator=g, device=DEV, dtype=torch.float64)  # noqa: E731
    pool = 64 if n == 112 else 256
    T = 1000.0 + 600.0 * rand(pool)
    P = (1.0 + 24.0 * rand(pool)) * M.P_ATM
    Y = torch.randn(pool, n - 1, generator=g, device=DEV, dtype=torch.float64) ** 2  # Dirichlet(1/2)
    T, x = _relax(n, T, P, Y / Y.sum(1, keepdim=True) / k["W"], 1e-5)
    a = torch.randint(pool, (num,), generator=g, device=DEV)
    b = torch.randint(pool, (num,), generator=g, device=DEV)
    mix = 1e-3 * rand(num)
    Y = x * k["W"]
    Y = (1 - mix)[:, None] * Y[a] + mix[:, None] * Y[b]
    T = ((1 - mix) * T[a] + mix * T[b]) * (1.0 + 1e-3 * (rand(num) - 0.5))
    P = P[a] * (1.0 + 1e-3 * (rand(num) - 0.5))
    return torch.cat([T[:, None], Y / Y.sum(1, keepdim=True)], 1).contiguous(), P.contiguous()


def _oscillators(num, seed):
    y, mu = M.van_der_pol_conditions(num, seed)
    return torch.from_numpy(np.ascontiguousarray(y.T)).to(DEV), torch.from_numpy(mu).to(DEV)


def _inputs(case, seed):
    if case["n"] == 2:
        return _oscillators(case["num"], seed)
    return _chemistry(case["n"], case["num"], case["state"], seed)


def _network_params(n, seed):
    """Glorot-sized parameters of the start network in the library's order, its padding zero."""
    r = np.random.default_rng(seed)
    i, o = n + 2, 3 * n
    ip, op = -(-i // 16) * 16, -(-o // 16) * 16
    parts = []
    for rows, cols, rv, cv in ((ip, 128, i, 128), (128, 128, 128, 128), (128, op, 128, o)):
        w, b = np.zeros((rows, cols)), np.zeros(cols)
        w[:rv, :cv] = r.uniform(-1, 1, (rv, cv)) * math.sqrt(6.0 / (rv + cv))
        parts += [w.ravel(), b]
    return np.concatenate(parts).astype(np.float32)


# ---- the measured calls -------------------------------------------------------------------------------------------

def _configure(case):
    """The library set up for a case, as a program does once before its calls."""
    acc.set_learned_start(False)
    acc.cleanup()
    acc.set_abort_on_error(False)
    acc.set_const_time_step(False)
    acc.set_tolerances(ATOL, RTOL)
    n = case["n"]
    if n == 2:
        acc.select_mechanism(acc.MECH_VAN_DER_POL)
    else:
        for size in ((14, 54, 112) if case["path"] == "zones" else (n,)):
            acc.set_kinetics(_net(size)[0])
    acc.set_precision(acc.PRECISION_MIXED if case["precision"] == "mixed" else acc.PRECISION_FP64)
    acc.set_jacobian(acc.JACOBIAN_FINITE_DIFFERENCE if case.get("jacobian") == "fd" else acc.JACOBIAN_ANALYTIC)
    acc.initialize(max(case["num"], case.get("num54", 0), case.get("num14", 0)), 0)


def prepare(case, seed):
    if case["path"] == "train":
        # the samples a program has logged: normalized features, and stages that follow from them
        r = np.random.default_rng(seed)
        n = case["n"]
        x = np.clip(r.standard_normal((case["num"], n + 2)), -16, 16).astype(np.float32)
        a, b = r.standard_normal((n + 2, 24)) / math.sqrt(n + 2), r.standard_normal((24, 3 * n)) / math.sqrt(24)
        t = (np.tanh(x @ a) @ b + 0.1 * r.standard_normal((case["num"], 3 * n))).astype(np.float32)
        return {"case": case, "x": x, "t": t, "p": _network_params(n, 1)}
    _configure(case)
    s = {"case": case}
    dt = DT_VDP if case["n"] == 2 else DT_CHEM
    s["dt"], s["t_end"] = dt, case["steps"] * dt
    if case["path"] == "zones":
        s["parts"] = []
        for size, num in ((112, case["num"]), (54, case["num54"]), (14, case["num14"])):
            y0, pr = _chemistry(size, num, case["state"], seed)
            s["parts"].append((num, y0, torch.empty_like(y0), pr, torch.zeros(num, dtype=torch.int32, device=DEV)))
    else:
        y0, pr = _inputs(case, seed)
        if case["path"] == "host":
            s["y0"], s["pr"] = np.ascontiguousarray(y0.T.cpu().numpy()), pr.cpu().numpy()
        else:
            s["y0"], s["pr"], s["y"] = y0, pr, torch.empty_like(y0)
            s["codes"] = torch.zeros(case["num"], dtype=torch.int32, device=DEV)
    if case.get("learned"):
        n = case["n"]
        acc.mlp_init(n, 1)
        acc.mlp_set_params(_network_params(n, 1))
        mu, sd = np.full(n + 2, -10.0), np.full(n + 2, 8.0)
        mu[0], sd[0], mu[n], sd[n], mu[n + 1], sd[n + 1] = 0.7, 0.2, math.log(5e-7), 1.0, 13.8, 0.9
        zs = np.full(3 * n, 1e-4)
        zs[::n] = 0.5  # the temperature's stages
        acc.mlp_set_normalization(mu, sd, zs)
        acc.set_learned_start(True)
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    if case["path"] == "host":
        y = s["y0"].copy()
        acc.integrate(case["num"], 0.0, s["t_end"], s["dt"], y, s["pr"])
        return {"y": y, "codes": acc.get_status(case["num"])}
    if case["path"] == "train":
        acc.mlp_init(case["n"], 1)
        acc.mlp_set_params(s["p"])
        loss = acc.mlp_train_host(s["x"], s["t"], case["steps"], case["batch"], 1e-3, seed=3)
        return {"params": acc.mlp_params(), "loss": loss}
    st = _stream()
    with torch.cuda.stream(st):
        if case["path"] == "zones":
            args = []
            for num, y0, y, pr, codes in s["parts"]:
                y.copy_(y0)
                args += [num, y.data_ptr(), pr.data_ptr(), codes.data_ptr()]
            acc.integrate_device_hetero3(*args, 0.0, s["t_end"], s["dt"], st.cuda_stream)
            return {"y%d" % p[2].shape[1]: p[2] for p in s["parts"]} | {"codes%d" % p[2].shape[1]: p[4] for p in s["parts"]}
        s["y"].copy_(s["y0"])
        acc.integrate_device(case["num"], 0.0, s["t_end"], s["dt"], s["y"].data_ptr(), s["pr"].data_ptr(), s["codes"].data_ptr(), st.cuda_stream)
    return {"y": s["y"], "codes": s["codes"]}


# ---- what a pass cannot do without --------------------------------------------------------------------------------

#: typical events of one condition over one global step: LU pairs, Newton iterations, right-hand sides, Jacobians,
#: error estimates
EVENTS = {2: (5, 8, 29, 1, 5), 14: (4.5, 11, 38, 1.2, 6), 54: (21, 55, 185, 4, 24), 112: (21, 55, 185, 4, 24)}


def _step_flops(n, fd):
    lu, newton, f, jac, es = EVENTS[n]
    if n == 2:
        fr, fj = 8, 8
    else:
        ns, nr = M.NETWORKS[n][:2]
        fr = 34 * ns + 50 * nr
        fj = n * fr if fd else fr + 108 * nr + 6 * ns * ns
    return lu * (10.0 / 3.0 * n ** 3 + 2 * n * n) + newton * (10 * n * n + 66 * n) + f * fr + jac * fj + es * (2 * n * n + 48 * n)


def work(case):
    if case["path"] == "train":
        i, o = case["n"] + 2, 3 * case["n"]
        weights = i * 128 + 128 * 128 + 128 * o
        samples = case["num"] // case["batch"] * case["batch"] * case["steps"]
        return {"bytes": samples * (i + o) * 4 + 2 * 4 * weights, "flops": samples * 6 * weights}
    parts = [(case["n"], case["num"])]
    if case["path"] == "zones":
        parts += [(54, case["num54"]), (14, case["num14"])]
    fd = case.get("jacobian") == "fd"
    return {"bytes": sum(num * (16 * n + 12) for n, num in parts), "flops": sum(num * case["steps"] * _step_flops(n, fd) for n, num in parts)}


# ---- values in 64 bits --------------------------------------------------------------------------------------------

def exact(case, seed):
    """The oscillator's solution by small classical Runge-Kutta steps; every multiplier of the other systems' stiff
    transients would take far longer than 20 seconds to resolve that way, and a training run's batches are drawn by
    the library."""
    if case["n"] != 2:
        return None
    y, mu = _oscillators(case["num"], seed)
    a, b = y[:, 0].clone(), y[:, 1].clone()
    h = 5e-6
    rhs = lambda u, v: (v, mu * (1.0 - u * u) * v - u)  # noqa: E731
    for _ in range(case["steps"] * round(DT_VDP / h)):
        k1, l1 = rhs(a, b)
        k2, l2 = rhs(a + h / 2 * k1, b + h / 2 * l1)
        k3, l3 = rhs(a + h / 2 * k2, b + h / 2 * l2)
        k4, l4 = rhs(a + h * k3, b + h * l3)
        a = a + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
        b = b + h / 6 * (l1 + 2 * l2 + 2 * l3 + l4)
    out = torch.stack([a, b], 1)
    if case["path"] == "host":
        return {"y": np.ascontiguousarray(out.T.cpu().numpy()), "codes": None}
    return {"y": out, "codes": None}
