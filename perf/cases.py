"""Performance cases of the fibre library: what its users have it compute, from
one short fibre to thousands of uneven ones, through the public entry points.

Every case is one of two kinds:

  advance   a ``FiberBatch`` of Hodgkin-Huxley fibres takes ``steps`` Strang
            split steps and its states (and spike data) are read back; the
            simulated time goes on from pass to pass, as in a running program
  gradient  the gradient of a Vm-trace misfit with respect to per-fibre
            (g_Na, g_K, g_L, sigma): ``MonodomainTraces`` forward, backward

``exact`` computes the same results in FP64 with plain torch: the same
discrete scheme (Heun halves, one tridiagonal solve, the clamp and pulse rules),
accurate exponentials, parallel cyclic reduction for the solve, and reverse mode
by torch.autograd one split step at a time.
"""
from __future__ import annotations

import math

import numpy as np
import torch

AM, CM = 500.0, 1.0
V_STIM = 20.0
N_STATES = 4
GNA, GK, GL = 120.0, 36.0, 0.3
RESTING = (-75.0, 0.05, 0.6, 0.325)
# + - * / exp of one right-hand side of the model, and of the diffusion per node
OPS_RHS, OPS_SOLVE = 61.0, 64.0
MOST_NODE_HEUN_STEPS = 5.2e9   # work of the largest listed case (Heun steps times nodes)


def _advance(name, **kw):
    case = dict(kind="advance", fibers=1, lo=1001, hi=1001, steps=256, n0D=1, dt=1e-3, scheme="CN",
                precision="fp64", exp="approx", thomas="partitioned", schedule="auto", stimulation="pulse",
                only_if_stimulated=False, spikes=False)
    case.update(kw)
    return dict(name=name, **case) if name else case


def _gradient(name, **kw):
    case = dict(kind="gradient", fibers=256, lo=1000, hi=1000, steps=500, dt=1e-3, scheme="CN", sensors=32,
                tape="auto", interval=100)
    case.update(kw)
    return dict(name=name, **case) if name else case


def listed():
    return [
        # the smallest call: the single short fibre of the settings example, ten Heun steps per
        # split step (five per half), firing table; launches and latency
        _advance("one_fibre_101", lo=101, hi=101, steps=50, n0D=5, dt=2e-3, scheme="IE", stimulation="table"),
        # one 10 cm fibre, the propagating action potential every installation is checked with
        _advance("one_fibre_1001", steps=1000, spikes=True),
        # FiberBatch as it is constructed by default (split kernels, untuned), a few short fibres
        _advance("default_split_16", fibers=16, lo=200, hi=600, steps=100, dt=2e-3, scheme="IE", schedule="split",
                 stimulation="table"),
        # a 7 x 7 bundle of long fibres as the reference's bundles run it: implicit Euler, motor
        # units, onlyComputeIfHasBeenStimulated
        _advance("bundle_49", fibers=49, lo=1481, hi=1481, steps=400, dt=2e-3, scheme="IE", stimulation="table",
                 only_if_stimulated=True),
        # a medium batch with equal fibres, the device's exp
        _advance("batch_512_libm", fibers=512, lo=1001, hi=1001, steps=300, scheme="IE", exp="libm"),
        # the batched workload of the benchmark: 4096 uneven fibres with spike detection
        _advance("batch_4096", fibers=4096, lo=400, hi=2000, steps=1000, spikes=True),
        # the same with FP32 gate storage
        _advance("batch_4096_mixed", fibers=4096, lo=400, hi=2000, steps=600, precision="mixed"),
        # the longest fibres the partitioned solve takes
        _advance("long_fibres_200", fibers=200, lo=2049, hi=4096, steps=300, dt=2e-3, scheme="IE",
                 stimulation="table"),
        # the bit-exact serial solve, many short fibres
        _advance("serial_1024", fibers=1024, lo=101, hi=301, steps=200, scheme="IE", thomas="serial",
                 stimulation="table"),
        # untuned split kernels on a large batch
        _advance("default_split_1024", fibers=1024, lo=301, hi=1481, steps=200, schedule="split", spikes=True),
        # parameter estimation: gradient through the whole tape in HBM
        _gradient("gradient_256"),
        # the same through checkpoints, uneven fibres, implicit Euler
        _gradient("gradient_checkpoints_64", fibers=64, lo=301, hi=1481, steps=400, scheme="IE", tape="segments"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.2:
        hi = rng.randint(60, 1600)
        case = _gradient(None, fibers=_log_int(rng, 4, 300), lo=max(40, hi - rng.randint(0, 500)), hi=hi,
                         steps=rng.randint(60, 500), scheme=rng.choice(["CN", "IE"]), sensors=rng.randint(4, 32),
                         tape=rng.choice(["auto", "segments"]), interval=rng.randint(30, 120))
        return case
    serial = rng.random() < 0.15
    hi = _log_int(rng, 90, 1000) if serial else _log_int(rng, 90, 4096)
    fibers = _log_int(rng, 1, 4096)
    n0D = rng.choice([1, 1, 1, 2, 5])
    steps = _log_int(rng, 40, 200) if serial else _log_int(rng, 40, 800)
    steps = max(20, min(steps, int(0.5 * MOST_NODE_HEUN_STEPS / (2.0 * n0D * fibers * hi))))
    precision = "mixed" if rng.random() < 0.25 and not serial else "fp64"
    stimulation = rng.choice(["pulse", "table"])
    return _advance(None, fibers=fibers, lo=max(64, int(hi * rng.uniform(0.2, 1.0))), hi=max(64, hi), steps=steps,
                    n0D=n0D, dt=rng.choice([1e-3, 2e-3]), scheme=rng.choice(["CN", "IE"]), precision=precision,
                    exp=rng.choice(["approx", "approx", "approx", "libm"]),
                    thomas="serial" if serial else "partitioned", schedule=rng.choice(["auto", "auto", "split"]),
                    stimulation=stimulation, only_if_stimulated=stimulation == "table" and rng.random() < 0.3,
                    spikes=precision == "fp64" and rng.random() < 0.5)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _inputs(case, seed):
    """meshes, conductivities and stimulation of a case, from the seed alone"""
    rng = np.random.default_rng([seed, 17])
    F = case["fibers"]
    # the meshes' sizes belong to the case
    n = np.random.default_rng([F, case["lo"], case["hi"]]).integers(case["lo"], case["hi"] + 1, size=F).astype(np.int32)
    # node positions with a little scatter, as an unstructured 3D mesh gives them
    h = 0.01 * (1.0 + 0.02 * rng.uniform(-1.0, 1.0, int(n.sum()) - F))
    pf = rng.uniform(3.0, 4.5, F) / (AM * CM)
    nmj = (n * rng.uniform(0.35, 0.65, F)).astype(np.int32)
    t_pass = case["steps"] * case["dt"]
    d = dict(n=n, h=h, pf=pf, nmj=nmj, sb=np.maximum(nmj - 1, 0).astype(np.int32),
             se=np.minimum(nmj + 2, n).astype(np.int32))
    if case["kind"] == "gradient" or case["stimulation"] == "pulse":
        d.update(onset=rng.uniform(0.0, min(2.0, 0.5 * t_pass), F), duration=np.full(F, 0.1),
                 amplitude=np.full(F, 1200.0))
    else:
        n_mu = 10
        # one row per 0.1 ms; each motor unit fires at 2 percent of the rows, and once early
        table = (rng.random((400, n_mu)) < 0.02).astype(np.uint8)
        table[rng.integers(0, 2, n_mu), np.arange(n_mu)] = 1
        d.update(table=table, mu=rng.integers(1, n_mu + 1, F).astype(np.int32), freq=np.full(F, 10.0),
                 repeat=np.zeros(F), begin=np.zeros(F))
    if case["kind"] == "gradient":
        theta = np.stack([rng.uniform(100, 140, F), rng.uniform(30, 42, F), rng.uniform(0.2, 0.4, F), pf * AM * CM], 1)
        d.update(theta_true=theta, theta0=theta * rng.uniform(0.95, 1.05, theta.shape),
                 sensors=np.stack([np.round(np.linspace(0, k - 1, case["sensors"])).astype(np.int32) for k in n]))
    return d


def _rows(t0, dt, steps, n0D=1):
    return np.stack([t0 + np.arange(steps) * dt, np.full(steps, dt), np.full(steps, dt / 2 / n0D),
                     np.full(steps, dt)], 1)


def prepare(case, seed):
    from opendihu_amd.fibers import FiberBatch
    d = _inputs(case, seed)
    gradient = case["kind"] == "gradient"
    auto = gradient or case["schedule"] == "auto"
    batch = FiberBatch(n_nodes=d["n"], element_lengths=d["h"], prefactor=d["pf"], scheme=case["scheme"],
                       precision=case.get("precision", "fp64"), exp_mode=case.get("exp", "approx"),
                       thomas=case.get("thomas", "partitioned"), kernels="fused" if auto else "split",
                       value_for_stimulated_point=V_STIM)
    if "onset" in d:
        batch.set_current_stimulation(d["sb"], d["se"], d["onset"], d["duration"], d["amplitude"])
    else:
        batch.set_firing_table_stimulation(d["sb"], d["se"], d["table"], d["mu"], d["freq"], d["repeat"], d["begin"],
                                           log_capacity=1 << 16)
    if gradient:
        from opendihu_amd.adjoint import AdjointProblem
        problem = AdjointProblem(batch, _rows(0.0, case["dt"], case["steps"]), d["sensors"],
                                 checkpoint_interval=case["interval"], am=AM, cm=CM, tape=case["tape"])
        target = problem.forward_tensor(torch.tensor(d["theta_true"], device="cuda"))
        theta = torch.tensor(d["theta0"], device="cuda", requires_grad=True)
        return dict(case=case, batch=batch, problem=problem, theta=theta, target=target)
    if case["only_if_stimulated"]:
        batch.set_only_compute_if_stimulated(True)
    if case["spikes"]:
        batch.enable_spike_detection(0.0)
    if auto:
        # as the settings front end does at initialisation
        batch.autotune(_rows(0.0, case["dt"], min(64, case["steps"]), case["n0D"]), n0D=case["n0D"])
    return dict(case=case, batch=batch, t=0.0)


def run(state):
    case, batch = state["case"], state["batch"]
    if case["kind"] == "gradient":
        from opendihu_amd.adjoint import MonodomainTraces
        traces = MonodomainTraces.apply(state["theta"], state["problem"])
        loss = 0.5 * ((traces - state["target"]) ** 2).sum()
        grad, = torch.autograd.grad(loss, state["theta"])
        return dict(traces=traces.detach(), grad=grad)
    batch.advance(state["t"], case["dt"], case["steps"], dt0D=case["dt"] / 2 / case["n0D"], n0D=case["n0D"])
    state["t"] += case["steps"] * case["dt"]
    out = dict(states=[batch.get_state(k) for k in range(N_STATES)])
    if case["spikes"]:
        out["spikes"] = list(batch.spikes())
    return out


def _nodes(case):
    return case["fibers"] * 0.5 * (case["lo"] + case["hi"])


def work(case):
    N, K = _nodes(case), case["steps"]
    step = 2.0 * case.get("n0D", 1) * (2 * OPS_RHS + 5 * N_STATES) + OPS_SOLVE
    if case["kind"] == "gradient":
        # the traces written and their adjoints read; each reverse step about twice a forward one
        return dict(bytes=N * 8.0 * N_STATES + 2 * 8.0 * K * case["fibers"] * case["sensors"], flops=3.0 * N * K * step)
    # every state read once and written once, the element lengths read once
    gate = 4.0 if case["precision"] == "mixed" else 8.0
    extra = 2 * 8.0 + 2 * 4.0 if case["spikes"] else 0.0
    return dict(bytes=N * (2 * 8.0 + 2 * gate * (N_STATES - 1) + 8.0 + extra), flops=N * K * step)


# ---------------------------------------------------------------------------
# the same results in FP64 with plain torch
# ---------------------------------------------------------------------------
def _exp(x, approx):
    return torch.exp(1024.0 * torch.log1p(x / 1024.0)) if approx else torch.exp(x)


def _vtrap(x, approx):
    """x / (E(x) - 1)"""
    em1 = torch.expm1(1024.0 * torch.log1p(x / 1024.0)) if approx else torch.expm1(x)
    return torch.where(x == 0.0, torch.ones_like(x), x / torch.where(em1 == 0.0, torch.ones_like(x), em1))


def _rates(y, p, approx):
    V, m, h, n = y
    i_stim, gna, gk, gl = p
    am, bm = _vtrap(-(V + 50.0) / 10.0, approx), 4.0 * _exp(-(V + 75.0) / 18.0, approx)
    ah, bh = 0.07 * _exp(-(V + 75.0) / 20.0, approx), 1.0 / (_exp(-(V + 45.0) / 10.0, approx) + 1.0)
    an, bn = 0.1 * _vtrap(-(V + 65.0) / 10.0, approx), 0.125 * _exp((V + 75.0) / 80.0, approx)
    m3, n2 = m * m * m, n * n
    return (i_stim - gna * m3 * h * (V - 40.0) - gk * n2 * n2 * (V + 87.0) - gl * (V + 64.387),
            am * (1.0 - m) - bm * m, ah * (1.0 - h) - bh * h, an * (1.0 - n) - bn * n)


def _heun(y, p, dt, approx, clamp=None):
    r = _rates(y, p, approx)
    ys = [a + dt * b for a, b in zip(y, r)]
    if clamp is not None:
        ys[0] = torch.where(clamp, torch.full_like(ys[0], V_STIM), ys[0])
    rs = _rates(ys, p, approx)
    out = [a + 0.5 * dt * (b + c) for a, b, c in zip(y, r, rs)]
    if clamp is not None:
        out[0] = torch.where(clamp, torch.full_like(out[0], V_STIM), out[0])
    return out


class _Diffusion:
    """A x = B u of every fibre (rows padded to the longest fibre with identity
    rows), by parallel cyclic reduction with the coefficients of one dt"""

    def __init__(self, d, dt, implicit, device):
        n, F = d["n"], d["n"].size
        nmax = int(n.max())
        off = np.concatenate([[0], np.cumsum(n - 1)])
        h = np.ones((F, nmax))
        has = np.zeros((F, nmax), bool)
        for f in range(F):
            h[f, :n[f] - 1] = d["h"][off[f]:off[f + 1]]
            has[f, :n[f] - 1] = True
        h, has = torch.tensor(h, device=device), torch.tensor(has, device=device)
        pad = torch.arange(nmax, device=device)[None] >= torch.tensor(n.astype(np.int64), device=device)[:, None]
        self.dt, self.implicit, self.h, self.has, self.pad = dt, implicit, h, has, pad
        self.factor(torch.tensor(d["pf"], device=device))

    @staticmethod
    def _left(x):
        return torch.nn.functional.pad(x[:, :-1], (1, 0))

    def _shift(self, x, s):
        s0 = min(abs(s), x.shape[1])
        return torch.nn.functional.pad(x[:, :x.shape[1] - s0], (s0, 0)) if s > 0 else \
            torch.nn.functional.pad(x[:, s0:], (0, s0))

    def factor(self, pf):
        zero = torch.zeros_like(self.h)
        self.k = torch.where(self.has, pf[:, None] / self.h, zero)
        self.m = torch.where(self.has, self.h / (6.0 * self.dt), zero)
        th = 1.0 if self.implicit else 0.5
        self.off_b = -(1.0 - th) * self.k - self.m
        diag = (1.0 - th) * self.k - 2.0 * self.m
        self.diag_b = diag + self._left(diag)
        c = th * self.k - self.m
        diag = -th * self.k - 2.0 * self.m
        b = torch.where(self.pad, torch.ones_like(c), diag + self._left(diag))
        a = self._left(c)
        self.levels, s = [], 1
        while s < c.shape[1]:
            # rows past either end: unit diagonal, no coupling
            bm, bp = self._shift(b - 1.0, s) + 1.0, self._shift(b - 1.0, -s) + 1.0
            al, ga = -a / bm, -c / bp
            b = b + al * self._shift(c, s) + ga * self._shift(a, -s)
            a, c = al * self._shift(a, s), ga * self._shift(c, -s)
            self.levels.append((s, al, ga))
            s *= 2
            if float(torch.maximum((a / b).abs().max(), (c / b).abs().max())) < 1e-40:
                break
        self.b = b

    def b_times(self, u):
        cu = self.off_b * u
        return self._left(cu) + self.diag_b * u + self.off_b * torch.nn.functional.pad(u[:, 1:], (0, 1))

    def solve(self, r):
        for s, al, ga in self.levels:
            r = r + al * self._shift(r, s) + ga * self._shift(r, -s)
        return r / self.b

    def k1(self, u):
        """the stiffness matrix of prefactor 1"""
        fl = torch.where(self.has, (torch.nn.functional.pad(u[:, 1:], (0, 1)) - u) / self.h, torch.zeros_like(u))
        return fl - self._left(fl)

    def step(self, u):
        return torch.where(self.pad, u, self.solve(self.b_times(u)))


def _stimulus(case, d, device):
    """function (t) -> (stimulated fibres, computing fibres) of one Heun step, in time order"""
    F = d["n"].size
    has_been = np.zeros(F, bool)
    only = case.get("only_if_stimulated", False)
    if "onset" in d:
        def flags(t):
            on = (t >= d["onset"] - 1e-13) & (t < d["onset"] + d["duration"] - 1e-13)
            return torch.tensor(on, device=device), None
        return flags
    last = d["begin"] - 1e-13 - 1.0 / d["freq"]
    col = d["mu"] % d["table"].shape[1]

    def flags(t):
        check = (t >= last + 1.0 / d["freq"]) & (t >= d["begin"] - 1e-13)   # no repeat window, no jitter
        row = np.floor(np.abs(t * d["freq"]) + 0.5).astype(np.int64) % d["table"].shape[0]
        on = check & (d["table"][row, col] != 0)
        np.logical_or(has_been, on, out=has_been)
        return torch.tensor(on, device=device), (torch.tensor(has_been.copy(), device=device) if only else None)
    return flags


def _exact_advance(case, d, device):
    n, F = d["n"], d["n"].size
    nmax = int(n.max())
    approx = case["exp"] == "approx"
    diff = _Diffusion(d, case["dt"], case["scheme"] == "IE", device)
    y = [torch.full((F, nmax), v, dtype=torch.float64, device=device) for v in RESTING]
    i = torch.arange(nmax, device=device)[None]
    inset = (i >= torch.tensor(d["sb"], device=device)[:, None]) & (i < torch.tensor(d["se"], device=device)[:, None])
    pulse = "onset" in d
    flags = _stimulus(case, d, device)
    dt0 = case["dt"] / 2 / case["n0D"]

    def half(y, t):
        for j in range(case["n0D"]):
            on, compute = flags(t + j * dt0)
            hit = inset & on[:, None]
            i_stim = hit * float(d["amplitude"][0]) if pulse else torch.zeros_like(y[0])
            new = _heun(y, (i_stim, GNA, GK, GL), dt0, approx, None if pulse else hit)
            y = new if compute is None else [torch.where(compute[:, None], a, b) for a, b in zip(new, y)]
        return y

    for k in range(case["steps"]):
        t = k * case["dt"]
        y = half(y, t)
        y[0] = diff.step(y[0])
        y = half(y, t + 0.5 * case["dt"])
    keep = ~diff.pad
    out = dict(states=[v[keep] for v in y])
    if case["spikes"]:
        out["spikes"] = [None, None]
    return out


class _Solve(torch.autograd.Function):
    @staticmethod
    def forward(ctx, u, pf, diff):
        x = diff.step(u)
        ctx.diff = diff
        ctx.save_for_backward(u, x)
        return x

    @staticmethod
    def backward(ctx, g):
        diff, (u, x) = ctx.diff, ctx.saved_tensors
        w = torch.where(diff.pad, torch.zeros_like(g), diff.solve(torch.where(diff.pad, torch.zeros_like(g), g)))
        v = x if diff.implicit else 0.5 * (u + x)
        gpf = -(w * diff.k1(torch.where(diff.pad, torch.zeros_like(v), v))).sum(1)
        return diff.b_times(w), gpf, None


def _exact_gradient(case, d, device):
    n, F, K, dt = d["n"], d["n"].size, case["steps"], case["dt"]
    nmax = int(n.max())
    i = torch.arange(nmax, device=device)[None]
    inset = (i >= torch.tensor(d["sb"], device=device)[:, None]) & (i < torch.tensor(d["se"], device=device)[:, None])
    sensors = torch.tensor(d["sensors"].astype(np.int64), device=device)
    pad = i >= torch.tensor(n.astype(np.int64), device=device)[:, None]
    flags = _stimulus(case, d, device)
    on = [[flags(k * dt)[0], flags(k * dt + 0.5 * dt)[0]] for k in range(K)]
    amp = float(d["amplitude"][0])

    def step(k, y, theta, diff):
        y = list(y)
        for half in range(2):
            p = ((inset & on[k][half][:, None]) * amp, theta[:, 0:1], theta[:, 1:2], theta[:, 2:3])
            y = _heun(y, p, 0.5 * dt, True)
            if half == 0:
                y[0] = _Solve.apply(y[0], theta[:, 3] / (AM * CM), diff)
        return y

    def forward(theta, keep):
        diff = _Diffusion(dict(d, pf=theta[:, 3].cpu().numpy() / (AM * CM)), dt, case["scheme"] == "IE", device)
        y = [torch.full((F, nmax), v, dtype=torch.float64, device=device) for v in RESTING]
        tape, traces = [], torch.empty((K, F, sensors.shape[1]), dtype=torch.float64, device=device)
        with torch.no_grad():
            for k in range(K):
                if keep:
                    tape.append(y)
                y = step(k, y, theta, diff)
                traces[k] = torch.gather(y[0], 1, sensors)
        return traces, tape, diff

    target, _, _ = forward(torch.tensor(d["theta_true"], device=device), False)
    theta = torch.tensor(d["theta0"], device=device)
    traces, tape, diff = forward(theta, True)
    resid = traces - target
    lam = [torch.zeros((F, nmax), dtype=torch.float64, device=device) for _ in range(N_STATES)]
    grad = torch.zeros_like(theta)
    for k in range(K - 1, -1, -1):
        lam[0] = lam[0].scatter_add(1, sensors, resid[k])
        y = [v.detach().requires_grad_(True) for v in tape[k]]
        th = theta.detach().requires_grad_(True)
        got = torch.autograd.grad(step(k, y, th, diff), y + [th], lam)
        lam = [torch.where(pad, torch.zeros_like(v), v) for v in got[:N_STATES]]
        grad += got[N_STATES]
        tape[k] = None
    return dict(traces=traces, grad=grad)


def exact(case, seed):
    device = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    d = _inputs(case, seed)
    if case["kind"] == "gradient":
        return _exact_gradient(case, d, device)
    # about 400 elementwise passes per Heun step over the padded batch
    if case["fibers"] * case["hi"] * float(case["steps"]) * case["n0D"] > 1.2e10:
        return None
    return _exact_advance(case, d, device)
