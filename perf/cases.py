"""The workloads that spinsim_amd's speed is measured on, as a user's program runs them.

Three kinds of call cover the package: one simulation through
``Simulator.evaluate`` (fields from a single pulse of a few steps to 1e7
steps of a noisy carrier, spin half and spin one, either frame, every
integration rule, results as numpy arrays or as device tensors), a sweep of
many simulations through ``BatchPlan`` or ``evaluate_batch`` (uneven lengths,
full or compact operators), and the training step of a set of control pulses
through ``ControlledSimulator`` (forward and backward).

A case is a dict of plain values.  ``prepare`` draws what the caller brings
(sweep parameters, initial states, noise, control amplitudes) from the seed;
``exact`` integrates the same inputs with plain torch operations in 64 bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch
import torch.utils.checkpoint

import spinsim_amd as ss

TAU = 2 * math.pi
SPINS = {"half": ss.SpinQuantumNumber.HALF, "one": ss.SpinQuantumNumber.ONE}
METHODS = {"magnus_cf4": ss.IntegrationMethod.MAGNUS_CF4,
           "midpoint": ss.IntegrationMethod.MIDPOINT_SAMPLE,
           "half_step": ss.IntegrationMethod.HALF_STEP}
EXPONENTIALS = {"default": None, "lie_trotter": ss.ExponentiationMethod.LIE_TROTTER,
                "lie_trotter_8": ss.ExponentiationMethod.LIE_TROTTER_8}


# ---- fields -----------------------------------------------------------------
# Each as the Python function a user writes, and as torch operations over many
# sample times for exact(): f(t, s) -> the field's entries, s[k] the k-th sweep
# parameter of each time's simulation.

def _larmor(time_sample, sweep_parameters, field_sample):
    field_sample[2] = sweep_parameters[0]


def _rabi(time_sample, sweep_parameters, field_sample):
    field_sample[0] = 2 * sweep_parameters[1] * math.cos(sweep_parameters[0] * time_sample)
    field_sample[2] = sweep_parameters[0] + sweep_parameters[2]


def _rabi_one(time_sample, sweep_parameters, field_sample):
    field_sample[0] = 2 * sweep_parameters[1] * math.cos(sweep_parameters[0] * time_sample)
    field_sample[2] = sweep_parameters[0] + sweep_parameters[2]
    field_sample[3] = sweep_parameters[3]


def _gaussian(time_sample, sweep_parameters, field_sample):
    d = time_sample - sweep_parameters[1]
    field_sample[0] = sweep_parameters[0] * math.exp(-d * d / (2 * sweep_parameters[2] ** 2))


def _tilted(time_sample, sweep_parameters, field_sample):
    field_sample[0] = sweep_parameters[0] * math.cos(sweep_parameters[3] * time_sample) + 3e4
    field_sample[1] = sweep_parameters[1] * math.sin(sweep_parameters[3] * time_sample)
    field_sample[2] = sweep_parameters[2] + 3e4 * math.sin(6e3 * time_sample)


def _tilted_eight(time_sample, sweep_parameters, field_sample):
    c = math.cos(sweep_parameters[3] * time_sample)
    s = math.sin(sweep_parameters[3] * time_sample)
    field_sample[0] = sweep_parameters[0] * c + 3e4
    field_sample[1] = sweep_parameters[1] * s
    field_sample[2] = sweep_parameters[2] + 3e4 * s
    field_sample[3] = 2e4 * c
    field_sample[4] = 5e4 * c
    field_sample[5] = 2e4
    field_sample[6] = 4e4 * s - 1e4
    field_sample[7] = 2.5e4 * c


def _noisy(noise):
    def get_field(time_sample, sweep_parameters, field_sample):
        z = 7e5
        for k in range(8):
            d = time_sample - sweep_parameters[8 + k]
            z += sweep_parameters[k] * math.exp(-d * d / (2 * sweep_parameters[16 + k] ** 2))
        field_sample[2] = 2 * math.pi * z + noise(time_sample)
        field_sample[0] = 2 * math.pi * 1e3 * math.cos(2 * math.pi * 7e5 * time_sample)
    return get_field


def _bias(time_sample, sweep_parameters, field_sample):
    field_sample[2] = 2 * math.pi * 1e5


FIELDS = {"larmor": _larmor, "rabi": _rabi, "rabi_one": _rabi_one, "gaussian": _gaussian,
          "tilted": _tilted, "tilted_eight": _tilted_eight}


def _torch_field(name):
    def zero(t):
        return torch.zeros_like(t)

    def larmor(t, s):
        return [zero(t), zero(t), zero(t) + s[0]]

    def rabi(t, s):
        return [2 * s[1] * torch.cos(s[0] * t), zero(t), zero(t) + (s[0] + s[2])]

    def rabi_one(t, s):
        return rabi(t, s) + [zero(t) + s[3]]

    def gaussian(t, s):
        return [s[0] * torch.exp(-(t - s[1]) ** 2 / (2 * s[2] ** 2)), zero(t), zero(t)]

    def tilted(t, s):
        return [s[0] * torch.cos(s[3] * t) + 3e4, s[1] * torch.sin(s[3] * t),
                s[2] + 3e4 * torch.sin(6e3 * t)]

    def tilted_eight(t, s):
        c, n = torch.cos(s[3] * t), torch.sin(s[3] * t)
        return [s[0] * c + 3e4, s[1] * n, s[2] + 3e4 * n, 2e4 * c, 5e4 * c, zero(t) + 2e4,
                4e4 * n - 1e4, 2.5e4 * c]
    return locals()[name]


# ---- cases --------------------------------------------------------------------
def _single(name, field, spin, rows, dt, dt_out, **options):
    c = {"kind": "single", "field": field, "spin": spin, "rows": rows, "dt": dt, "dt_out": dt_out,
         "method": "magnus_cf4", "exponential": "default", "frame": True, "precision": "fp64",
         "output": "torch", **options}
    return {"name": name, **c} if name else c


def _sweep(name, spin, sims, shortest, longest, dt, dt_out, **options):
    c = {"kind": "sweep", "spin": spin, "sims": sims, "shortest": shortest, "longest": longest,
         "dt": dt, "dt_out": dt_out, "precision": "fp64", "compact": False, "graph": True, **options}
    return {"name": name, **c} if name else c


def _pulses(name, spin, sims, rows, dt, dt_out, knots, **options):
    c = {"kind": "pulses", "spin": spin, "sims": sims, "rows": rows, "dt": dt, "dt_out": dt_out,
         "knots": knots, "axes": "xy", "order": 3, "precision": "fp64", "deterministic": False,
         **options}
    return {"name": name, **c} if name else c


def listed():
    return [
        # one shaped pulse of a few dozen outputs, results straight into numpy:
        # the interactive call, all launches and host work
        _single("pulse_few_outputs", "gaussian", "half", 40, 50e-9, 500e-9, output="numpy"),
        # free precession, short output steps: the state product weighs as much
        # as the integration
        _single("larmor_half", "larmor", "half", 200000, 100e-9, 500e-9),
        # the driven spin-one system with a quadratic shift: 1e6 steps
        _single("rabi_one", "rabi_one", "one", 100000, 100e-9, 1e-6),
        # the same drive for 20 ms with the results as numpy arrays, as the
        # reference returns them
        _single("rabi_one_numpy", "rabi_one", "one", 20011, 100e-9, 1e-6, output="numpy"),
        # the same drive in the float32-bulk mode
        _single("rabi_one_fp32_bulk", "rabi_one", "one", 100000, 100e-9, 1e-6,
                precision="fp32_bulk"),
        # a field that turns on every axis, laboratory frame, second-order
        # rule, Lie-Trotter exponentials; lengths that divide nothing
        _single("tilted_half_lab", "tilted", "half", 30011, 100e-9, 700e-9, method="half_step",
                exponential="lie_trotter", frame=False),
        # a noisy carrier: 1e7 short steps, eight transients and an
        # interpolated noise table in the callback
        _single("noisy_half", "noisy", "half", 100000, 10e-9, 1e-6),
        # a few dozen spin-one runs of uneven length, planned and run in one
        # call: the small sweep
        _sweep("sweep_one_few", "one", 45, 1000, 5000, 100e-9, 1e-6, graph=False),
        # the large ensemble, captured once and replayed: operators, states and
        # Bloch vectors of 1e8 output rows
        _sweep("ensemble_half", "half", 4096, 1000, 50000, 50e-9, 1e-6),
        # the same ensemble for states and Bloch vectors, float32-bulk
        _sweep("ensemble_half_fp32_bulk", "half", 4096, 1000, 50000, 50e-9, 1e-6,
               precision="fp32_bulk", compact=True),
        # a training step of 1024 spin-one transfer pulses
        _pulses("pulses_one", "one", 1024, 2000, 20e-9, 1e-6, 2000),
        # a small optimisation: linear controls on every axis, repeatable sums
        _pulses("pulses_half_few", "half", 24, 333, 50e-9, 500e-9, 97, axes="xyz", order=1,
                deterministic=True),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["single", "single", "single", "sweep", "sweep", "pulses"])
    fine = rng.choice([1, 3, 5, 7, 10, 12, 20, 33])
    dt = round(_log(rng, 10e-9, 100e-9), 10)
    if kind == "single":
        field, spin = rng.choice([("larmor", "half"), ("rabi", "half"), ("rabi_one", "one"),
                                  ("rabi_one", "one"), ("gaussian", "half"), ("gaussian", "one"),
                                  ("tilted", "half"), ("tilted", "one"), ("tilted_eight", "one"),
                                  ("noisy", "half")])
        # (a tilted or pulsed field has no carrier for the frame to follow)
        frame = True if field in ("rabi", "rabi_one", "noisy", "larmor") else rng.random() < 0.5
        rows = int(_log(rng, 30, 3e5))
        exponential = "lie_trotter_8" if field == "tilted_eight" else \
            rng.choice(["default", "default", "lie_trotter"])
        return _single("", field, spin, rows, dt, fine * dt, frame=frame, exponential=exponential,
                       method=rng.choice(["magnus_cf4", "magnus_cf4", "magnus_cf4", "midpoint",
                                          "half_step"]),
                       precision="fp32_bulk" if field in ("rabi", "rabi_one") and
                       rng.random() < 0.2 else "fp64",
                       output="numpy" if rows < 20000 and rng.random() < 0.5 else "torch")
    if kind == "sweep":
        spin = rng.choice(["half", "half", "one"])
        sims = int(_log(rng, 2, 2000))
        longest = int(min(_log(rng, 200, 50000), 4e7 / sims))
        precision = rng.choice(["fp64", "fp64", "fp64", "fp32_bulk"])
        return _sweep("", spin, sims, max(1, longest // rng.choice([1, 3, 50])), longest, dt,
                      fine * dt, compact=spin == "half" and rng.random() < 0.3,
                      precision=precision, graph=rng.random() < 0.5)
    spin = rng.choice(["half", "one"])
    sims = int(_log(rng, 2, 600))
    rows = int(min(_log(rng, 50, 4000), 1e6 / sims))
    order = rng.choice([1, 3, 3])
    return _pulses("", spin, sims, rows, min(dt, 40e-9), fine * min(dt, 40e-9),
                   max(8, rows * rng.randint(2, 8) // 8), order=order,
                   axes=rng.choice(["x", "xy", "xy", "xyz"]), deterministic=rng.random() < 0.3)


def work(case):
    """Least bytes (inputs once, outputs once) and float64 operations.

    Per exponential of a generator of norm well below one: the generator from
    the samples, the coefficients of I, G (and G^2) and one product onto the
    operator -- about 130 operations for spin half and 480 for spin one; two
    samples with their frame, about 60.  A training step propagates state and
    costate once more and forms the derivative of each exponential: about the
    same again.
    """
    d = 2 if case["spin"] == "half" else 3
    per_row = 8 + 16 * d * d + 16 * d + 24
    rows = case["rows"] if case["kind"] == "single" else int(_lengths(case).sum())
    fine = round(case["dt_out"] / case["dt"])
    per_step = {2: 130, 3: 480}[d] * (1 if case.get("method") == "midpoint" else 2) + 60
    if case["kind"] == "single":
        return {"bytes": rows * per_row, "flops": rows * fine * per_step}
    if case["kind"] == "sweep":
        if case["compact"]:
            per_row -= 32
        return {"bytes": rows * per_row, "flops": rows * fine * per_step}
    amplitudes = case["sims"] * len(case["axes"]) * case["knots"] * 8
    # operators and states are kept between the passes: written once, read once
    return {"bytes": 2 * amplitudes + 2 * rows * (16 * d * d + 16 * d),
            "flops": 2 * rows * fine * per_step}


def _lengths(case):
    """Output rows of each simulation."""
    if case["kind"] == "pulses":
        return np.full(case["sims"], case["rows"])
    u = np.random.default_rng(case["sims"]).uniform(size=case["sims"])
    return np.rint(case["shortest"] + u * (case["longest"] - case["shortest"])).astype(np.int64)


def _unit(rng, d, n=None):
    v = rng.normal(size=(n or 1, d)) + 1j * rng.normal(size=(n or 1, d))
    v /= np.linalg.norm(v, axis=1, keepdims=True)
    return v if n else v[0]


def _sweep_rows(rng, field, span, n=1):
    """Sweep parameters (n, P) in rad/s and s; span: the simulated time."""
    def uniform(lo, hi):
        return rng.uniform(lo, hi, n)

    if field == "larmor":
        return np.stack([TAU * uniform(500, 5000)], 1)
    if field in ("rabi", "rabi_one"):
        cols = [np.full(n, TAU * 7e5), TAU * uniform(500, 5000), TAU * rng.normal(0, 200, n)]
        return np.stack(cols + ([TAU * uniform(500, 2000)] if field == "rabi_one" else []), 1)
    if field == "gaussian":  # a pulse of area pi to 3 pi in the middle of the run
        width = span * uniform(0.08, 0.12)
        return np.stack([uniform(math.pi, 3 * math.pi) / (math.sqrt(TAU) * width),
                         np.full(n, span / 2), width], 1)
    if field in ("tilted", "tilted_eight"):
        return np.stack([TAU * uniform(1e4, 4e4), TAU * uniform(5e3, 2e4), TAU * uniform(1e4, 3e4),
                         TAU * uniform(1e4, 3e4)], 1)
    return np.concatenate([rng.uniform(1e3, 1e4, 8), rng.uniform(0, span, 8),
                           rng.uniform(5e-6, 50e-6, 8)])[None]


def _noise(rng, span):
    """1/f noise (2 pi 50 rad/s standard deviation) on a 1 us grid over span."""
    grid = np.arange(max(8, int(span / 1e-6) + 2)) * 1e-6
    spec = np.fft.rfft(rng.normal(size=grid.size))
    freq = np.fft.rfftfreq(grid.size, 1e-6)
    spec[0] = 0
    spec[1:] /= np.sqrt(freq[1:])
    noise = np.fft.irfft(spec, grid.size)
    return grid, noise * (TAU * 50 / noise.std())


def _inputs(case, seed):
    """Everything the caller brings, as host arrays."""
    rng = np.random.default_rng(seed)
    d = 2 if case["spin"] == "half" else 3
    if case["kind"] == "single":
        span = case["rows"] * case["dt_out"]
        return {"sweep": _sweep_rows(rng, case["field"], span)[0], "psi0": _unit(rng, d),
                "noise": _noise(rng, span) if case["field"] == "noisy" else None}
    if case["kind"] == "sweep":
        field = "rabi" if d == 2 else "rabi_one"
        return {"sweep": _sweep_rows(rng, field, 0.0, case["sims"]), "psi0": _unit(rng, d)}
    span = case["rows"] * case["dt_out"]
    return {"psi0": _unit(rng, d), "grid": np.linspace(0.0, span, case["knots"]),
            "amplitudes": rng.normal(0, TAU * 5e3, (case["sims"], len(case["axes"]),
                                                    case["knots"]))}


def _end(rows, dt_out):
    """An end time that gives exactly `rows` outputs."""
    return (rows + 0.5) * dt_out


# ---- the calls ------------------------------------------------------------------
def prepare(case, seed):
    given = _inputs(case, seed)
    spin = SPINS[case["spin"]]
    dt, dt_out = case["dt"], case["dt_out"]
    if case["kind"] == "single":
        if case["field"] == "noisy":
            field = _noisy(ss.generate_interpolation_sampler(*given["noise"]))
        else:
            field = FIELDS[case["field"]]
        sim = ss.Simulator(field, spin, exponentiation_method=EXPONENTIALS[case["exponential"]],
                           use_rotating_frame=case["frame"],
                           integration_method=METHODS[case["method"]],
                           precision=case["precision"])
        args = (0.0, _end(case["rows"], dt_out), dt, dt_out, given["psi0"], given["sweep"])
        return {"kind": "single", "sim": sim, "args": args, "output": case["output"]}
    if case["kind"] == "sweep":
        sim = ss.Simulator(_rabi if case["spin"] == "half" else _rabi_one, spin,
                           precision=case["precision"])
        args = (0.0, _end(_lengths(case), dt_out), dt, dt_out, given["psi0"], given["sweep"])
        options = {"with_spin": True, "compact": case["compact"]}
        state = {"kind": "sweep", "sim": sim, "args": args, "options": options, "plan": None}
        if case["graph"]:
            state["plan"] = ss.BatchPlan(sim, *args, **options).capture()
        return state
    controls = [ss.Control(a, given["grid"], order=case["order"]) for a in case["axes"]]
    sim = ss.ControlledSimulator(spin, controls, _bias, precision=case["precision"])
    amplitudes = torch.tensor(given["amplitudes"], device="cuda", requires_grad=True)
    args = (0.0, _end(case["rows"], dt_out), dt, dt_out, given["psi0"])
    return {"kind": "pulses", "sim": sim, "amplitudes": amplitudes, "args": args,
            "deterministic": case["deterministic"]}


def run(state):
    if state["kind"] == "single":
        r = state["sim"].evaluate(*state["args"], output=state["output"])
        return {"time": r.time, "operators": r.time_evolution, "states": r.state, "spin": r.spin}
    if state["kind"] == "sweep":
        if state["plan"] is not None:
            plan = state["plan"].replay()
            return {"time": plan.time, "operators": plan.u, "states": plan.state,
                    "spin": plan.spin_out}
        r = state["sim"].evaluate_batch(*state["args"], **state["options"])
        return {"time": r.time, "operators": r.time_evolution, "states": r.state, "spin": r.spin}
    amplitudes = state["amplitudes"]
    amplitudes.grad = None
    psi = state["sim"].final_state(amplitudes, *state["args"],
                                   deterministic=state["deterministic"])
    loss = (1 - psi[:, -1].abs() ** 2).sum()
    loss.backward()
    return {"final": psi.detach(), "loss": loss.detach(), "gradient": amplitudes.grad}


# ---- the same in plain 64-bit torch ----------------------------------------------
def _mm(a, b):
    return (a.unsqueeze(-1) * b.unsqueeze(-3)).sum(-2)


def _generator(g, d):
    """-i G of the field entries g (each (n,)), (n, d, d)."""
    g = [x.to(torch.complex128) for x in g]
    if d == 2:
        x, y, z = (0.5 * v for v in g[:3])
        rows = [[z, x - 1j * y], [x + 1j * y, -z]]
    else:
        zero = torch.zeros_like(g[0])
        x, y, z, q, u1, u2, v1, v2 = (g + [zero] * 8)[:8]
        a = (x - 1j * y + v1 - 1j * v2) / math.sqrt(2)
        b = (x - 1j * y - v1 + 1j * v2) / math.sqrt(2)
        u = u1 - 1j * u2
        rows = [[z + q / 3, a, u], [a.conj(), -2 * q / 3, b], [u.conj(), b.conj(), q / 3 - z]]
    return -1j * torch.stack([torch.stack(r, -1) for r in rows], -2)


def _expm1(a):
    """exp(a) - 1: closed form, or the series scaled and squared."""
    if a.shape[-1] == 2:  # a^2 = -theta^2
        theta = torch.sqrt(a[..., 0, 0].abs() ** 2 + a[..., 0, 1].abs() ** 2 + 1e-300)
        c = (-2 * torch.sin(0.5 * theta) ** 2).unsqueeze(-1).unsqueeze(-1)
        s = torch.sinc(theta / math.pi).unsqueeze(-1).unsqueeze(-1)
        return c * torch.eye(2, dtype=a.dtype, device=a.device) + s * a
    nu = float(a.detach().abs().sum(-1).max()) if a.numel() else 0.0
    squares = max(0, math.ceil(math.log2(nu / 0.1))) if nu > 0.1 else 0
    a = a * 0.5 ** squares
    nu *= 0.5 ** squares
    order, term = 1, nu
    while term > 1e-20 and order < 20:
        order += 1
        term *= nu / order
    eye = torch.eye(a.shape[-1], dtype=a.dtype, device=a.device)
    t = eye + a / order
    for k in range(order - 1, 1, -1):
        t = eye + _mm(a, t) / k
    b = _mm(a, t) if order > 1 else a
    for _ in range(squares):
        b = 2 * b + _mm(b, b)
    return b


def _fine_step(u, tf, tc, rot, dt, field, method, d, frame):
    """One integration step applied to the operators u, from the times tf."""
    def sample(offset):
        t_rel = (tf + offset) - tc
        f = field(t_rel + tc)
        if not frame:
            return f
        xy = torch.complex(f[0], f[1]) * torch.exp(-1j * (rot * t_rel))
        out = [xy.real, xy.imag, f[2] - rot] + list(f[3:])
        if len(f) == 8:
            uu = torch.complex(f[4], f[5]) * torch.exp(-2j * (rot * t_rel))
            vv = torch.complex(f[6], f[7]) * torch.exp(-1j * (rot * t_rel))
            out[4:] = [uu.real, uu.imag, vv.real, vv.imag]
        return out

    root = math.sqrt(3)
    if method == "midpoint":
        exps = [[dt * x for x in sample(0.5 * dt)]]
    elif method == "half_step":
        exps = [[0.5 * dt * x for x in sample(o)] for o in (0.0, dt)]
    else:
        a = sample(0.5 * dt * (1 - 1 / root))
        b = sample(0.5 * dt * (1 + 1 / root))
        w0, w1 = (1.5 + root) / 6, (1.5 - root) / 6
        exps = [[dt * (w0 * x + w1 * y) for x, y in zip(a, b)],
                [dt * (w1 * x + w0 * y) for x, y in zip(a, b)]]
    for g in exps:
        u = u + _mm(_expm1(_generator(g, d)), u)
    return u


def _operators(tc, dt, dt_out, field, method, d, frame, checkpoint=False):
    """Operators (n, d, d) of the output steps starting at tc; field(t) -> entries."""
    fine = round(dt_out / dt)
    dt = dt_out / fine
    u = torch.eye(d, dtype=torch.complex128, device=tc.device).expand(*tc.shape, d, d)
    rot = field(tc + dt_out / 2)[2] if frame else None
    tf = tc.clone()
    for _ in range(fine):
        if checkpoint:
            u = torch.utils.checkpoint.checkpoint(_fine_step, u, tf, tc, rot, dt, field, method, d,
                                                  frame, use_reentrant=False)
        else:
            u = _fine_step(u, tf, tc, rot, dt, field, method, d, frame)
        tf = tf + dt
    if frame:
        w = torch.exp(-1j * (rot * dt_out) * (0.5 if d == 2 else 1.0))
        exits = [w, w.conj()] if d == 2 else [w, torch.ones_like(w), w.conj()]
        u = torch.stack(exits, -1).unsqueeze(-1) * u
    return u


def _states(u, psi0):
    """States (..., n, d) before each of the n operators along dimension -3."""
    n, d = u.shape[-3], u.shape[-1]
    p = u.clone()
    s = 1
    while s < n:
        p[..., s:, :, :] = _mm(p[..., s:, :, :], p[..., :-s, :, :])
        s *= 2
    first = psi0.expand(*u.shape[:-3], 1, d)
    return torch.cat([first, (p[..., :-1, :, :] * psi0).sum(-1)], -2)


def _bloch(v):
    if v.shape[-1] == 2:
        p = v[..., 0] * v[..., 1].conj()
        return torch.stack([p.real, -p.imag, 0.5 * (v[..., 0].abs() ** 2 - v[..., 1].abs() ** 2)],
                           -1)
    c = v[..., 1].conj()
    a, b = c * (v[..., 0] + v[..., 2]), c * (v[..., 0] - v[..., 2])
    return torch.stack([math.sqrt(2) * a.real, -math.sqrt(2) * b.imag,
                        v[..., 0].abs() ** 2 - v[..., 2].abs() ** 2], -1)


def _interpolate(grid, amplitudes, order, t):
    """Linear or cubic interpolation of amplitudes (B, M) or (M,) on a grid of
    even steps at times t ((B, n) or (n,)), zero outside; tangents are the
    means of the neighbouring slopes, at the ends the end slope."""
    m = grid.numel()
    guess = ((t - grid[0]) / (grid[1] - grid[0])).long().clamp(0, m - 2)
    guess = torch.where(grid[guess] > t, guess - 1, guess).clamp(0, m - 2)
    i = torch.where(grid[guess + 1] <= t, guess + 1, guess).clamp(0, m - 2)
    h = grid[i + 1] - grid[i]
    p = (t - grid[i]) / h

    def at(x, k):
        return torch.gather(x, -1, k)
    a0, a1 = at(amplitudes, i), at(amplitudes, i + 1)
    if order == 1:
        out = a0 * (1 - p) + a1 * p
    else:
        slope = torch.diff(amplitudes, dim=-1) / torch.diff(grid)
        tangent = torch.cat([slope[..., :1], 0.5 * (slope[..., 1:] + slope[..., :-1]),
                             slope[..., -1:]], -1)
        l, r = at(tangent, i) * h, at(tangent, i + 1) * h
        out = (a0 * (2 * p ** 3 - 3 * p ** 2 + 1) + a1 * (3 * p ** 2 - 2 * p ** 3)
               + l * (p ** 3 - 2 * p ** 2 + p) + r * (p ** 3 - p ** 2))
    return torch.where((t >= grid[0]) & (t <= grid[-1]), out, torch.zeros_like(out))


def exact(case, seed):
    given = _inputs(case, seed)
    d = 2 if case["spin"] == "half" else 3
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    dt, dt_out = case["dt"], case["dt_out"]

    def there(x):
        return torch.as_tensor(np.ascontiguousarray(x), device=dev)
    psi0 = there(given["psi0"])
    if case["kind"] == "single":
        tc = there(dt_out * np.arange(case["rows"], dtype=np.float64))
        s = there(given["sweep"])
        if case["field"] == "noisy":
            grid, noise = (there(x) for x in given["noise"])

            def field(t):
                z = torch.full_like(t, 7e5)
                for k in range(8):
                    z = z + s[k] * torch.exp(-(t - s[8 + k]) ** 2 / (2 * s[16 + k] ** 2))
                return [TAU * 1e3 * torch.cos(TAU * 7e5 * t), torch.zeros_like(t),
                        TAU * z + _interpolate(grid, noise, 3, t)]
        else:
            base = _torch_field(case["field"])

            def field(t):
                return base(t, s)
        u = _operators(tc, dt, dt_out, field, case["method"], d, case["frame"])
        v = _states(u, psi0)
        return {"time": tc, "operators": u, "states": v, "spin": _bloch(v)}
    lengths = _lengths(case)
    if case["kind"] == "sweep":
        if int(lengths.sum()) * round(dt_out / dt) > 2.5e9:
            return None
        base = _torch_field("rabi" if d == 2 else "rabi_one")
        parts = []
        step = max(1, int(4e6 // case["longest"]))
        for k in range(0, case["sims"], step):  # a block of simulations, padded to the longest
            rows = lengths[k:k + step]
            s = there(given["sweep"][k:k + step].T[:, :, None])
            tc = there(dt_out * np.arange(rows.max(), dtype=np.float64)).expand(len(rows), -1)
            tc = tc.contiguous()
            u = _operators(tc, dt, dt_out, lambda t: base(t, s), "magnus_cf4", d, True)
            v = _states(u, psi0)
            keep = there(np.arange(rows.max())[None] < rows[:, None])
            parts.append((tc[keep], u[keep], v[keep]))
        tc, u, v = (torch.cat(x) for x in zip(*parts))
        columns = case["compact"] and case["graph"]  # (the plan's own store)
        return {"time": tc, "operators": u[:, :, 0].contiguous() if columns else u, "states": v,
                "spin": _bloch(v)}
    if case["sims"] * case["rows"] * round(dt_out / dt) > 1.1e8:
        return None
    grid = there(given["grid"])
    amplitudes = there(given["amplitudes"]).requires_grad_(True)
    tc = there(dt_out * np.arange(case["rows"], dtype=np.float64)).expand(case["sims"], -1)

    def field(t):
        f = [torch.zeros_like(t), torch.zeros_like(t), torch.full_like(t, TAU * 1e5)]
        for k, axis in enumerate(case["axes"]):
            j = "xyz".index(axis)
            f[j] = f[j] + _interpolate(grid, amplitudes[:, k], case["order"], t)
        return f
    u = _operators(tc.contiguous(), dt, dt_out, field, "magnus_cf4", d, True, checkpoint=True)
    while u.shape[1] > 1:  # products of neighbours, later ones on the left
        pairs = _mm(u[:, 1::2], u[:, 0:u.shape[1] // 2 * 2:2])
        u = pairs if u.shape[1] % 2 == 0 else torch.cat([pairs, u[:, -1:]], 1)
    psi = (u[:, 0] * psi0).sum(-1)
    loss = (1 - psi[:, -1].abs() ** 2).sum()
    loss.backward()
    return {"final": psi.detach(), "loss": loss.detach(), "gradient": amplitudes.grad}
