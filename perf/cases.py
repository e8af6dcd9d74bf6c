"""Performance cases: the solves that users of diffrax_amd run, through diffeqsolve.

Four families, each over its range of batch sizes, precisions and directions:
  lv    Lotka-Volterra, Dopri5, shared parameters, 100 saves of a fixed span
  vdp   Van der Pol ensembles with per-instance stiffness, span and save times, Tsit5
  node  the 64-256-256-64 neural ODE, Tsit5, 32 saves, both matmul forms
  sde   Ornstein-Uhlenbeck paths driven by given Brownian increments, Heun
Every case is a dict of plain values.  `prepare` makes what the caller holds (tensors on the
GPU), `run` is one call as a user writes it, `exact` the same quantities in float64 from
plain torch (tight fixed-step integration of the same equations), `work` the bytes and
operations that the path cannot do without.
"""
import math

import numpy as np
import torch

import diffrax_amd as dfx

LV_Q = (1.5, 1.0, 3.0, 1.0)
NODE_SHAPES = ((256, 64), (256,), (256, 256), (256,), (64, 256), (64,))
NODE_PARAMS = sum(math.prod(s) for s in NODE_SHAPES)


def listed():
    return [
        # One trajectory of a small system, as in an interactive session or an inner loop:
        # the cost is the call itself.
        dict(name="lv_1", kind="lv", batch=1, dtype="f64", n_ts=100, grad=False, dt0=0.1),
        # A small ensemble from random initial states (the batch a parameter study starts with).
        dict(name="lv_1024", kind="lv", batch=1024, dtype="f64", n_ts=100, grad=False, dt0=0.1),
        # The headline ensemble: uneven Van der Pol oscillators, one per lane of the GPU.
        dict(name="vdp_65536", kind="vdp", batch=65536, dtype="f64", n_ts=64, grad=False,
             dt0=0.1),
        # A mid-sized odd ensemble in the float32-state form, automatic first step.
        dict(name="vdp_f32_20011", kind="vdp", batch=20011, dtype="f32", n_ts=64, grad=False,
             dt0=None),
        # Fitting such an ensemble: forward and gradient for every initial state and mu.
        dict(name="vdp_grad_65536", kind="vdp", batch=65536, dtype="f64", n_ts=64, grad=True,
             dt0=0.1),
        # Serving a neural ODE to a handful of requests: latency of one tile and a remainder.
        dict(name="node_f32_33", kind="node", batch=33, matmul="f32", n_ts=32, grad=False,
             dt0=0.1, pcoeff=0.0),
        # Neural-ODE inference over a full batch, float32 products.
        dict(name="node_f32_8192", kind="node", batch=8192, matmul="f32", n_ts=32, grad=False,
             dt0=0.1, pcoeff=0.0),
        # The same in the bfloat16-MFMA form, at a batch that does not divide into the chip.
        dict(name="node_bf16_10007", kind="node", batch=10007, matmul="bf16", n_ts=32,
             grad=False, dt0=0.1, pcoeff=0.0),
        # One training step of the neural ODE (loss, gradients of all weights and y0).
        dict(name="node_grad_f32_8192", kind="node", batch=8192, matmul="f32", n_ts=32,
             grad=True, dt0=0.1, pcoeff=0.0),
        # A smaller training batch in the bfloat16-MFMA form, PI step control.
        dict(name="node_grad_bf16_3001", kind="node", batch=3001, matmul="bf16", n_ts=32,
             grad=True, dt0=0.1, pcoeff=0.2),
        # Simulating SDE paths forward from given increments.
        dict(name="sde_50003x8x500", kind="sde", paths=50003, d=8, steps=500, dtype="f32",
             grad=False),
        # Pathwise gradient of a terminal loss over a large set of long paths.
        dict(name="sde_grad_262144x16x1000", kind="sde", paths=262144, d=16, steps=1000,
             dtype="f32", grad=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("lv", "vdp", "node", "node", "sde"))
    if kind == "lv":
        return dict(kind="lv", batch=_log_int(rng, 1, 8192), dtype=rng.choice(("f64", "f32")),
                    n_ts=rng.randint(2, 128), grad=rng.random() < 0.3,
                    dt0=rng.choice((0.1, None)))
    if kind == "vdp":
        return dict(kind="vdp", batch=_log_int(rng, 64, 65536),
                    dtype=rng.choice(("f64", "f64", "f32")), n_ts=rng.randint(2, 64),
                    grad=rng.random() < 0.4, dt0=rng.choice((0.1, None)))
    if kind == "node":
        grad = rng.random() < 0.5
        return dict(kind="node", batch=_log_int(rng, 1, 8192 if grad else 16384),
                    matmul=rng.choice(("f32", "bf16")), n_ts=rng.randint(2, 32), grad=grad,
                    dt0=rng.choice((0.1, 0.1, None)), pcoeff=rng.choice((0.0, 0.0, 0.2)))
    dtype = rng.choice(("f32", "f32", "f32", "f64"))
    return dict(kind="sde", paths=_log_int(rng, 64, 131072), d=rng.choice((4, 8, 16, 32)),
                steps=rng.randint(50, 1000), dtype=dtype, grad=rng.random() < 0.5)


# ---- inputs ------------------------------------------------------------------------------
_DTYPE = {"f64": torch.float64, "f32": torch.float32}


def _lv_inputs(case, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(0.5, 2.0, (case["batch"], 2)), np.linspace(0.0, 10.0, case["n_ts"])


def _vdp_inputs(case, seed):
    rng = np.random.default_rng(seed)
    B = case["batch"]
    mu = np.exp(rng.uniform(np.log(0.1), np.log(5.0), B))
    y0 = rng.uniform(-2.0, 2.0, (B, 2))
    t1 = rng.uniform(5.0, 50.0, B)
    ts = np.linspace(0.0, 1.0, case["n_ts"])[None, :] * t1[:, None]
    ts[:, -1] = t1
    return mu, y0, t1, ts


def _node_inputs(case, seed):
    """Xavier-normal weights, small biases, N(0, 1) states, N(0, 0.5) targets (float32)."""
    rng = np.random.default_rng(seed)
    params = []
    for s in NODE_SHAPES:
        std = math.sqrt(2.0 / (s[0] + s[1])) if len(s) == 2 else 0.1
        params.append((rng.standard_normal(s) * std).astype(np.float32))
    y0 = rng.standard_normal((case["batch"], 64)).astype(np.float32)
    ts = np.linspace(0.0, 1.0, case["n_ts"])
    tgt = None
    if case["grad"]:
        tgt = rng.standard_normal((case["batch"], case["n_ts"], 64), dtype=np.float32)
        tgt *= np.float32(0.5)
    return params, y0, ts, tgt


def _sde_inputs(case, seed, device):
    """theta, mu, sigma, y0 from numpy; the increments N(0, dt) from torch's generator."""
    rng = np.random.default_rng(seed)
    P, d, N = case["paths"], case["d"], case["steps"]
    theta = rng.uniform(0.5, 2.0, d).astype(np.float32)
    mu = rng.standard_normal(d).astype(np.float32)
    sigma = rng.uniform(0.1, 0.5, d).astype(np.float32)
    y0 = rng.standard_normal((P, d)).astype(np.float32)
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    dW = torch.empty((N, P, d), dtype=torch.float32, device=device)
    for n in range(0, N, 100):
        dW[n:n + 100].normal_(0.0, math.sqrt(1.0 / N), generator=gen)
    return theta, mu, sigma, y0, dW


def prepare(case, seed):
    dev = torch.device("cuda")
    kind = case["kind"]
    if kind in ("lv", "vdp"):
        dt = _DTYPE[case["dtype"]]
        controller = dfx.PIDController(rtol=1e-6, atol=1e-8 if kind == "lv" else 1e-9)
        if kind == "lv":
            y0, ts = _lv_inputs(case, seed)
            st = dict(term=dfx.ODETerm(dfx.LotkaVolterra()), solver=dfx.Dopri5(), t1=10.0,
                      saveat=dfx.SaveAt(ts=torch.tensor(ts, dtype=torch.float64)),
                      max_steps=4096)
            args = torch.tensor(LV_Q, dtype=dt, device=dev)
        else:
            mu, y0, t1, ts = _vdp_inputs(case, seed)
            st = dict(term=dfx.ODETerm(dfx.VanDerPol()), solver=dfx.Tsit5(),
                      t1=torch.tensor(t1, dtype=torch.float64, device=dev),
                      saveat=dfx.SaveAt(ts=torch.tensor(ts, dtype=torch.float64, device=dev)),
                      max_steps=16384)
            args = torch.tensor(mu, dtype=dt, device=dev)
        y0 = torch.tensor(y0, dtype=dt, device=dev)
        if case["grad"]:
            y0.requires_grad_()
            args.requires_grad_()
        st.update(case=case, y0=y0, args=args, controller=controller)
        return st
    if kind == "node":
        params, y0, ts, tgt = _node_inputs(case, seed)
        params = [torch.tensor(p, device=dev, requires_grad=case["grad"]) for p in params]
        return dict(case=case, params=params,
                    term=dfx.ODETerm(dfx.MLPField(*params, matmul=case["matmul"])),
                    y0=torch.tensor(y0, device=dev, requires_grad=case["grad"]),
                    saveat=dfx.SaveAt(ts=torch.tensor(ts, dtype=torch.float64)),
                    target=None if tgt is None else torch.tensor(tgt, device=dev),
                    controller=dfx.PIDController(rtol=1e-5, atol=1e-7, pcoeff=case["pcoeff"],
                                                 icoeff=1.0 - case["pcoeff"]))
    theta, mu, sigma, y0, dW = _sde_inputs(case, seed, dev)
    dt = _DTYPE[case["dtype"]]
    args = tuple(torch.tensor(a, dtype=dt, device=dev, requires_grad=case["grad"])
                 for a in (theta, mu, sigma))
    return dict(case=case, args=args, y0=torch.tensor(y0, dtype=dt, device=dev),
                terms=dfx.MultiTerm(dfx.ODETerm(dfx.OUDrift()),
                                    dfx.ControlTerm(dfx.DiagonalNoise(), dfx.IncrementPath(dW))))


# ---- one call ----------------------------------------------------------------------------
def _solution(sol):
    return {"ys": sol.ys.detach(), "ts": sol.ts, "result": sol.result,
            "num_steps": sol.stats["num_steps"],
            "num_accepted_steps": sol.stats["num_accepted_steps"],
            "num_rejected_steps": sol.stats["num_rejected_steps"]}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("lv", "vdp"):
        def bound(args):
            if kind == "lv":
                return tuple(args.unbind(0)) if case["grad"] else LV_Q
            return args
        sol = dfx.diffeqsolve(state["term"], state["solver"], 0.0, state["t1"], case["dt0"],
                              state["y0"], bound(state["args"]), saveat=state["saveat"],
                              stepsize_controller=state["controller"],
                              max_steps=state["max_steps"], throw=not case["grad"])
        if not case["grad"]:
            return _solution(sol)
        loss = (sol.ys ** 2).mean()
        gy, ga = torch.autograd.grad(loss, (state["y0"], state["args"]))
        return {"loss": loss.detach(), "y0_grad": gy, "args_grad": ga, **_solution(sol)}
    if kind == "node":
        sol = dfx.diffeqsolve(state["term"], dfx.Tsit5(), 0.0, 1.0, case["dt0"], state["y0"],
                              saveat=state["saveat"], stepsize_controller=state["controller"],
                              throw=not case["grad"])
        if not case["grad"]:
            return _solution(sol)
        loss = ((sol.ys - state["target"]) ** 2).mean()
        grads = torch.autograd.grad(loss, [state["y0"], *state["params"]])
        return {"loss": loss.detach(), "grads": list(grads), **_solution(sol)}
    sol = dfx.diffeqsolve(state["terms"], dfx.Heun(), 0.0, 1.0, 1.0 / case["steps"],
                          state["y0"], state["args"], saveat=dfx.SaveAt(t1=True),
                          stepsize_controller=dfx.ConstantStepSize())
    if not case["grad"]:
        return {"ys": sol.ys, "ts": sol.ts}
    loss = (sol.ys ** 2).mean()
    grads = torch.autograd.grad(loss, state["args"])
    return {"loss": loss.detach(), "grads": list(grads), "ys": sol.ys.detach(), "ts": sol.ts}


# ---- the same quantities in float64 ---------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _rk4(f, y, h):
    k1 = f(y)
    k2 = f(y + (0.5 * h) * k1)
    k3 = f(y + (0.5 * h) * k2)
    k4 = f(y + h * k3)
    return y + (h / 6.0) * (k1 + 2.0 * (k2 + k3) + k4)


def _planar(kind, q, n_par, grad):
    """The field of a planar system on stacked rows [2 (+ 2 + 2 + 2 n_par), B]: the state
    and, with grad, the columns of its derivative by the initial state and parameters."""
    def f(Y):
        x, v = Y[0], Y[1]
        out = torch.empty_like(Y)
        if kind == "lv":
            a, b, g, dl = q
            out[0] = a * x - b * x * v
            out[1] = dl * x * v - g * v
        else:
            out[0] = v
            out[1] = q[0] * (1.0 - x * x) * v - x
        if grad:
            S0, S1 = Y[2::2], Y[3::2]          # d x / d p, d v / d p for every column p
            if kind == "lv":
                out[2::2] = (a - b * v) * S0 - (b * x) * S1
                out[3::2] = (dl * v) * S0 + (dl * x - g) * S1
                out[6] += x                    # d/d alpha
                out[8] -= x * v                # d/d beta
                out[11] -= v                   # d/d gamma
                out[13] += x * v               # d/d delta
            else:
                out[2::2] = S1
                out[3::2] = (-2.0 * q[0] * x * v - 1.0) * S0 + (q[0] * (1.0 - x * x)) * S1
                out[7] += (1.0 - x * x) * v    # d/d mu
        return out
    return f


def _exact_planar(case, seed):
    dev = _device()
    kind = case["kind"]
    dt = _DTYPE[case["dtype"]]
    # the parameters and states as the case's precision holds them
    held = lambda a: torch.tensor(a, dtype=dt).double().to(dev)
    if kind == "lv":
        y0, ts = _lv_inputs(case, seed)
        q = [held(v) for v in LV_Q]
        ts = torch.tensor(ts, device=dev)[:, None]
        sub = max(1, int(math.ceil(4000 / max(case["n_ts"] - 1, 1))))
    else:
        mu, y0, _, ts = _vdp_inputs(case, seed)
        q = [held(mu)]
        ts = torch.tensor(ts.T.copy(), device=dev)
        sub = max(1, int(math.ceil(12600 / max(case["n_ts"] - 1, 1))))
    B, grad, n_par = case["batch"], case["grad"], len(q)
    Y = torch.zeros((2 + (4 + 2 * n_par if grad else 0), B), dtype=torch.float64, device=dev)
    Y[:2] = held(y0).T
    if grad:
        Y[2] = 1.0
        Y[5] = 1.0
    f = _planar(kind, q, n_par, grad)
    rows = [Y]
    for n in range(1, case["n_ts"]):
        h = (ts[n] - ts[n - 1]) / sub
        for _ in range(sub):
            Y = _rk4(f, Y, h)
        rows.append(Y)
    R = torch.stack(rows)                       # [n_ts, rows, B]
    ys = R[:, :2].permute(2, 0, 1)
    out = {"ys": ys, "ts": None, "result": None, "num_steps": None,
           "num_accepted_steps": None, "num_rejected_steps": None}
    if not grad:
        return out
    gb = 2.0 * R[:, :2] / ys.numel()
    cols = (gb[:, :1] * R[:, 2::2] + gb[:, 1:] * R[:, 3::2]).sum(0)   # [2 + n_par, B]
    args = cols[2:].sum(1) if kind == "lv" else cols[2]
    return {"loss": (ys ** 2).mean(), "y0_grad": cols[:2].T, "args_grad": args, **out}


def _exact_node(case, seed):
    dev = _device()
    params, y0, ts, tgt = _node_inputs(case, seed)
    grad = case["grad"]
    W1, b1, W2, b2, W3, b3 = ps = [
        torch.tensor(p, dtype=torch.float64, device=dev).requires_grad_(grad) for p in params]
    y0 = torch.tensor(y0, dtype=torch.float64, device=dev).requires_grad_(grad)
    zero = torch.zeros((), dtype=torch.float64, device=dev)
    sp = lambda s: torch.logaddexp(s, zero)
    f = lambda y: torch.tanh(sp(sp(y @ W1.T + b1) @ W2.T + b2) @ W3.T + b3)
    with torch.set_grad_enabled(grad):
        y, rows = y0, [y0]
        sub = max(1, int(math.ceil((90 if grad else 240) / max(case["n_ts"] - 1, 1))))
        for n in range(1, case["n_ts"]):
            h = float(ts[n] - ts[n - 1]) / sub
            for _ in range(sub):
                y = _rk4(f, y, h)
            rows.append(y)
        ys = torch.stack(rows, dim=1)
    out = {"ys": ys.detach(), "ts": None, "result": None, "num_steps": None,
           "num_accepted_steps": None, "num_rejected_steps": None}
    if not grad:
        return out
    loss = ((ys - torch.tensor(tgt, device=dev)) ** 2).mean()
    grads = torch.autograd.grad(loss, [y0, *ps])
    return {"loss": loss.detach(), "grads": list(grads), **out}


def _exact_sde(case, seed):
    """Heun's steps in float64, with the derivatives by theta, mu and sigma carried along."""
    dev = _device()
    theta, mu, sigma, y0, dW = _sde_inputs(case, seed, dev)
    theta, mu, sigma = (torch.tensor(a, dtype=torch.float64, device=dev)
                        for a in (theta, mu, sigma))
    N = case["steps"]
    h = 1.0 / N
    y = torch.tensor(y0, dtype=torch.float64, device=dev)
    St, Sm, Ss = (torch.zeros_like(y) for _ in range(3)) if case["grad"] else (None,) * 3
    c = h * theta
    damp = 1.0 - c + 0.5 * c * c               # d y1 / d y0 of one step
    for n in range(N):
        w = dW[n].double()
        k0 = c * (mu - y) + sigma * w
        z = y + k0
        if case["grad"]:
            # y1 = y + (k0 + k1) / 2 with k1 = c (mu - z) + sigma w
            St = damp * St + 0.5 * h * ((1.0 - c) * (mu - y) + (mu - z))
            Sm = damp * Sm + 0.5 * c * (2.0 - c)
            Ss = damp * Ss + (1.0 - 0.5 * c) * w
        y = y + 0.5 * (k0 + c * (mu - z) + sigma * w)
    ys = y[:, None, :]
    if not case["grad"]:
        return {"ys": ys, "ts": None}
    g = 2.0 * y / y.numel()
    return {"loss": (y ** 2).mean(), "grads": [(g * S).sum(0) for S in (St, Sm, Ss)],
            "ys": ys, "ts": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "node":
        return _exact_node(case, seed)
    if kind == "sde":
        return _exact_sde(case, seed)
    return _exact_planar(case, seed)


# ---- what the path cannot do without -------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("lv", "vdp"):
        B, n, w = case["batch"], case["n_ts"], 8 if case["dtype"] == "f64" else 4
        q = 4 if kind == "lv" else 1
        per_instance_times = 8 * (n + 1) if kind == "vdp" else 0
        bytes_ = B * ((2 + 2 * n) * w + 8 * n + 16 + per_instance_times + (w if q == 1 else 0))
        # mean attempted steps of the family at these tolerances; 166 operations a step and
        # 63 a save forward, about 376 a step and 65 a save backward
        steps = 85 if kind == "lv" else 280
        flops = B * (166 * steps + 63 * n)
        if case["grad"]:
            bytes_ += B * (2 * n * w + (2 + q) * w)
            flops += B * (376 * steps * 0.77 + 65 * n)
        return {"bytes": bytes_, "flops": int(flops)}
    if kind == "node":
        B, n = case["batch"], case["n_ts"]
        evals = 6 * 3 + 1                       # three accepted steps and the first stage
        flops = B * evals * 196608
        bytes_ = B * (64 * 4 * (1 + n) + 8 * n + 16) + 4 * NODE_PARAMS
        if case["grad"]:                        # both products of the backward pass
            flops *= 3
            bytes_ += B * 64 * 4 * (2 * n + 1) + 4 * NODE_PARAMS
        return {"bytes": bytes_, "flops": flops}
    P, d, N = case["paths"], case["d"], case["steps"]
    w = 8 if case["dtype"] == "f64" else 4
    bytes_ = 4 * N * P * d + 2 * w * P * d
    flops = 13 * N * P * d
    if case["grad"]:
        flops += 20 * N * P * d
    return {"bytes": bytes_, "flops": flops}
