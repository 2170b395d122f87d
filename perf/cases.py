"""Performance cases: the work a user of the framework has it do, through its
public entry points, over the range it is used in.

Kinds of case
  grid      one model (FastScape): a start field in device memory is put into
            the model, `steps` time-steps are taken, the elevations are the
            result.  `advance` steps are taken while preparing, so the start
            field has the drainage depth of a run that far along.  `fill`
            fills depressions before every step.
  ensemble  realizations of uneven sizes and parameters (Ensemble): restart
            every one from its start field, run, fetch every field
  runs      inversion.exact_runs: the exact runs of a batch of candidates,
            from their parameters to their final fields, as the search's
            top-k reruns and the training set are made
  forward   UNet.forward on host arrays
  rank      UNet.rank: the misfit of every candidate against one target
  grad      UNet.loss_grad: the loss and every gradient of one batch
"""
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "barnes2019-landscape_amd"))

import fastscape_amd as fa  # noqa: E402
from fastscape_amd import inversion  # noqa: E402

# exact() simulates in numpy up to this many cell-steps
EXACT_CELL_STEPS = 3.2e7
SQRT2 = 1.414213562373095048801688724209698078569671875376948
# width, height of the network's levels and its convolutions (in, out, level),
# in the order of the parameter vector
CONVS = [(8, 32, 0), (32, 32, 0), (32, 64, 1), (64, 64, 1), (64, 128, 2), (128, 128, 2),
         (128, 160, 3), (160, 160, 3), (288, 128, 2), (128, 128, 2), (192, 64, 1), (64, 64, 1),
         (96, 32, 0), (32, 32, 0)]


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _grid(name, W, H, preset, steps, advance=0, fill=False):
    return {"name": name, "kind": "grid", "width": W, "height": H, "preset": preset,
            "steps": steps, "advance": advance, "fill": fill}


def listed():
    return [
        # the smallest run: a test-sized grid, launches and waits only
        _grid("run_101", 101, 101, "benchmark", 121),
        # the reference's own comparison run: its constants (n = 2), whose
        # drainage leaves the halo tiles within ten steps
        _grid("compare_501", 501, 501, "reference", 121),
        # the benchmark's first configuration
        _grid("run_1000", 1000, 1000, "benchmark", 121),
        # the middle of a long run, drainage 17 to 32 levels deep, ragged size
        _grid("midrun_1500x1101", 1500, 1101, "benchmark", 40, advance=600),
        # deep drainage on a large ragged grid
        _grid("deep_4097x3001", 4097, 3001, "reference", 6, advance=40),
        # the headline grid
        _grid("run_10000", 10000, 10000, "benchmark", 8, advance=5),
        # stepping with depression filling switched on
        _grid("filled_700x501", 700, 501, "benchmark", 4, fill=True),
        # an ensemble of uneven realizations, restarted and run
        {"name": "ensemble_mixed", "kind": "ensemble", "count": 12, "low": 300, "high": 1400,
         "steps": 120},
        # the exact reruns of the inversion's 32 best candidates
        {"name": "inversion_top32", "kind": "runs", "count": 32, "side": 256, "steps": 300},
        # one small prediction: latency
        {"name": "predict_64", "kind": "forward", "height": 64, "width": 64, "batch": 1,
         "max_batch": 16},
        # ranking candidates at the inversion's size
        {"name": "rank_256", "kind": "rank", "height": 256, "width": 256, "count": 256,
         "max_batch": 32},
        # the forward and backward pass of one training batch
        {"name": "grad_256", "kind": "grad", "height": 256, "width": 256, "batch": 32,
         "max_batch": 32},
    ]


def _spread(rng, low, high):
    """A whole number spread over the logarithm of [low, high]."""
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    kind = rng.choice(["grid", "grid", "grid", "deep", "fill", "ensemble", "runs", "forward",
                       "rank", "grad"])
    if kind in ("grid", "deep", "fill"):
        W, H = _spread(rng, 40, 6000), _spread(rng, 40, 6000)
        budget = 3e8   # cell-steps
        if kind == "fill":
            W, H = _spread(rng, 40, 1000), _spread(rng, 40, 1000)
            budget = 4e6
        steps = max(1, min(rng.randint(1, 120), int(budget / (W * H))))
        c = _grid("", W, H, "reference" if kind == "deep" else "benchmark", steps,
                  advance=rng.choice([0, 20, 60] if kind == "deep" else [0, 5, 300]),
                  fill=kind == "fill")
        del c["name"]
        if kind == "fill" or W * H > 4000000:
            c["advance"] = min(c["advance"], 20) if kind != "fill" else 0
        return c
    if kind == "ensemble":
        low = _spread(rng, 33, 500)
        return {"kind": "ensemble", "count": rng.randint(1, 16), "low": low,
                "high": _spread(rng, low, 1400), "steps": rng.randint(10, 100)}
    if kind == "runs":
        return {"kind": "runs", "count": _spread(rng, 1, 64), "side": 32 * rng.randint(1, 8),
                "steps": rng.randint(20, 150)}
    H, W = 32 * _spread(rng, 1, 8), 32 * _spread(rng, 1, 8)
    if kind == "rank":
        return {"kind": "rank", "height": H, "width": W, "count": _spread(rng, 1, 256),
                "max_batch": rng.choice([16, 32])}
    batch = _spread(rng, 1, 32)
    return {"kind": kind, "height": H, "width": W, "batch": batch, "max_batch": max(16, batch)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _Field:
    """A model's elevation field as an array that torch can look at; it keeps
    the model, which owns the memory."""

    def __init__(self, model):
        self.model = model
        self.__cuda_array_interface__ = {
            "shape": (model.height, model.width), "typestr": "<f8", "version": 3, "strides": None,
            "data": (model.device_h(), False)}


def _field(model):
    t = torch.as_tensor(_Field(model), device="cuda")
    t.model = model   # the memory lives as long as the tensor, whoever drops the state
    return t


def _preset(case):
    return fa.preset(fa.PRESET_REFERENCE if case["preset"] == "reference"
                     else fa.PRESET_BENCHMARK)


def _realizations(case, seed):
    """Uneven sides, spread over the logarithm of the case's range (the same
    ones whatever the seed), and the ensemble workload's parameters."""
    n = case["count"]
    sides = np.exp(np.random.default_rng(n).uniform(
        np.log(case["low"]), np.log(case["high"] + 1), (n, 2)))
    params = inversion.sample_params(n, np.random.default_rng(seed))
    return [dict(width=max(5, int(w)), height=max(5, int(h)), K=K, U=U, m=m,
                 seed=(int(seed) * 1000 + r) % 2**32)
            for r, ((w, h), (K, U, m)) in enumerate(zip(sides, params))]


def _candidates(case, seed):
    return inversion.sample_params(case["count"], np.random.default_rng(seed))


def _net_inputs(case, seed):
    """Network weights as training starts from them (He-normal, small biases),
    terrains, normalised parameters and standardised topographies."""
    rng = np.random.default_rng(seed)
    H, W = case["height"], case["width"]
    n = case.get("batch", 1)
    p = []
    for cin, cout, _ in CONVS:
        p.append(rng.standard_normal(9 * cin * cout, dtype=np.float32) * (2 / (9 * cin)) ** 0.5)
        p.append(rng.standard_normal(cout, dtype=np.float32) * 0.02)
    p.append(rng.standard_normal(33, dtype=np.float32) * (1 / 32) ** 0.5)
    terrain = rng.random((n, H, W), dtype=np.float32)
    terrain[:, :2] = terrain[:, -2:] = 0
    terrain[:, :, :2] = terrain[:, :, -2:] = 0
    params = rng.uniform(-1, 1, (case.get("count", n), 3)).astype(np.float32)
    y, x = np.mgrid[0:H, 0:W] / 40.0
    wave = rng.uniform(0, 6, (n, 2, 1, 1))
    target = np.sin(y + wave[:, 0]) + np.sin(x + wave[:, 1])
    target = (target + 0.3 * rng.standard_normal((n, H, W))).astype(np.float32)
    return np.concatenate(p).astype(np.float32), terrain, params, target


def prepare(case, seed):
    kind = case["kind"]
    if kind == "grid":
        m = fa.FastScape(case["width"], case["height"], _preset(case), engine_seed=seed)
        m.step(case["advance"])
        m.set_depression_fill(case["fill"])
        return {"kind": kind, "model": m, "start": _field(m).clone(), "steps": case["steps"]}
    if kind == "ensemble":
        ens = fa.Ensemble([fa.realization(r["width"], r["height"],
                                          fa.preset(fa.PRESET_BENCHMARK, keq=r["K"], ueq=r["U"],
                                                    meq=r["m"]), r["seed"])
                           for r in _realizations(case, seed)])
        ens.autotune(1, 100)
        return {"kind": kind, "ensemble": ens, "steps": case["steps"],
                "start": [ens.getH(r) for r in range(len(ens))]}
    if kind == "runs":
        return {"kind": kind, "params": _candidates(case, seed), "side": case["side"],
                "steps": case["steps"], "seed": seed}
    weights, terrain, params, target = _net_inputs(case, seed)
    net = fa.UNet(case["height"], case["width"], max_batch=case["max_batch"])
    net.set_params(weights)
    return {"kind": kind, "net": net, "terrain": terrain, "params": params, "target": target}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "grid":
        m = state["model"]
        _field(m).copy_(state["start"])
        torch.cuda.current_stream().synchronize()   # the model steps on its own stream
        m.step(state["steps"])
        return _field(m)
    if kind == "ensemble":
        ens = state["ensemble"]
        for r, h in enumerate(state["start"]):
            ens.setH(r, h)
        ens.run(state["steps"] - 1)
        return [ens.getH(r) for r in range(len(ens))]
    if kind == "runs":
        n, side = len(state["params"]), state["side"]
        out = np.empty((n, side, side))

        def keep(i, h):
            out[i] = h

        inversion.exact_runs(state["params"], state["seed"], side, state["steps"], batch=n,
                             on_result=keep)
        return out
    net = state["net"]
    if kind == "forward":
        return net.forward(state["terrain"], state["params"])
    if kind == "rank":
        return net.rank(state["terrain"][0], state["params"], state["target"][0])
    loss, grad = net.loss_grad(state["terrain"], state["params"], state["target"])
    return {"loss": np.float32(loss), "grad": grad}


def _cells(case):
    if case["kind"] == "grid":
        return case["width"] * case["height"]
    if case["kind"] == "runs":
        return case["count"] * case["side"] ** 2
    return sum(r["width"] * r["height"] for r in _realizations(case, 0))


def work(case):
    """A time-step reads every elevation and writes every new one; per cell,
    eight drops and their comparison, one count and one Newton iteration.  A
    network pass reads its inputs and weights and writes its outputs."""
    kind = case["kind"]
    if kind in ("grid", "ensemble", "runs"):
        n = _cells(case) * case["steps"]
        return {"bytes": 16.0 * n, "flops": 40.0 * n}
    H, W = case["height"], case["width"]
    B = case.get("batch", case.get("count"))
    per = sum(18.0 * i * o * (H >> lv) * (W >> lv) for i, o, lv in CONVS)
    weights = 4.0 * sum(9 * i * o + o for i, o, _ in CONVS)
    if kind == "rank":
        return {"bytes": weights + 8.0 * H * W + 16.0 * B, "flops": per * B}
    if kind == "forward":
        return {"bytes": weights + B * (8.0 * H * W + 12), "flops": per * B}
    return {"bytes": 2 * weights + B * (8.0 * H * W + 12), "flops": 3 * per * B}


# ---------------------------------------------------------------------------
# the same results in 64 bits, with numpy and torch alone
# ---------------------------------------------------------------------------
def _terrain64(W, H, seed):
    """Uniform [0, 1) from mt19937(seed), two words per cell; rings 0 and 1 are 0."""
    gen = np.random.MT19937()
    gen._legacy_seeding(int(seed) & 0xFFFFFFFF)
    raw = gen.random_raw(2 * W * H).astype(np.float64).reshape(-1, 2)
    h = ((raw[:, 0] + raw[:, 1] * 4294967296.0) / 18446744073709551616.0).reshape(H, W)
    h = np.minimum(h, np.nextafter(1.0, 0.0))
    h[:2] = h[-2:] = 0
    h[:, :2] = h[:, -2:] = 0
    return h


def _filled64(h):
    """The Priority-Flood+epsilon surface, by relaxation to its fixed point."""
    f = h.copy()
    f[2:-2, 2:-2] = np.inf
    while True:
        low = np.full_like(f[2:-2, 2:-2], np.inf)
        for dy in (1, 2, 3):
            for dx in (1, 2, 3):
                if (dy, dx) != (2, 2):
                    low = np.minimum(low, f[dy:dy + low.shape[0], dx:dx + low.shape[1]])
        new = np.minimum(f[2:-2, 2:-2], np.maximum(h[2:-2, 2:-2], np.nextafter(low, np.inf)))
        if np.array_equal(new, f[2:-2, 2:-2]):
            return f
        f[2:-2, 2:-2] = new


def _steps64(h, p, steps, fill=False):
    """Time-steps of the field h (H x W): steepest-descent receivers, upstream
    counts, uplift and the implicit stream-power update, level by level."""
    H, W = h.shape
    off = np.array([-1, -W - 1, -W, -W + 1, 1, W + 1, W, W - 1])
    dist = np.array([p["dx"], p["dx"] * SQRT2] * 4)
    mine = np.arange(W * H)
    inner = np.zeros((H, W), bool)
    inner[2:-2, 2:-2] = True
    inner = inner.ravel()
    cells = np.flatnonzero(inner)
    keq = p["K"] * p["dt"]
    for _ in range(steps):
        if fill:
            h = _filled64(h.reshape(H, W))
        h = h.ravel().copy()
        slope = np.stack([(h[cells] - h[cells + o]) / d for o, d in zip(off, dist)])
        best = slope.argmax(0)
        drains = slope[best, np.arange(len(cells))] > 0
        rcv = mine.copy()
        rcv[cells[drains]] = (cells + off[best])[drains]
        diag = np.zeros(W * H, bool)
        diag[cells] = best % 2 == 1
        lev, jump = (rcv != mine).astype(np.int64), rcv
        while True:
            more = lev[jump]
            if not more.any():
                break
            lev, jump = lev + more, jump[jump]
        order = np.argsort(lev, kind="stable")
        ends = np.cumsum(np.bincount(lev))
        count = np.ones(W * H)
        for k in range(len(ends) - 1, 0, -1):
            at = order[ends[k - 1]:ends[k]]
            np.add.at(count, rcv[at], count[at])
        h[inner] += p["U"] * p["dt"]
        length = np.where(diag, (p["dx"] * SQRT2) ** p["n"], p["dx"] ** p["n"])
        fact = keq * (count * p["area"]) ** p["m"] / length
        for k in range(1, len(ends)):
            at = order[ends[k - 1]:ends[k]]
            h0, hn, f = h[at], h[rcv[at]], fact[at]
            new, go = h0.copy(), np.arange(len(at))
            while len(go):
                x = new[go] - hn[go]
                step = ((new[go] - h0[go]) + f[go] * x ** p["n"]) / (
                    1 + f[go] * p["n"] * x ** (p["n"] - 1))
                was = new[go]
                new[go] = was - step
                go = go[np.abs(new[go] - was) > p["tol"]]
            h[at] = new
    return h.reshape(H, W)


def _params64(preset, **other):
    p = dict(K=2e-6, n=2, m=0.8, U=2e-3, dt=1000.0, dx=1.0, area=40000.0, tol=1e-3)
    if preset == "benchmark":
        p.update(K=1e-5, n=1, m=0.4, dx=100.0, area=1e4)
    p.update(other)
    return p


def _conv64(x, w, b):
    """3x3 convolution + ReLU of x (B, H, W, in) with w (9, out, in)."""
    B, H, W, _ = x.shape
    pad = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    y = b
    for t in range(9):
        y = y + pad[:, t // 3:t // 3 + H, t % 3:t % 3 + W] @ w[t].T
    return torch.relu(y)


def _net64(v, terrain, params):
    """The network's output (B, H, W) for the parameter vector v."""
    B, H, W = terrain.shape
    at, layers = 0, []
    for cin, cout, _ in CONVS:
        w = v[at:at + 9 * cin * cout].reshape(9, cout, cin)
        at += 9 * cin * cout
        layers.append((w, v[at:at + cout]))
        at += cout
    x = torch.cat([terrain[..., None], params[:, None, None, :].expand(B, H, W, 3),
                   torch.zeros(B, H, W, 4, dtype=v.dtype, device=v.device)], -1)
    skips = []
    for lv in range(4):
        x = _conv64(_conv64(x, *layers[2 * lv]), *layers[2 * lv + 1])
        if lv < 3:
            skips.append(x)
            x = x.reshape(B, H >> lv + 1, 2, W >> lv + 1, 2, -1).mean((2, 4))
    for j, lv in enumerate((2, 1, 0)):
        x = x.repeat_interleave(2, 1).repeat_interleave(2, 2)
        x = torch.cat([x, skips[lv]], -1)
        x = _conv64(_conv64(x, *layers[8 + 2 * j]), *layers[9 + 2 * j])
    return x @ v[at:at + 32] + v[at + 32]


def exact(case, seed):
    kind = case["kind"]
    if kind == "grid":
        if _cells(case) * (case["steps"] + case["advance"]) > EXACT_CELL_STEPS:
            return None
        if case["fill"] and _cells(case) * case["steps"] > 4e5:
            return None
        p = _params64(case["preset"])
        h = _steps64(_terrain64(case["width"], case["height"], seed), p, case["advance"])
        return _steps64(h, p, case["steps"], case["fill"])
    if kind in ("ensemble", "runs"):
        if _cells(case) * case["steps"] > EXACT_CELL_STEPS:
            return None
        if kind == "runs":
            side = case["side"]
            rows = [dict(width=side, height=side, K=K, U=U, m=m, seed=seed)
                    for K, U, m in _candidates(case, seed)]
        else:
            rows = _realizations(case, seed)
        out = [_steps64(_terrain64(r["width"], r["height"], r["seed"]),
                        _params64("benchmark", K=r["K"], U=r["U"], m=r["m"]), case["steps"])
               for r in rows]
        return np.stack(out) if kind == "runs" else out
    v, terrain, params, target = (
        torch.from_numpy(a).double().to("cuda" if torch.cuda.is_available() else "cpu")
        for a in _net_inputs(case, seed))
    B = len(params)
    out, grad, loss = [], torch.zeros_like(v), 0.0
    for b in range(0, B, 4):
        part = slice(b, min(B, b + 4))
        if kind == "forward":
            out.append(_net64(v, terrain[part], params[part]))
        elif kind == "rank":
            y = _net64(v, terrain.expand(len(params[part]), -1, -1), params[part])
            d = (y - target)[:, 2:-2, 2:-2]
            out.append(d.square().mean((1, 2)).sqrt())
        else:
            v.requires_grad_(True)
            some = (_net64(v, terrain[part], params[part]) - target[part]).square().sum()
            some = some / target.numel()
            grad += torch.autograd.grad(some, v)[0]
            loss += some.item()
    if kind == "grad":
        return {"loss": loss, "grad": grad.cpu().numpy()}
    return torch.cat(out).cpu().numpy()
