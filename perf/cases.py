"""What a user of this engine has it do, as measurable cases.

Three groups of calls, through the public entry points (the Python front end,
and the C ABI where records are taken as the drop-in adapters take them):

  plain    one Monte Carlo simulation of one of the four models
           (gs_run_plain), from a quick look at 1e4 particles to the headline
           workload's model at 2e7, with and without exit records;
  batch    many simulations of mixed models in one call (gs_run_batch);
  predict  the learned surrogate's inference on host or device buffers, and
  train    its training (forward, backward, Adam).

Sizes are those of the benchmark, the tests and the shipped data set: K0 1e22
to 1e23 cm^2/s, dt 50 to 500 s, injection log-uniform 0.01-100 GeV, 30 log
bins, 65,536 queries per call, minibatches of 512 rows.  Cases are kept below
about a second per pass.
"""
import ctypes
import math
import os

import numpy as np
import torch

from geliosphere_amd import abi, surrogate
from geliosphere_amd import engine as engine_mod

_DATA = os.path.join(os.path.dirname(os.path.abspath(engine_mod.__file__)), "data")
_MODELS = {"fp": abi.MODEL_1D_FP, "bp": abi.MODEL_1D_BP, "sp": abi.MODEL_2D_SOLARPROP, "ge": abi.MODEL_2D_GELIOSPHERE}
# FP64 operations of one particle-step of each model's equations.
_FLOPS_PER_STEP = {"fp": 42.0, "bp": 40.0, "sp": 164.0, "ge": 258.6}
_WEIGHTS = (abi.W_POWERLAW, abi.W_WEBER, abi.W_USOSKIN, abi.W_BURGER)
_WEIGHTS_1D = (abi.W_POWERLAW, abi.W_YAMADA)


def _plain(name, model, n, **over):
    case = {"kind": "plain", "model": model, "n": n, "K0": 5e22, "V": 400.0, "dt": 500.0, "r": 1.0, "theta": 90.0,
            "tilt": 10.0, "polarity": 1.0, "weights": 1, "records": False}
    case.update(over)
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # A quick look at a spectrum: few particles, so the longest
        # trajectory sets the time, not the throughput.
        _plain("bp_1e4", "bp", 10_000),
        # The reference CLI's default run: one million particles with every
        # exit record returned in id order (the records become log.dat).
        _plain("bp_records_1e6", "bp", 1_000_000, weights=2, records=True),
        # The headline workload's dominant model at throughput size.
        _plain("bp_2e7", "bp", 20_000_003),
        # The headline workload's other model: heavy-tailed lifetimes.
        _plain("fp_2e7", "fp", 20_000_003, weights=2),
        # 2D sweep points: both models, both polarities, wide current sheet,
        # every 2D spectrum; one modest and one large particle count.
        _plain("sp_3e4", "sp", 30_011, dt=100.0, tilt=75.0, polarity=-1.0, weights=4),
        _plain("ge_3e5", "ge", 300_007, dt=100.0, tilt=45.0, weights=4),
        # A 2D quick look at the coarse time step of the batch benchmark.
        _plain("ge_2e3", "ge", 2_000, dt=500.0, r=5.0, theta=60.0),
        # The batch benchmark's mix of models at reduced particle counts, as
        # data generation and Monte Carlo fallback run it.
        {"name": "batch_64", "kind": "batch", "sims": 64, "n_lo": 1000, "n_hi": 200_000},
        # One query from a fitting loop: the smallest call there is.
        {"name": "predict_host_1", "kind": "predict", "rows": 1, "device": False, "sd": True},
        # A parameter scan through host arrays (an odd number of rows).
        {"name": "predict_host_2e4", "kind": "predict", "rows": 20_011, "device": False, "sd": False},
        # The benchmark's inference call: 65,536 device-resident queries.
        {"name": "predict_device_65536", "kind": "predict", "rows": 65_536, "device": True, "sd": True},
        # Training epochs over a part of the shipped data set's size.
        {"name": "train_6500", "kind": "train", "rows": 6500, "batch": 512, "epochs": 2},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("plain", "plain", "plain", "plain", "batch", "predict", "predict", "train"))
    if kind == "batch":
        return {"kind": "batch", "sims": rng.randint(8, 64), "n_lo": 1000, "n_hi": _log_uniform(rng, 10_000, 200_000)}
    if kind == "predict":
        return {"kind": "predict", "rows": _log_uniform(rng, 1, 65_536), "device": rng.random() < 0.5,
                "sd": rng.random() < 0.5}
    if kind == "train":
        batch = rng.choice((512, 1024))
        return {"kind": "train", "rows": _log_uniform(rng, batch, 6500), "batch": batch, "epochs": 1}
    model = rng.choice(tuple(_MODELS))
    two_d = model in ("sp", "ge")
    case = _plain(None, model, 0, K0=10.0 ** rng.uniform(22.3, 23.0), V=400.0 if two_d else rng.uniform(300.0, 800.0),
                  dt=rng.choice((100.0, 500.0)), r=rng.uniform(1.0, 80.0), theta=rng.uniform(10.0, 170.0),
                  tilt=rng.uniform(5.0, 75.0) if two_d else 10.0, polarity=rng.choice((1.0, -1.0)) if two_d else 1.0,
                  weights=rng.randint(1, 4 if two_d else 2), records=not two_d and rng.random() < 0.25)
    top = max(work(c)["flops"] for c in listed() if c["kind"] == "plain")
    most = 0.5 * top / (_FLOPS_PER_STEP[model] * _mean_steps(case))
    case["n"] = _log_uniform(rng, 1000, min(most, 500_000 if case["records"] else 2e7))
    return case


def _mean_steps(c):
    """Mean steps of a particle: measured at r = 1 AU, K0 = 5e22 cm^2/s, V =
    400 km/s, then scaled as the lifetimes scale with dt, K0 and r."""
    depth = max(1.0 - (c["r"] / 100.0) ** 2, 0.05)
    if c["model"] == "fp":
        return 53.0 * (500.0 / c["dt"]) ** 0.5
    if c["model"] == "bp":
        return 14_760.0 * (500.0 / c["dt"]) * (c["K0"] / 5e22) ** -0.41 * depth
    base = 100_400.0 if c["polarity"] < 0 and c["model"] == "sp" else 37_000.0
    return base * (50.0 / c["dt"]) * (c["K0"] / 5e22) ** -0.41 * depth


# ------------------------------------------------------------------ state
_shared = {}


def _engine():
    """One engine for the whole program, launch shapes from the shipped
    autotuner cache, as the benchmark sets it up."""
    if "engine" not in _shared:
        eng = engine_mod.Engine(0)
        eng.autotune_load(os.path.join(_DATA, "autotune.txt"))
        _shared["engine"] = eng
    return _shared["engine"]


def _params(c, seed):
    two_d = c["model"] in ("sp", "ge")
    weights = (_WEIGHTS if two_d else _WEIGHTS_1D)[:c["weights"]]
    return abi.make_params(_MODELS[c["model"]], K0_cm2s=c["K0"], V_kms=c["V"], dt=c["dt"], N=c["n"], seed=seed + 1,
                           r_inj=c["r"], theta_deg=c["theta"], tilt_deg=c["tilt"], polarity=c["polarity"],
                           weights=weights)


def _batch_params(c, seed):
    """Simulations drawn as the batch benchmark draws them, with the coarser
    time steps and fewer particles."""
    rng = np.random.RandomState(1234)   # the simulations; `seed` keys their particles
    sims = []
    for i in range(c["sims"]):
        model = ("fp", "bp", "sp", "ge")[rng.randint(4)]
        two_d = model in ("sp", "ge")
        n = int(round(math.exp(rng.uniform(math.log(c["n_lo"]), math.log(c["n_hi"])))))
        sims.append(abi.make_params(
            _MODELS[model], K0_cm2s=10.0 ** rng.uniform(22.3, 23.0), V_kms=400.0 if two_d else rng.uniform(300.0, 800.0),
            dt=500.0 if two_d else (100.0, 500.0)[rng.randint(2)], N=n, seed=seed * 1000 + i + 1,
            r_inj=rng.uniform(1.0, 80.0), theta_deg=rng.uniform(10.0, 170.0),
            tilt_deg=rng.uniform(5.0, 75.0) if two_d else 10.0,
            polarity=(1.0, -1.0)[rng.randint(2)] if two_d else 1.0))
    return sims


def _queries(rows, seed):
    """Feature rows over the data set's ranges (surrogate.features)."""
    rng = np.random.RandomState(seed % (1 << 31))
    two_d = rng.randint(2, size=rows)
    sub = np.where(two_d == 1, rng.randint(2, size=rows), 1)
    x = np.empty((rows, surrogate.N_IN), dtype=np.float32)
    x[:, 0] = two_d
    x[:, 1] = sub
    x[:, 2] = rng.uniform(22.01, 22.99, rows)
    x[:, 3] = np.where(two_d == 1, rng.uniform(5.0, 75.0, rows), rng.uniform(300.0, 800.0, rows))
    x[:, 4] = np.where(two_d == 1, rng.choice([-1.0, 1.0], rows), 1.0)
    x[:, 5] = rng.uniform(1.0, 80.0, rows)
    x[:, 6] = rng.uniform(10.0, 170.0, rows)
    x[:, 7] = np.log10(rng.choice([50.0, 100.0, 500.0], rows))
    return x


def _ensemble():
    if "ensemble" not in _shared:
        sg = surrogate.Surrogate(0)
        sg.load(os.path.join(_DATA, "surrogate_weights.npz"))
        _shared["ensemble"] = sg
    return _shared["ensemble"]


class _OnDevice:
    """A torch tensor as the device array that predict_device takes."""

    def __init__(self, t, dtype):
        self.tensor, self.shape, self.dtype = t, tuple(t.shape), np.dtype(dtype)
        self.ptr = ctypes.c_void_p(t.data_ptr())


def prepare(case, seed):
    kind = case["kind"]
    if kind == "plain":
        state = {"kind": kind, "engine": _engine(), "params": _params(case, seed), "records": case["records"]}
        if case["records"]:
            state["buffer"] = (abi.GsExitRecord * case["n"])()
        return state
    if kind == "batch":
        return {"kind": kind, "engine": _engine(), "sims": _batch_params(case, seed)}
    if kind == "predict":
        x = _queries(case["rows"], seed)
        state = {"kind": kind, "model": _ensemble(), "device": case["device"], "sd": case["sd"], "x": x}
        if case["device"]:
            rows, no = case["rows"], surrogate.N_OUT
            state["x"] = _OnDevice(torch.from_numpy(x).cuda(), np.float32)
            state["mean"] = _OnDevice(torch.empty(rows, no, device="cuda"), np.float32)
            state["sd_out"] = _OnDevice(torch.empty(rows, no, device="cuda"), np.float32) if case["sd"] else None
            state["flags"] = _OnDevice(torch.empty(rows, dtype=torch.uint8, device="cuda"), np.uint8)
            torch.cuda.synchronize()
        return state
    rows = case["rows"]
    rng = np.random.RandomState((seed + 7) % (1 << 31))
    x = _queries(rows, seed)
    # modulation-like targets: smooth in the inputs, a few noisy or empty bins
    e = np.linspace(0.0, 1.0, surrogate.N_OUT)
    depth = (x[:, 5:6] / 100.0 - 1.0) * (24.0 - x[:, 2:3])
    y = (depth * np.exp(-3.0 * e)[None, :] + rng.normal(0.0, 0.02, (rows, surrogate.N_OUT))).astype(np.float32)
    w = (1.0 / (rng.uniform(0.0, 1e-3, y.shape) + 1e-4)).astype(np.float32)
    w[rng.uniform(size=w.shape) < 0.05] = 0.0
    model = surrogate.Surrogate(0, batch=case["batch"], lr=1e-4, seed=7)
    return {"kind": "train", "model": model, "x": x, "y": y, "w": w, "epochs": case["epochs"]}


# ------------------------------------------------------------------ the calls
def _arrays(spectra):
    """The spectra's arrays and counters, whole."""
    names = ("n_particles", "n_events", "n_outside", "total_steps", "n_nan", "n_step_cap", "n_acc_inexact",
             "n_acc_overflow")
    return {"count": np.array([np.ctypeslib.as_array(s.count) for s in spectra]).astype(np.int64),
            "sum_w": np.array([np.ctypeslib.as_array(s.sum_w) for s in spectra]),
            "sum_w2": np.array([np.ctypeslib.as_array(s.sum_w2) for s in spectra]),
            "stats": np.array([[getattr(s, k) for k in names] for s in spectra], dtype=np.int64)}


def run(state):
    kind = state["kind"]
    if kind == "plain":
        eng, p = state["engine"], state["params"]
        if not state["records"]:
            return _arrays([eng.run_plain(p)[0]])
        # the C ABI call of the drop-in adapters, into the caller's buffer
        s, n = abi.GsSpectrum(), ctypes.c_uint64(0)
        buf = state["buffer"]
        rc = engine_mod.lib().gs_run_plain(eng._ctx, ctypes.byref(p), ctypes.byref(s), buf, len(buf), ctypes.byref(n))
        if rc:
            raise RuntimeError("gs_run_plain: status %d" % rc)
        out = _arrays([s])
        kept = min(n.value, len(buf))
        out["records"] = np.frombuffer(buf, dtype=np.float64).reshape(-1, 6)[:kept, :5]
        out["ids"] = np.frombuffer(buf, dtype=np.int64).reshape(-1, 6)[:kept, 5]
        return out
    if kind == "batch":
        return _arrays(state["engine"].run_batch(state["sims"]))
    if kind == "predict":
        if state["device"]:
            state["model"].predict_device(state["x"], state["mean"], state["sd_out"], state["flags"])
            out = {"mean": state["mean"].tensor, "flags": state["flags"].tensor}
            if state["sd_out"] is not None:
                out["sd"] = state["sd_out"].tensor
            return out
        mean, sd, flags = state["model"].predict(state["x"], want_sd=state["sd"])
        out = {"mean": mean, "flags": flags}
        if sd is not None:
            out["sd"] = sd
        return out
    loss = state["model"].train(state["x"], state["y"], state["w"], state["epochs"])
    return {"loss": loss, "params": state["model"].get_params()}


# ------------------------------------------------------------------ what a call cannot do without
_SPECTRUM_BYTES = ctypes.sizeof(abi.GsSpectrum) + ctypes.sizeof(abi.GsParams)
_HIDDEN, _LAYERS, _MEMBERS = 256, 4, 4
_NET_PARAMS = (surrogate.N_IN * _HIDDEN + (_LAYERS - 1) * _HIDDEN * _HIDDEN + _HIDDEN * surrogate.N_OUT)


def work(case):
    kind = case["kind"]
    if kind == "plain":
        records = 48.0 * case["n"] if case["records"] else 0.0
        return {"bytes": _SPECTRUM_BYTES + records, "flops": case["n"] * _mean_steps(case) * _FLOPS_PER_STEP[case["model"]]}
    if kind == "batch":
        flops = 0.0
        for p in _batch_params(case, 0):
            c = {"model": [k for k, v in _MODELS.items() if v == p.model][0], "dt": p.dt, "r": p.r_inj,
                 "K0": p.K0 / abi.K0_CM2_TO_AU2, "polarity": p.polarity}
            flops += p.n_particles * _mean_steps(c) * _FLOPS_PER_STEP[c["model"]]
        return {"bytes": case["sims"] * _SPECTRUM_BYTES, "flops": flops}
    if kind == "predict":
        rows = case["rows"]
        out = surrogate.N_OUT * 4 * (2 if case["sd"] else 1) + 1
        return {"bytes": rows * (surrogate.N_IN * 4 + out) + _MEMBERS * _NET_PARAMS * 2,
                "flops": 2.0 * rows * _MEMBERS * _NET_PARAMS}
    steps = case["epochs"] * (case["rows"] // case["batch"])
    per_step = case["batch"] * _MEMBERS * _NET_PARAMS * 6.0
    # data set once, then per step the parameters, two moments and the shadow
    return {"bytes": case["rows"] * (surrogate.N_IN + 2 * surrogate.N_OUT) * 4 + steps * _MEMBERS * _NET_PARAMS * 28,
            "flops": steps * per_step}


def exact(case, seed):
    """The surrogate's outputs from its weights in 64 bits.  A Monte Carlo
    run has no such value within seconds (1e4 to 1e6 dependent steps per
    particle), and a training run depends on the library's minibatch order."""
    if case["kind"] != "predict":
        return None
    d = np.load(os.path.join(_DATA, "surrogate_weights.npz"), allow_pickle=False)
    x = (_queries(case["rows"], seed).astype(np.float64) - d["mean"].astype(np.float64)) / d["sd"].astype(np.float64)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    members, hidden, layers = (int(v) for v in d["config"])
    pad = 32
    widths = [pad] + [hidden] * layers + [pad]
    flat = torch.from_numpy(d["params"].astype(np.float64)).to(dev).reshape(members, -1)
    inputs = torch.zeros(case["rows"], pad, dtype=torch.float64, device=dev)
    inputs[:, :x.shape[1]] = torch.from_numpy(x).to(dev)
    outs = []
    for m in range(members):
        a, at = inputs, 0
        for i, (n_in, n_out) in enumerate(zip(widths[:-1], widths[1:])):
            weight = flat[m, at:at + n_in * n_out].reshape(n_out, n_in)
            at += n_in * n_out
            a = a @ weight.t() + flat[m, at:at + n_out]
            at += n_out
            if i < layers:
                a = a * torch.sigmoid(a)
        outs.append(a[:, :surrogate.N_OUT])
    y = torch.stack(outs)
    # The members' spread (and the flags set from it) is of the size of their
    # bf16 rounding: 64 bits say nothing about it.
    return {"mean": y.mean(0), "flags": None, "sd": None} if case["sd"] else {"mean": y.mean(0), "flags": None}
