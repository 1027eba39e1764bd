"""The work that a user of this framework has it do, as measurable cases.

Each case goes through the package's public Python surface (Solver, Ensemble,
cnn.Network) or, for the batched tridiagonal solve, the C entry point for
callers with device buffers.  Kinds:

  run       Solver.run (or Solver.step) of a river or a channel: the time step
            that the library exists for, between two host events of a program
            (rep.py downloads fields every so many steps)
  ensemble  Ensemble.run: scenarios of several rivers stepped together
  macro     one macro step of the surrogate driver: the network's prediction
            into the state, then sediment steps on the predicted flow and the
            repeated bed change
  train     Network.train_samples, one optimiser step of the surrogate's
            training on samples captured from a state
  forward   Network.forward on loaded host images
  thomas    hd_thomas_batch_noalloc on device arrays

Sizes are those of the synthetic workloads of hydist_amd.synth (the 300 x 60
channel, the 980 x 1048 river and its scaled forms, rivers of 256-1024 a
side) and of the surrogate driver (8 layers, batches of 1-4 images on the
river's grid).
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-hydist_amd"))

from hydist_amd import _lib, cnn, synth  # noqa: E402
from hydist_amd._lib import Ensemble, Solver  # noqa: E402
from hydist_amd.case import BED_EVERY_STEP  # noqa: E402

LAYERS = 8
SCALES = dict(s_u=1.0, s_v=1.0, s_z=1.0, s_b=1e30, s_q=3000.0, s_h=10.0, d_u=0.02, d_v=0.02, d_z=0.01)
WET_RIVER = 85600        # wet cells of the 980 x 1048 river


def listed():
    return [
        # a host loop around a small case: one step per call, latency alone
        {"name": "channel_step", "kind": "run", "shape": "channel", "N": 300, "M": 60, "steps": 1, "spin": 40,
         "sediment": False, "single": True},
        # the small channel between two outputs a few minutes apart
        {"name": "channel_run", "kind": "run", "shape": "channel", "N": 300, "M": 60, "steps": 30, "spin": 40,
         "sediment": False, "single": False},
        # the 980 x 1048 river while its flow starts from rest, each pass a
        # what-if run from the same saved state
        {"name": "river_start", "kind": "run", "shape": "river", "scale": 1.0, "axis": "i", "river": 2, "steps": 20,
         "spin": 5, "sediment": False, "single": False, "restart": True},
        # the same river once its flow is established, five minutes a pass
        {"name": "river_run", "kind": "run", "shape": "river", "scale": 1.0, "axis": "i", "river": 2, "steps": 60,
         "spin": 300, "sediment": False, "single": False},
        # an odd-sized smaller river along the other axis
        {"name": "river_ragged", "kind": "run", "shape": "river", "scale": 0.37, "axis": "j", "river": 7, "steps": 37,
         "spin": 150, "sediment": False, "single": False},
        # suspended sediment and bed change in every step
        {"name": "river_sediment", "kind": "run", "shape": "river", "scale": 1.0, "axis": "i", "river": 2, "steps": 24,
         "spin": 150, "sediment": True, "single": False},
        # scenarios of several rivers in one batch, sediment on
        {"name": "ensemble_12", "kind": "ensemble", "members": 12, "side_min": 256, "side_max": 640, "river": 4,
         "steps": 10, "spin": 40},
        # the surrogate driver's macro step on the river
        {"name": "macro_river", "kind": "macro", "scale": 1.0, "river": 2, "substeps": 6},
        # the surrogate's training: the driver's images on the river's grid,
        # and the small river's
        {"name": "train_river", "kind": "train", "N": 980, "M": 1048, "batch": 2},
        {"name": "train_small", "kind": "train", "N": 98, "M": 105, "batch": 4},
        # prediction of host images
        {"name": "forward_mid", "kind": "forward", "H": 248, "W": 265, "batch": 2},
        # tridiagonal systems of a half-step's number and lengths
        {"name": "thomas_lines", "kind": "thomas", "systems": 2000, "rows_min": 24, "rows_max": 503},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "sediment", "ensemble", "macro", "train", "forward", "thomas"])
    if kind == "run" and rng.random() < 0.3:
        return {"kind": "run", "shape": "channel", "N": int(_log(rng, 40, 400)), "M": rng.randint(12, 90),
                "steps": int(_log(rng, 1, 60)), "spin": rng.randint(5, 60), "sediment": False, "single": False}
    if kind in ("run", "sediment"):
        return {"kind": "run", "shape": "river", "scale": round(_log(rng, 0.12, 1.0), 3), "axis": rng.choice(["i", "j"]),
                "river": rng.randint(2, 9), "steps": int(_log(rng, 1, 60 if kind == "run" else 24)),
                "spin": rng.choice([5, 60, 200]), "sediment": kind == "sediment", "single": False}
    if kind == "ensemble":
        return {"kind": "ensemble", "members": rng.randint(2, 10), "side_min": rng.randint(200, 300),
                "side_max": rng.randint(301, 600), "river": rng.randint(2, 9), "steps": rng.randint(1, 10), "spin": 20}
    if kind == "macro":
        return {"kind": "macro", "scale": round(_log(rng, 0.15, 1.0), 3), "river": rng.randint(2, 9),
                "substeps": rng.randint(1, 12)}
    if kind == "train":
        N, M = int(_log(rng, 30, 980)), int(_log(rng, 30, 1048))
        return {"kind": "train", "N": N, "M": M, "batch": rng.randint(1, 2) if N * M > 200000 else rng.randint(1, 4)}
    if kind == "forward":
        H, W = int(_log(rng, 9, 500)), int(_log(rng, 9, 500))
        return {"kind": "forward", "H": H, "W": W, "batch": rng.randint(1, 3)}
    lo = rng.randint(2, 60)
    return {"kind": "thomas", "systems": int(_log(rng, 1, 2000)), "rows_min": lo, "rows_max": lo + int(_log(rng, 1, 450))}


# ---------------------------------------------------------------- time steps

@functools.lru_cache(maxsize=24)
def _river(scale, axis, river, sediment, hours):
    return synth.config(3 if sediment else 2, scale=scale, hours=hours, seed=river, axis=axis, SL=24)


@functools.lru_cache(maxsize=24)
def _member(k, river, lo, hi, hours):
    return synth.ensemble_member(k, seed=river, side_min=lo, side_max=hi, hours=hours)


def _scenario(base, rng):
    """`base` with seeded inflow and roughness: another scenario of that river."""
    c = synth.dataclasses.replace(base, arrays=dict(base.arrays))
    inflow = rng.uniform(0.75, 1.25)
    for k in ("bc_up", "bc_down", "bc_left", "bc_right"):
        c.arrays[k] = base.arrays[k] * inflow
    c.arrays["hsnham"] = base.arrays["hsnham"] * (1.0 + 0.1 * rng.uniform(-1.0, 1.0))
    return c


class _Device:
    """Memory of a context for torch (the device structs that
    Solver.struct_ptrs hands to a caller's own code).  The tensor made from it
    holds this object, and this object the context that owns the memory."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": tuple(shape), "typestr": typestr,
                                         "version": 2}


ARG = ["bienQ", "daui", "dauj", "cuoii", "cuoij", "moci", "mocj", "khouot", "boundary_type", "h", "v", "u", "z", "t_u",
       "t_v", "t_z", "Htdu", "Htdv", "H_moi", "htaiz", "htaiz_bd", "ubt", "ubp", "vbt", "vbd", "hsnham", "VISCOIDX",
       "Kx1", "Ky1", "Tsyw", "Tsxw", "bc_up", "bc_down", "bc_left", "bc_right", "hi", "FS", "tFS", "CC_u", "CC_d",
       "CC_l", "CC_r", "VTH", "Kx", "Ky", "Fw", "Qbx", "Qby", "dH"]


def _fields(solver, names):
    """Device views of 2-D fields of a context."""
    arg, _ = solver.struct_ptrs()
    head = 8 + 4 * 8
    raw = torch.as_tensor(_Device(solver, arg, (head + 8 * len(ARG),), "|u1"), device="cuda").cpu().numpy()
    ptr = raw[head:].view(np.int64)
    shape = (solver.N + 3, solver.M + 3)
    return [torch.as_tensor(_Device(solver, ptr[ARG.index(n)], shape, "<i4" if n == "khouot" else "<f8"), device="cuda")
            for n in names]


FLOW = ["u", "v", "z", "khouot", "H_moi"]
SEDIMENT = FLOW + ["FS", "dH", "VTH"]


def _prepare_run(case, rng):
    n, spin = case["steps"], case["spin"]
    window = max(n, 240)
    if case["shape"] == "channel":
        base = synth.channel_case(N=case["N"], M=case["M"], nsteps=3600, Q=500.0 * case["M"] / 60.0)
    else:
        base = _river(case["scale"], case["axis"], case["river"], case["sediment"], 1.0)
    c = _scenario(base, rng)
    over = {}
    if case["sediment"]:
        c.bed_mode = BED_EVERY_STEP
        over = dict(sediment_start=0.0, bed_change_start=0.0)
    opts = c.opts(**over)
    g = Solver(c)
    g.init()
    t0 = g.run(0.0, spin, opts)
    home = g.clone()
    return {"solver": g, "home": home, "opts": opts, "t": t0, "t0": t0, "steps": n, "single": case["single"],
            "end": t0 if case.get("restart") else t0 + window * c.dT, "span": n * c.dT,
            "out": _fields(g, SEDIMENT if case["sediment"] else FLOW)}


def _run_run(s):
    # on in time from where the last pass ended; at the end of its window, or
    # in every pass of a what-if case, back to the saved state
    if s["t"] + s["span"] > s["end"] and s["t"] != s["t0"]:
        s["solver"].copy_state_from(s["home"])
        s["t"] = s["t0"]
    if s["single"]:
        s["t"] = s["solver"].step(s["t"], s["opts"])
    else:
        s["t"] = s["solver"].run(s["t"], s["steps"], s["opts"])
    return s["out"]


def _prepare_ensemble(case, rng):
    ms = []
    for k in range(case["members"]):
        c = _scenario(_member(k, case["river"], case["side_min"], case["side_max"], 1.0), rng)
        g = Solver(c)
        g.init()
        ms.append(g)
    opts = c.opts()
    ens = Ensemble(ms)
    t0 = ens.run(0.0, case["spin"], opts)
    homes = [m.clone() for m in ms]
    out = [x for m in ms for x in _fields(m, ["u", "v", "z", "FS", "khouot"])]
    return {"ensemble": ens, "members": ms, "homes": homes, "opts": opts, "t": t0, "t0": t0, "steps": case["steps"],
            "end": t0 + 120 * c.dT, "span": case["steps"] * c.dT, "out": out}


def _run_ensemble(s):
    if s["t"] + s["span"] > s["end"]:
        for m, home in zip(s["members"], s["homes"]):
            m.copy_state_from(home)
        s["t"] = s["t0"]
    s["t"] = s["ensemble"].run(s["t"], s["steps"], s["opts"])
    return s["out"]


# ------------------------------------------------------------- the surrogate

def _weights(rng):
    """He-uniform weights in the network's padded layout ([9][cout][cin],
    channels 32 / 64 / 32), the last layer small."""
    out = []
    for l in range(LAYERS):
        ci, co = (32 if l == 0 else 64), (32 if l == LAYERS - 1 else 64)
        ri, ro = (8 if l == 0 else 64), (3 if l == LAYERS - 1 else 64)
        a = math.sqrt(6.0 / (9.0 * ri)) * (0.1 if l == LAYERS - 1 else (1.0 if l == 0 else 0.5))
        w, b = np.zeros((9, co, ci), np.float32), np.zeros(co, np.float32)
        w[:, :ro, :ri] = rng.uniform(-a, a, (9, ro, ri))
        b[:ro] = rng.uniform(-0.05, 0.05, ro)
        out.append((w, b))
    return out


def _network(H, W, batch, weights):
    net = cnn.Network(H, W, batch=batch, layers=LAYERS)
    net.set_scales(**SCALES)
    for l, (w, b) in enumerate(weights):
        net.set_layer(l, w, b)
    return net


def _prepare_macro(case, rng):
    c = _scenario(_river(case["scale"], "i", case["river"], True, 2.0), rng)
    c.bed_mode = BED_EVERY_STEP
    opts = c.opts(sediment_start=0.0, bed_change_start=0.0)
    g = Solver(c)
    g.init()
    t0 = g.run(0.0, 120, opts)
    weights = _weights(rng)
    # a trained network predicts increments far smaller than an untrained one's
    weights[-1] = (weights[-1][0] * np.float32(0.02), weights[-1][1] * np.float32(0.02))
    net = _network(c.N + 3, c.M + 3, 1, weights)
    return {"solver": g, "home": g.clone(), "net": net, "opts": opts, "t0": t0, "calls": 0, "steps": 60,
            "substeps": case["substeps"], "dT": c.dT, "q": float(c.arrays["bc_left"][0]), "zb": 0.05,
            "out": _fields(g, SEDIMENT)}


def _run_macro(s):
    # the surrogate driver's call; every eighth one starts again from the last
    # verified state, as after a check that failed
    g, t, m = s["solver"], s["t0"], s["substeps"]
    if s["calls"] and s["calls"] % 8 == 0:
        g.copy_state_from(s["home"])
    s["calls"] += 1
    s["net"].predict_into(g, s["q"], s["zb"])
    if m > 1:
        t = g.sediment_run(t, m - 1, s["opts"])
    g.bed_snapshot()
    g.sediment_run(t, 1, s["opts"])
    g.bed_extrapolate(s["steps"] - m)
    return s["out"]


def _smooth(rng, H, W, amp):
    """A smooth field: a few seeded plane waves."""
    i, j = np.arange(H)[:, None], np.arange(W)[None, :]
    f = np.zeros((H, W))
    for _ in range(4):
        ki, kj = rng.uniform(-0.15, 0.15, 2)
        f += rng.uniform(0.3, 1.0) * np.sin(ki * i + kj * j + rng.uniform(0, 2 * math.pi))
    return amp * f / 2.0


def _band(rng, H, W):
    """A river-like wet band across the image."""
    i, j = np.arange(H)[:, None], np.arange(W)[None, :]
    mid = H / 2 + 0.3 * H * np.sin(j * (2 * math.pi / max(W, 8)) + rng.uniform(0, 6))
    return np.abs(i - mid) < max(2.0, 0.12 * H)


def _states(case, seed):
    """Per sample: wet mask, depth, and the fields u, v, z now and at the horizon."""
    rng = np.random.default_rng([seed, 11])
    H, W = case["N"] + 3, case["M"] + 3
    out = []
    for _ in range(case["batch"]):
        wet = _band(rng, H, W)
        wet[0], wet[-2:], wet[:, 0], wet[:, -2:] = False, False, False, False
        h = np.where(wet, 4.0 + _smooth(rng, H, W, 1.0), 0.0)
        now = [_smooth(rng, H, W, a) for a in (0.6, 0.6, 0.3)]
        then = [f + _smooth(rng, H, W, d) for f, d in zip(now, (0.02, 0.02, 0.01))]
        out.append((wet, h, now, then, rng.uniform(2000.0, 4000.0), rng.uniform(-0.3, 0.3)))
    return out


def _prepare_train(case, seed):
    N, M, B = case["N"], case["M"], case["batch"]
    net = _network(N + 3, M + 3, B, _weights(np.random.default_rng([seed, 12])))
    net.data_alloc(B)
    header = synth.make_case_header(20.0, 20.0, 5.0, 24)
    g = Solver(params=synth.params_from_dict(synth.parse_case_header(header)), N=N, M=M, series_len=3, total_time=3)
    for k, (wet, h, now, then, q, zb) in enumerate(_states(case, seed)):
        g.set("khouot", np.where(wet, 0, 2))
        g.set("h", h)
        for role, fields in ((0, now), (1, then)):
            for name, f in zip(("u", "v", "z"), fields):
                g.set(name, f)
            net.capture(k, role, g, q, zb)
    g.close()
    return {"net": net, "idx": list(range(B)), "lr": 5e-4}


def _run_train(s):
    loss = s["net"].train_samples(s["idx"], s["lr"])
    return [loss] + [list(s["net"].get_grad(l)) for l in range(LAYERS)]


def _images(case, seed):
    rng = np.random.default_rng([seed, 13])
    H, W = case["H"], case["W"]
    x = np.zeros((case["batch"], H, W, 8), np.float32)
    for b in range(case["batch"]):
        wet = _band(rng, H, W)
        for c, a in enumerate((0.6, 0.6, 0.3)):
            x[b, ..., c] = np.where(wet, _smooth(rng, H, W, a), 0.0)
        x[b, ..., 4] = wet
        x[b, ..., 5], x[b, ..., 6] = rng.uniform(0.7, 1.3), rng.uniform(-0.3, 0.3)
        x[b, ..., 7] = np.where(wet, 0.4 + _smooth(rng, H, W, 0.1), 0.0)
    return x


def _prepare_forward(case, seed):
    net = _network(case["H"], case["W"], case["batch"], _weights(np.random.default_rng([seed, 12])))
    net.load(_images(case, seed))
    return {"net": net}


# ------------------------------------------------------- tridiagonal systems

def _systems(case, seed):
    """Diagonally dominant systems, as a half-step's lines have them: lengths
    uniform in [rows_min, rows_max] and of the case alone (a mask's lines keep
    their lengths), flat arrays A (lower), B, C (upper), D."""
    rows = np.random.default_rng(14).integers(case["rows_min"], case["rows_max"] + 1, case["systems"])
    rng = np.random.default_rng([seed, 14])
    off = np.concatenate([[0], np.cumsum(rows)[:-1]])
    n = int(rows.sum())
    A, C = rng.uniform(-0.6, 0.2, n), rng.uniform(-0.6, 0.2, n)
    B = 1.0 + np.abs(A) * rng.uniform(0.6, 1.2, n) + np.abs(C) * rng.uniform(0.6, 1.2, n)
    D = rng.normal(0.0, 1.0, n)
    A[off] = 0.0
    C[off + rows - 1] = 0.0
    return rows, off, A, B, C, D


def _prepare_thomas(case, seed):
    rows, off, *abcd = _systems(case, seed)
    dev = [torch.from_numpy(a).cuda() for a in abcd]
    return {"systems": len(rows), "rows": int(rows.sum()), "off": torch.from_numpy(off.astype(np.int32)).cuda(),
            "sn": torch.from_numpy((rows - 1).astype(np.int32)).cuda(), "abcd": dev,
            "x": torch.zeros(int(rows.sum()), dtype=torch.float64, device="cuda")}


def _run_thomas(s):
    _lib.check(_lib.load().hd_thomas_batch_noalloc(
        0, s["systems"], s["off"].data_ptr(), s["sn"].data_ptr(), *(a.data_ptr() for a in s["abcd"]),
        s["x"].data_ptr(), s["rows"], torch.cuda.current_stream().cuda_stream))
    return s["x"]


# ------------------------------------------------------------------ the case

def prepare(case, seed):
    k = case["kind"]
    if k in ("train", "forward", "thomas"):
        return {"kind": k, **{"train": _prepare_train, "forward": _prepare_forward,
                              "thomas": _prepare_thomas}[k](case, seed)}
    rng = np.random.default_rng([seed, 10])
    return {"kind": k, **{"run": _prepare_run, "ensemble": _prepare_ensemble, "macro": _prepare_macro}[k](case, rng)}


def run(state):
    k = state["kind"]
    if k == "run":
        return _run_run(state)
    if k == "ensemble":
        return _run_ensemble(state)
    if k == "macro":
        return _run_macro(state)
    if k == "train":
        return _run_train(state)
    if k == "forward":
        return state["net"].forward()
    return _run_thomas(state)


FLOP_PIXEL = 2 * 9 * (8 * 64 + (LAYERS - 2) * 64 * 64 + 64 * 3)    # one forward pass


def work(case):
    k = case["kind"]
    if k == "run":
        if case["shape"] == "channel":
            wet = case["N"] * (case["M"] - 4)
        else:
            wet = WET_RIVER * case["scale"] ** 2
        # fields read and written per wet cell and step, FP64
        return {"bytes": (304 + 116 if case["sediment"] else 256) * wet * case["steps"], "flops": 0}
    if k == "ensemble":
        side = 0.5 * (case["side_min"] + case["side_max"])
        return {"bytes": 304 * case["members"] * 80.0 * side * case["steps"], "flops": 0}
    if k == "macro":
        wet = WET_RIVER * case["scale"] ** 2
        return {"bytes": (2 * 88 + 2 * 80 + 2 * 16 + 176) * wet * case["substeps"], "flops": FLOP_PIXEL * wet}
    if k == "train":
        px = (case["N"] + 3) * (case["M"] + 3) * case["batch"]
        return {"bytes": px * 64 * 2 * 2 * 3 * LAYERS, "flops": 3 * FLOP_PIXEL * px}
    if k == "forward":
        px = case["H"] * case["W"] * case["batch"]
        return {"bytes": px * (32 + 12), "flops": FLOP_PIXEL * px}
    n = case["systems"] * 0.5 * (case["rows_min"] + case["rows_max"])
    return {"bytes": 40 * n, "flops": 8 * n}


# --------------------------------------------------------- the same in 64 bits

def _conv64(x, w):
    """3x3 zero-padded convolution, NHWC, w [9][cout][cin], in float64."""
    B, H, W, C = x.shape
    xp = torch.zeros((B, H + 2, W + 2, C), dtype=x.dtype, device=x.device)
    xp[:, 1:-1, 1:-1] = x
    y = 0
    for tap in range(9):
        dy, dx = tap // 3, tap % 3
        y = y + (xp[:, dy:dy + H, dx:dx + W].reshape(-1, C) @ w[tap].t()).reshape(B, H, W, -1)
    return y


def _net64(x8, params):
    a = torch.zeros(x8.shape[:3] + (32,), dtype=torch.float64, device=x8.device)
    a[..., :8] = x8
    a = torch.relu(_conv64(a, params[0][0]) + params[0][1])
    for w, b in params[1:-1]:
        a = a + torch.relu(_conv64(a, w) + b)
    return (_conv64(a, params[-1][0]) + params[-1][1])[..., :3]


def exact(case, seed):
    k = case["kind"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if k == "thomas":
        rows, off, A, B, C, D = _systems(case, seed)
        n, top = int(rows.sum()), int(rows.max())
        x, ap, bp = np.zeros(n), np.zeros(n), np.zeros(n)
        pa, pb = np.zeros(len(rows)), np.zeros(len(rows))
        for r in range(top):
            at = rows > r
            i = off[at] + r
            e = A[i] * pa[at] + B[i]
            pb[at] = (D[i] - A[i] * pb[at]) / e
            pa[at] = -C[i] / e
            ap[i], bp[i] = pa[at], pb[at]
        px = np.zeros(len(rows))
        for r in range(top - 1, -1, -1):
            at = rows > r
            i = off[at] + r
            px[at] = np.where(rows[at] - 1 == r, bp[i], bp[i] + ap[i] * px[at])
            x[i] = px[at]
        return x
    if k not in ("train", "forward"):
        return None      # FP64 throughout: 64 bits is what the case computes in
    params = [(torch.tensor(w, dtype=torch.float64, device=dev), torch.tensor(b, dtype=torch.float64, device=dev))
              for w, b in _weights(np.random.default_rng([seed, 12]))]
    d = torch.tensor([SCALES["d_u"], SCALES["d_v"], SCALES["d_z"]], dtype=torch.float64, device=dev)
    if k == "forward":
        x = torch.tensor(_images(case, seed), dtype=torch.float64, device=dev)
        with torch.no_grad():
            return (x[..., :3] + d * _net64(x, params)).cpu()
    xs, ys, ms = [], [], []
    for wet, h, now, then, q, zb in _states(case, seed):
        one = np.ones_like(h)
        ch = [np.where(wet, f, 0.0) for f in now] + [0.0 * one, 1.0 * wet, q / SCALES["s_q"] * one, zb * one,
                                                    h / SCALES["s_h"]]
        xs.append(np.stack(ch, -1))
        ys.append(np.stack([np.where(wet, f, 0.0) for f in then], -1))
        ms.append(1.0 * wet)
    x, y, m = (torch.tensor(np.stack(a), dtype=torch.float64, device=dev) for a in (xs, ys, ms))
    for w, b in params:
        w.requires_grad_(True)
        b.requires_grad_(True)
    e = (x[..., :3] + d * _net64(x.clamp(-8.0, 8.0), params) - y) / d
    loss = (m[..., None] * e * e).sum() / (3.0 * m.sum())
    loss.backward()
    return [float(loss.detach())] + [[w.grad.cpu(), b.grad.cpu()] for w, b in params]
