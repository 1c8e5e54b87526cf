"""The work that users of this framework have it do, as cases that can be timed.

Each case is one call sequence of a user's program through the public entry
points: the propagator (misfit and gradient of a shot, synthetic data, batches
of shots), the drop-in op API with its files, the learned preconditioner
(training step, inference) and its single layers through the C API. Sizes are
those of the benchmark workloads, the tests and the README, at fewer time steps
where a whole run would take seconds: every time step does the same work.

`exact` evaluates the same mathematics in float64 with plain torch.
"""
from __future__ import annotations

import ctypes as C
import json
import math
import os
import sys
import tempfile

import numpy as np
import torch
import torch.nn.functional as F

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "efwi-3d_amd"))

import FWI_ops_3d as ops  # noqa: E402
import fwi_utils  # noqa: E402
from efwi import _native as N  # noqa: E402
from efwi.propagator import GridSpec, Propagator, ShotSpec  # noqa: E402
from efwi.unet import UNet3D  # noqa: E402

DEV = "cuda:0"


# ---------------------------------------------------------------------------
# The cases.
# ---------------------------------------------------------------------------
def _gradient(name, nz, nx, ny, p, nt, step, **more):
    """Physical grid (without the C-PML's p cells per face), nt time steps, receivers every `step` cells."""
    return dict({"name": name, "kind": "gradient", "nz": nz, "nx": nx, "ny": ny, "npml": p, "nt": nt, "step": step,
                 "shots": 1, "formulation": 0, "every": 0, "resident": 0, "illum": False}, **more)


def listed():
    return [
        # the smallest grid a user tries the method on: kernels of a few microseconds, launches count
        _gradient("gradient-32", 32, 32, 32, 6, 120, 4),
        # the plain method's own workload, every surface cell a receiver, with the illumination that the learned
        # preconditioner reads: one evaluation of an inversion loop
        _gradient("gradient-64", 64, 64, 64, 10, 500, 1, illum=True),
        # the production stencil's grid: kernels of hundreds of microseconds, bound by memory
        _gradient("gradient-120x200x200", 120, 200, 200, 20, 150, 2),
        # the largest grid: the boundary ring of all steps does not fit there, early segments are replayed
        _gradient("gradient-ckpt-160x320x320", 160, 320, 320, 20, 49, 2, every=8, resident=3),
        # making observed data: the forward pass alone
        _gradient("synthetic-64x160x160", 64, 160, 160, 10, 500, 1, kind="synthetic"),
        # many shots of a small survey in one call (persistent launches), consistent formulation
        _gradient("batch-32-12shots", 32, 32, 32, 6, 120, 4, kind="batch", shots=12, formulation=1),
        # a few shots of the wide batched survey in one call
        _gradient("batch-64x160x160-4shots", 64, 160, 160, 10, 100, 2, kind="batch", shots=4),
        # a program written for the reference's op API: files, windows, autograd down to vp, vs, rho
        _gradient("dropin-64-2shots", 64, 64, 64, 10, 200, 2, kind="dropin", shots=2),
        # one training step of the preconditioner on a training pair of its own size
        {"name": "unet-train-96x128x128", "kind": "train", "nz": 96, "nx": 128, "ny": 128},
        # the preconditioner inside an inversion of the production grid
        {"name": "unet-infer-120x200x200", "kind": "infer", "nz": 120, "nx": 200, "ny": 200},
        # single layers, forward, input gradient and weight gradient: the full-resolution one (ragged rows) ...
        {"name": "layer-16to16-75x101x131", "kind": "layer", "nz": 75, "nx": 101, "ny": 131, "cin": 16, "cout": 16},
        # ... and the bottleneck's, where the volume is small
        {"name": "layer-64to64-24x32x32", "kind": "layer", "nz": 24, "nx": 32, "ny": 32, "cin": 64, "cout": 64},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gradient", "gradient", "gradient", "ckpt", "synthetic", "batch", "batch", "dropin", "train",
                       "infer", "layer", "layer"])
    if kind in ("train", "infer"):
        nz, nx, ny = (4 * rng.randint(lo, hi) for lo, hi in ((6, 30), (8, 50), (8, 50)))
        if kind == "train" and nz * nx * ny > 96 * 128 * 128:
            nz, nx, ny = nz // 8 * 4, nx // 8 * 4, ny
        return {"kind": kind, "nz": nz, "nx": nx, "ny": ny}
    if kind == "layer":
        cin, cout, lev = rng.choice([(16, 16, 1), (16, 16, 1), (48, 16, 1), (16, 32, 2), (32, 32, 2), (96, 32, 2),
                                     (32, 64, 4), (64, 64, 4)])
        lo, hi = (40, 110) if lev == 1 else (20, 60) if lev == 2 else (9, 34)
        return {"kind": kind, "nz": rng.randint(lo, hi), "nx": rng.randint(lo, hi), "ny": rng.randint(lo, hi + hi // 4),
                "cin": cin, "cout": cout}
    c = _gradient("", rng.randint(24, 128), rng.randint(24, 210), rng.randint(24, 210), rng.choice([6, 8, 10, 15, 20]),
                  _log_int(rng, 60, 400), rng.choice([1, 2, 3, 4]), kind="gradient" if kind == "ckpt" else kind)
    del c["name"]
    c["formulation"] = rng.choice([0, 0, 0, 1]) if kind != "dropin" else 0
    c["illum"] = kind == "gradient" and rng.random() < 0.4
    if kind == "ckpt":
        c["every"], c["resident"] = rng.randint(5, 16), rng.randint(1, 3)
    if kind == "batch":
        c["shots"] = rng.randint(3, 14)
        c["nz"], c["nx"], c["ny"] = (rng.randint(24, 56) for _ in range(3))
    if kind == "dropin":
        c["shots"] = rng.randint(1, 3)
        c["nz"], c["nx"], c["ny"] = (rng.randint(24, 72) for _ in range(3))
    # a drawn case costs at most what the production gradient does
    cells = math.prod(n + 2 * c["npml"] for n in (c["nz"], c["nx"], c["ny"])) * c["shots"]
    c["nt"] = max(30, min(c["nt"], int(9e8 / cells)))
    return c


# ---------------------------------------------------------------------------
# Inputs.
# ---------------------------------------------------------------------------
H, DT = 10.0, 1e-3


def _gen(seed, salt=0):
    return torch.Generator().manual_seed(int(seed) * 7919 + salt)


def _velocities(case, seed):
    """vp, vs (m/s) and rho (kg/m^3) of a seeded layered model with smooth lateral changes (physical grid)."""
    g = _gen(seed)
    nz, nx, ny = case["nz"], case["nx"], case["ny"]
    depth = torch.linspace(0.0, 1.0, nz, device=DEV).reshape(nz, 1, 1)
    edges, _ = torch.sort(torch.rand(3, generator=g) * 0.75 + 0.15)
    vps = torch.tensor([2000.0, 2500.0, 3000.0, 3500.0]) * (0.97 + 0.06 * torch.rand(4, generator=g))
    vp = torch.full((nz, 1, 1), float(vps[0]), device=DEV)
    for k in range(3):
        vp = torch.where(depth >= float(edges[k]), float(vps[k + 1]), vp)
    rough = torch.randn(1, 1, 4, 5, 5, generator=g).to(DEV)
    smooth = F.interpolate(rough, size=(nz, nx, ny), mode="trilinear", align_corners=True)[0, 0]
    vp = (vp * (1.0 + 0.02 * smooth.clamp(-2.5, 2.5))).contiguous()
    vs = (vp / 1.73).contiguous()
    return vp, vs, (310.0 * vp ** 0.25).contiguous()


def _pad(t, p):
    return F.pad(t[None, None], (p,) * 6, mode="replicate")[0, 0].contiguous()


def _lame(vp, vs, rho):
    r = rho / 1e3
    return (vp ** 2 - 2.0 * vs ** 2) * r, vs ** 2 * r, r


def _f0(case):
    return 15.0 if case["nt"] < 300 else 10.0


def _sources(case, seed):
    """Physical (z, x, y) of each shot."""
    g = _gen(seed, 1)
    return [(5, int(torch.randint(case["nx"] // 5, 4 * case["nx"] // 5, (1,), generator=g)),
             int(torch.randint(case["ny"] // 5, 4 * case["ny"] // 5, (1,), generator=g))) for _ in range(case["shots"])]


def _receivers(case):
    xs, ys = np.arange(0, case["nx"], case["step"]), np.arange(0, case["ny"], case["step"])
    gx, gy = np.meshgrid(xs, ys, indexing="ij")
    return np.stack([np.full(gx.size, 3), gx.ravel(), gy.ravel()], 1).astype(np.int32)


def _stf(case):
    f, t = _f0(case), np.arange(case["nt"]) * DT - 1.2 / _f0(case)
    e = (math.pi * f) ** 2
    return (np.cumsum((1 - 2 * e * t ** 2) * np.exp(-e * t ** 2)) * DT).astype(np.float32)


def _recorded(case, seed, src, k):
    """Recorded data of shot k, [3][nrec][nt] (x, y, z): the direct P wave of the source in a homogeneous rock, with
    1 % noise."""
    g = _gen(seed, 100 + k)
    alpha, rho = 2050.0, 2.1
    rec = torch.from_numpy(_receivers(case)).to(DEV).double()
    d = (rec - torch.tensor(src, device=DEV, dtype=torch.float64)) * H
    r = d.norm(dim=1).clamp_min(H)
    f = _f0(case)
    e = (math.pi * f) ** 2
    t = torch.arange(case["nt"], device=DEV, dtype=torch.float64) * DT - 1.2 / f
    t = t[None] - r[:, None] / alpha
    w = torch.exp(-e * t * t)
    s, ds = t * w, (1 - 2 * e * t * t) * w
    vr = -(1500.0 ** 2 * H ** 3 / (4 * math.pi * rho * alpha ** 2)) * (s / r[:, None] ** 2 + ds / (alpha * r[:, None])) * 0.7
    out = torch.stack([vr * (d[:, i] / r)[:, None] for i in (1, 2, 0)]).float()
    noise = torch.randn(3, 1, case["nt"], generator=g).to(DEV)
    return (out + 0.01 * out.abs().max() * noise).contiguous()


def _grid(case):
    p = case["npml"]
    every = case["every"]
    return GridSpec(case["nz"] + 2 * p, case["nx"] + 2 * p, case["ny"] + 2 * p, p, case["nt"], H, H, H, DT, _f0(case),
                    case["formulation"], memory_mode=1 if every else 0, checkpoint_every=every)


def _windows(case, k):
    """Window start and end (s), trace weights and source weight of a drop-in shot."""
    n, t = len(_receivers(case)), case["nt"] * DT
    return (np.linspace(0.0, 0.2 * t, n).astype(np.float32), np.linspace(0.9 * t, 0.99 * t, n).astype(np.float32),
            np.linspace(0.5, 1.5, n).astype(np.float32), np.float32(0.8 + 0.1 * k))


def _prepare_dropin(case, seed):
    folder = tempfile.TemporaryDirectory(prefix="fwi_case_")
    p, src, rec = case["npml"], _sources(case, seed), _receivers(case)
    para, survey, data = (os.path.join(folder.name, n) for n in ("para.json", "survey.json", "Data"))
    fwi_utils.paraGen_3d(case["nz"] + 2 * p, case["nx"] + 2 * p, case["ny"] + 2 * p, H, H, H, case["nt"], DT, _f0(case), p,
                         para, survey, data, if_win=True)
    shots = {"nShots": len(src)}
    for k, s in enumerate(src):
        w = _windows(case, k)
        shots[f"shot{k}"] = {"z_src": s[0], "x_src": s[1], "y_src": s[2], "nrec": len(rec), "z_rec": rec[:, 0].tolist(),
                             "x_rec": rec[:, 1].tolist(), "y_rec": rec[:, 2].tolist(), "win_start": w[0].tolist(),
                             "win_end": w[1].tolist(), "weights": w[2].tolist(), "src_weight": float(w[3])}
        for c, a in zip("xyz", _recorded(case, seed, s, k).cpu().numpy()):
            a.tofile(os.path.join(data, f"Shot_{c}{k}.bin"))
    with open(survey, "w") as fp:
        json.dump(shots, fp)
    vp, vs, rho = (t.requires_grad_(True) for t in _velocities(case, seed))
    opt = {"nz": case["nz"], "nx": case["nx"], "ny": case["ny"], "nPml": p, "para_fname": para}
    stf = torch.from_numpy(np.stack([_stf(case)] * len(src)))
    return {"folder": folder, "model": ops.FWI_3d(vp, vs, rho, stf, opt), "ids": torch.arange(len(src))}


def _layer_inputs(case, seed):
    """A layer's input activations, weights, bias and the gradient of its pre-activations: BF16 values as they come
    out of a ReLU layer and of the loss."""
    g = torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 5)
    V, ci, co = case["nz"] * case["nx"] * case["ny"], case["cin"], case["cout"]
    src = torch.randn(V, ci, generator=g, device=DEV).clamp_min_(0).bfloat16()
    w = (torch.randn(27, co, ci, generator=g, device=DEV) * math.sqrt(2.0 / (27 * ci))).bfloat16()
    b = torch.randn(co, generator=g, device=DEV) * 0.1
    d = torch.randn(V, co, generator=g, device=DEV)
    d = (d * (torch.rand(V, co, generator=g, device=DEV) < 0.5) * 1e-3).bfloat16()
    return src, w, b, d


# name, input channels, output channels, level of the network's convolutions
_NET = [("enc1a", 16, 16, 1), ("enc1b", 16, 16, 1), ("enc2a", 16, 32, 2), ("enc2b", 32, 32, 2), ("bot_a", 32, 64, 3),
        ("bot_b", 64, 64, 3), ("dec2a", 96, 32, 2), ("dec2b", 32, 32, 2), ("dec1a", 48, 16, 1), ("dec1b", 16, 16, 1)]


def _net_inputs(case, seed):
    """Weights (a checkpoint's), the input volume and the training target."""
    g = _gen(seed, 9)
    sd = {}
    for name, ci, co, _ in _NET:
        w = torch.randn(27, co, ci, generator=g) * math.sqrt(2.0 / (27 * (2 if name == "enc1a" else ci)))
        if name == "enc1a":
            w[:, :, 2:] = 0.0
        sd[name + ".w"], sd[name + ".b"] = w, torch.randn(co, generator=g) * 0.05
    sd["head.w"], sd["head.b"] = torch.randn(16, generator=g) * 0.05, torch.zeros(1)
    dims = (case["nz"], case["nx"], case["ny"])
    V = math.prod(dims)
    rough = torch.randn(1, 3, *(max(2, n // 4) for n in dims), generator=g).to(DEV)
    vol = F.interpolate(rough, size=dims, mode="trilinear", align_corners=True)[0].reshape(3, V)
    feat = torch.zeros(V, 16, device=DEV)
    feat[:, 0] = vol[0] / vol[0].abs().max()
    feat[:, 1] = torch.log10(vol[1] ** 2 / (vol[1] ** 2).max() + 1e-6) / 6 + 1
    return sd, dims, feat.bfloat16(), (1.5 + vol[2]).contiguous()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dropin":
        return dict(_prepare_dropin(case, seed), kind=kind)
    if kind == "layer":
        src, w, b, d = _layer_inputs(case, seed)
        dims = (case["nz"], case["nx"], case["ny"])
        L, ci, co, V = N.lib(), case["cin"], case["cout"], src.shape[0]
        s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        wt = torch.empty(27, ci, co, dtype=torch.bfloat16, device=DEV)
        assert L.efwi_nn_flip_weights(w.data_ptr(), ci, co, wt.data_ptr(), s) == 0
        bricks = L.efwi_nn_wgrad_scratch(co, ci, *dims, 1) // (27 * co * ci + co)
        per = int(min(24, max(2, bricks * (co // 16) * (ci // 16) // 768)))
        scratch = torch.empty(L.efwi_nn_wgrad_scratch(co, ci, *dims, per), device=DEV)
        new = lambda *n, t=torch.bfloat16: torch.empty(*n, dtype=t, device=DEV)  # noqa: E731
        return dict(kind=kind, case=case, src=src, w=w, b=b, d=d, wt=wt, per=per, scratch=scratch, dims=dims,
                    out=new(V, co), din=new(V, ci), dw=new(27, co, ci, t=torch.float32), db=new(co, t=torch.float32))
    if kind in ("train", "infer"):
        sd, dims, feat, target = _net_inputs(case, seed)
        net = UNet3D(0, seed=0)
        net.load_state_dict(sd)
        return {"kind": kind, "net": net, "dims": dims, "feat": feat, "target": target, "mask": torch.ones_like(target)}
    p = case["npml"]
    model = _lame(*(_pad(t, p) for t in _velocities(case, seed)))
    prop = Propagator(_grid(case), 0)
    if case["resident"]:
        prop.set_resident_segments(case["resident"])
    if case["illum"]:
        prop.set_illumination(True)
    stf, rec = _stf(case), _receivers(case) + p
    src = _sources(case, seed)
    shots = [ShotSpec(tuple(i + p for i in s), stf, rec) for s in src]
    obs = None if kind == "synthetic" else [_recorded(case, seed, s, k) for k, s in enumerate(src)]
    return {"kind": kind, "prop": prop, "model": model, "shots": shots, "obs": obs, "illum": case["illum"]}


# ---------------------------------------------------------------------------
# One pass.
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "dropin":
        m = state["model"]
        m.zero_grad(set_to_none=True)
        loss = m(state["ids"])
        loss.backward()
        return {"loss": loss.detach(), "vp": m.Vp.grad, "vs": m.Vs.grad, "rho": m.Rho.grad}
    if kind == "layer":
        return _run_layer(state)
    if kind == "train":
        net = state["net"]
        loss = net.train_step(state["feat"], state["target"], state["mask"], state["target"].numel(), state["dims"], lr=1e-5,
                              log_scaling=True)
        return {"loss": loss, "grads": net.grads}
    if kind == "infer":
        net = state["net"]
        return {"update": net.forward(state["feat"], state["dims"]), "scaling": net.scaling_log(state["dims"])}
    prop = state["prop"]
    prop.set_model(*state["model"])  # an inversion's every evaluation has its own model
    if kind == "batch":
        misfits, _ = prop.run_batch(state["shots"], 1, state["obs"])
        return {"misfits": misfits, "grads": [prop.batch_gradient(k) for k in range(len(misfits))]}
    if kind == "synthetic":
        return prop.run_shot(state["shots"][0], 2)[1]
    prop.zero_gradient()
    j, syn, _ = prop.run_shot(state["shots"][0], 1, state["obs"][0], want_syn=True)
    out = {"misfit": j, "syn": syn, "grad": prop.gradient()}
    if state["illum"]:
        out["illum"] = prop.illumination()
    return out


def _run_layer(st):
    L, case, dims = N.lib(), st["case"], st["dims"]
    ci, co = case["cin"], case["cout"]
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    P = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    rc = L.efwi_nn_conv3(P(st["src"]), ci, ci, P(st["w"]), P(st["b"]), P(st["out"]), co, co, None, 0, *dims, 0, 1, s)
    rc |= L.efwi_nn_wgrad(P(st["d"]), co, co, P(st["src"]), ci, ci, P(st["scratch"]), st["scratch"].numel(), P(st["dw"]),
                          P(st["db"]), *dims, st["per"], s)
    rc |= L.efwi_nn_conv3(P(st["d"]), co, co, P(st["wt"]), None, P(st["din"]), ci, ci, P(st["src"]), ci, *dims, 0, 0, s)
    if rc:
        raise RuntimeError(f"layer call failed ({rc})")
    return {"out": st["out"], "din": st["din"], "dw": st["dw"], "db": st["db"]}


# ---------------------------------------------------------------------------
# Work of one pass.
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: a time step reads and writes each state array once (forward: 9 fields, 3 model arrays; backward: both
    wavefields on the interior, the adjoint one everywhere, 3 model arrays and 3 gradients); a layer reads its inputs
    and writes its outputs once. Operations: those of the difference formulas, or of the matrix products."""
    kind = case["kind"]
    if kind in ("train", "infer", "layer"):
        V = case["nz"] * case["nx"] * case["ny"]
        if kind == "layer":
            ci, co = case["cin"], case["cout"]
            return {"bytes": 2.0 * V * (4 * ci + 3 * co) + 27 * ci * co * 8.0, "flops": 3 * 54.0 * ci * co * V}
        fl = by = 0.0
        for name, ci, co, lev in _NET:
            v = V / 8 ** (lev - 1)
            passes = 1 if kind == "infer" else 2 if name == "enc1a" else 3
            fl += passes * 54.0 * ci * co * v
            by += passes * 2.0 * v * (ci + co)
        return {"bytes": by, "flops": fl}
    p = case["npml"]
    npad = float(math.prod(case[k] + 2 * p for k in ("nz", "nx", "ny")))
    nint = float(case["nz"] * case["nx"] * case["ny"])
    steps = (case["nt"] - 1) * case["shots"]
    back = kind != "synthetic"
    return {"bytes": steps * (84.0 * npad + back * (84.0 * npad + 96.0 * nint)),
            "flops": steps * (130.0 * npad + back * (150.0 * npad + 190.0 * nint))}


# ---------------------------------------------------------------------------
# The same results in float64.
# ---------------------------------------------------------------------------
def _profile(n, p, h, f0, dt):
    """1-D C-PML profiles (K, a, b on the grid, then on the half grid) of one axis."""
    d0 = -9.0 * 3000.0 * math.log(float(np.float32(0.0008))) / (2.0 * p * h)
    amax = math.pi * f0
    i = np.arange(n, dtype=np.float64)
    out = []
    for left, right in ((p - i, p - n + i), (p - i - 0.5, p - n + i + 0.5)):
        q = np.maximum(left, right) / p
        on = q >= 0
        q = np.where(on, q, 0.0)
        damp = np.where(on, d0 * (0.25 * q + 0.75 * q ** 8), 0.0)
        K = 1.0 + q ** 8
        alpha = np.where(on, np.maximum(amax * (1.0 - q), 0.0), 0.0)
        b = np.exp(-(damp / K + alpha) * dt)
        with np.errstate(invalid="ignore", divide="ignore"):
            a = np.where(np.abs(damp) > 1e-6, damp * (b - 1.0) / (K * (damp + K * alpha)), 0.0)
        out += [K, a, b]
    return out


class _Exact:
    """The staggered-grid elastic scheme with C-PML, its adjoint and the imaging conditions, on the whole grid."""

    V = ("vz", "vx", "vy")
    S = ("szz", "sxx", "sxz", "syy", "sxy", "syz")

    def __init__(self, case, model):
        self.form, self.p, self.nt = case["formulation"], case["npml"], case["nt"]
        self.lam, self.mu, rho = (t.double() for t in model)
        self.shape = tuple(self.lam.shape)
        self.byc = 1.0 / rho
        self.dt = float(np.float32(DT))
        box = tuple(slice(2, n - 2) for n in self.shape)
        self.box = box
        for k in ("lam", "mu", "byc"):
            setattr(self, k, getattr(self, k)[box])
        self.l2m = self.lam + 2.0 * self.mu
        self.prof, self.pml = [], []
        for ax, n in enumerate(self.shape):
            rows = [torch.from_numpy(r[2:n - 2]).to(DEV).reshape([-1 if a == ax else 1 for a in range(3)])
                    for r in _profile(n, self.p, H, _f0(case), self.dt)]
            self.prof.append(dict(zip(("K", "a", "b", "Kh", "ah", "bh"), rows)))
            i = torch.arange(2, n - 2, device=DEV).reshape([-1 if a == ax else 1 for a in range(3)])
            self.pml.append(((i < self.p) | (i > n - self.p - 1)).double())
        # the velocity update's x and y slabs start one cell later in the reference formulation
        self.vprof = [dict(q) for q in self.prof]
        if self.form == 0:
            for ax in (1, 2):
                at = self.shape[ax] - self.p - 2
                for key, one in (("a", 0.0), ("ah", 0.0), ("K", 1.0), ("Kh", 1.0)):
                    t = self.vprof[ax][key].clone()
                    t.view(-1)[at] = one
                    self.vprof[ax][key] = t
        p = self.p
        self.inner = tuple(slice(p, n - p) for n in self.shape)                # interior, in the grid
        self.inbox = tuple(slice(p - 2, n - p - 2) for n in self.shape)        # the same, in the box
        band = torch.zeros(self.shape, dtype=torch.bool, device=DEV)
        band[tuple(slice(p - 2, n - p + 2) for n in self.shape)] = True
        band[tuple(slice(p + 3, n - p - 3) for n in self.shape)] = False
        self.band = band.reshape(-1).nonzero().reshape(-1)

    def zeros(self):
        f = {k: torch.zeros(self.shape, dtype=torch.float64, device=DEV) for k in self.V + self.S}
        f["psi"] = {}
        return f

    def _at(self, f, ax, d, where=None):
        sl = list(where or self.box)
        sl[ax] = slice(sl[ax].start + d, sl[ax].stop + d)
        return f[tuple(sl)]

    def db(self, f, ax, where=None):
        A = lambda d: self._at(f, ax, d, where)  # noqa: E731
        return (9 / 8 * (A(0) - A(-1)) - 1 / 24 * (A(1) - A(-2))) / H

    def df(self, f, ax, where=None):
        A = lambda d: self._at(f, ax, d, where)  # noqa: E731
        return (9 / 8 * (A(1) - A(0)) - 1 / 24 * (A(2) - A(-1))) / H

    def dsxy_x(self, f, where=None):
        if self.form == 1:
            return self.db(f, 1, where)
        A = lambda d: self._at(f, 1, d, where)  # noqa: E731
        return (9 / 8 * (A(0) - A(-1)) - 1 / 24 * (A(-1) - A(-2))) / H

    def psi(self, W, name):
        if name not in W["psi"]:
            W["psi"][name] = torch.zeros(self.shape, dtype=torch.float64, device=DEV)
        return W["psi"][name]

    def cpml(self, W, name, d, q, half):
        e = "h" if half else ""
        m = self.psi(W, name)[self.box]
        m.mul_(q["b" + e]).add_(q["a" + e] * d)
        return d / q["K" + e] + m

    def v_derivatives(self, W, where=None):
        db, df = self.db, self.df
        return {"vz_z": db(W["vz"], 0, where), "vx_x": db(W["vx"], 1, where), "vy_y": db(W["vy"], 2, where),
                "vx_z": df(W["vx"], 0, where), "vx_y": df(W["vx"], 2, where), "vz_x": df(W["vz"], 1, where),
                "vz_y": df(W["vz"], 2, where), "vy_x": df(W["vy"], 1, where), "vy_z": df(W["vy"], 0, where)}

    def s_derivatives(self, W, where=None):
        db, df = self.db, self.df
        return {"szz_z": df(W["szz"], 0, where), "sxz_x": db(W["sxz"], 1, where), "syz_y": db(W["syz"], 2, where),
                "sxz_z": db(W["sxz"], 0, where), "sxx_x": df(W["sxx"], 1, where), "sxy_y": db(W["sxy"], 2, where),
                "syz_z": db(W["syz"], 0, where), "sxy_x": self.dsxy_x(W["sxy"], where), "syy_y": df(W["syy"], 2, where)}

    HALF_V = ("vx_z", "vx_y", "vz_x", "vz_y", "vy_x", "vy_z")
    HALF_S = ("szz_z", "sxx_x", "syy_y")

    def stress(self, W, amp):
        d = self.v_derivatives(W)
        for k in d:
            d[k] = self.cpml(W, k, d[k], self.prof["zxy".index(k[-1])], k in self.HALF_V)
        b, dt, lam, mu, l2m = self.box, self.dt, self.lam, self.mu, self.l2m
        W["szz"][b] += (l2m * d["vz_z"] + lam * (d["vx_x"] + d["vy_y"])) * dt
        W["sxx"][b] += (l2m * d["vx_x"] + lam * (d["vz_z"] + d["vy_y"])) * dt
        W["syy"][b] += (l2m * d["vy_y"] + lam * (d["vz_z"] + d["vx_x"])) * dt
        W["sxz"][b] += mu * (d["vx_z"] + d["vz_x"]) * dt
        W["sxy"][b] += mu * (d["vx_y"] + d["vy_x"]) * dt
        W["syz"][b] += mu * (d["vy_z"] + d["vz_y"]) * dt
        for k in ("szz", "sxx", "syy"):
            W[k][self.src] += amp

    def velocity(self, W):
        d = self.s_derivatives(W)
        for k in d:
            d[k] = self.cpml(W, k, d[k], self.vprof["zxy".index(k[-1])] if k[-1] != "z" else self.prof[0], k in self.HALF_S)
        b, c = self.box, self.byc * self.dt
        W["vz"][b] += (d["szz_z"] + d["sxz_x"] + d["syz_y"]) * c
        W["vx"][b] += (d["sxz_z"] + d["sxx_x"] + d["sxy_y"]) * c
        W["vy"][b] += (d["syz_z"] + d["sxy_x"] + d["syy_y"]) * c

    def velocity_adjoint(self, A):
        """-(transposed difference) of the adjoint stresses, with the memory terms; then the velocity memories."""
        q, dt, b = self.prof, self.dt, self.box
        lam, mu, l2m = self.lam, self.mu, self.l2m
        ax = {"z": 0, "x": 1, "y": 2}
        new = {}
        for i in "xzy":
            j, k = [o for o in "xzy" if o != i]
            P = q[ax[i]]
            sij = lambda m, n: "s" + (m + n if m + n in ("xz", "xy", "yz") else n + m)  # noqa: E731
            t = P["a"] * -self.df(self.psi(A, f"v{i}_{i}"), ax[i])
            t = t + (l2m * -self.df(A[f"s{i}{i}"], ax[i]) + lam * (-self.df(A[f"s{j}{j}"], ax[i]) - self.df(A[f"s{k}{k}"], ax[i]))) / P["K"] * dt
            for o in (j, k):
                Q = q[ax[o]]
                t = t + mu / Q["Kh"] * -self.db(A[sij(i, o)], ax[o]) * dt + Q["ah"] * -self.db(self.psi(A, f"v{i}_{o}"), ax[o])
            new[f"v{i}"] = A[f"v{i}"][b] + t
        for k, t in new.items():
            A[k][b] = t
        c = self.byc * dt
        # memory of d(s)/d(axis): fed by the velocity that the derivative updates; decay on the derivative's grid, but
        # for two that the reference formulation decays on the other one
        for name, v in (("sxx_x", "vx"), ("sxz_x", "vz"), ("sxy_x", "vy"), ("sxz_z", "vx"), ("szz_z", "vz"), ("syz_z", "vy"),
                        ("sxy_y", "vx"), ("syz_y", "vz"), ("syy_y", "vy")):
            a = ax[name[-1]]
            half = name in self.HALF_S
            if self.form == 0 and name in ("syz_z", "syy_y"):
                half = not half
            m = self.psi(A, name)[b]
            m.mul_(q[a]["bh" if half else "b"]).add_(c * new[v]).mul_(self.pml[a])

    def stress_adjoint(self, A):
        q, dt, b, byc = self.prof, self.dt, self.box, self.byc
        lam, mu, l2m = self.lam, self.mu, self.l2m
        ax = {"z": 0, "x": 1, "y": 2}
        new = {}
        for i, o in ("xz", "xy", "yz"):
            t = 0.0
            for d, v in ((i, o), (o, i)):
                P = q[ax[d]]
                t = t + P["a"] * -self.df(self.psi(A, f"s{i}{o}_{d}"), ax[d]) - self.df(A[f"v{v}"], ax[d]) / P["K"] * byc * dt
            new[f"s{i}{o}"] = A[f"s{i}{o}"][b] + t
        for i in "xzy":
            P = q[ax[i]]
            new[f"s{i}{i}"] = A[f"s{i}{i}"][b] + P["ah"] * -self.db(self.psi(A, f"s{i}{i}_{i}"), ax[i]) - byc * self.db(A[f"v{i}"], ax[i]) / P["Kh"] * dt
        for k, t in new.items():
            A[k][b] = t
        sum3 = {i: lam * (new["szz"] + new["sxx"] + new["syy"]) + 2.0 * mu * new[f"s{i}{i}"] for i in "xzy"}
        for i in "xzy":
            for d in "xzy":
                a, Q = ax[d], q[ax[d]]
                m = self.psi(A, f"v{i}_{d}")[b]
                if i == d:
                    m.mul_(Q["b"]).add_(sum3[i] * dt)
                else:
                    s = "s" + (i + d if i + d in ("xz", "xy", "yz") else d + i)
                    m.mul_(Q["bh"]).add_(new[s] * mu * dt)
                m.mul_(self.pml[a])

    def shot(self, src, stf, rec, obs, fac, grad, illum):
        """src, rec on the padded grid; obs [3][nrec][nt]; fac [nrec or 1][nt]."""
        nt, dt, p = self.nt, self.dt, self.p
        self.src = src
        cells = (rec[:, 0] * self.shape[1] + rec[:, 1]) * self.shape[2] + rec[:, 2]
        W = self.zeros()
        syn = torch.zeros(3, len(cells), nt, dtype=torch.float64, device=DEV)
        amp = [2250000.0 * float(stf[it]) * dt for it in range(nt)]
        save = []
        light = torch.zeros(self.shape, dtype=torch.float64, device=DEV) if illum else None
        for it in range(nt - 1):
            if grad:
                save.append(torch.stack([W[k].reshape(-1)[self.band] for k in self.V + self.S]))
            self.stress(W, amp[it])
            self.velocity(W)
            for c, k in enumerate(("vx", "vy", "vz")):
                syn[c, :, it + 1] = W[k].reshape(-1)[cells]
            if illum:
                light += W["vz"] ** 2 + W["vx"] ** 2 + W["vy"] ** 2
        if not grad:
            return syn
        e = (obs.double() - syn) * fac
        e[:, :, 0] = 0.0
        misfit = float((e * e).sum())
        res = e * fac
        A = self.zeros()
        g = [torch.zeros(self.shape, dtype=torch.float64, device=DEV) for _ in range(3)]
        I, J = self.inner, self.inbox
        lam, mu, l2m, byc = (t[J] for t in (self.lam, self.mu, self.l2m, self.byc))

        def inject(it):
            for c, k in enumerate(("vx", "vy", "vz")):
                A[k].view(-1).index_add_(0, cells, res[c, :, it].contiguous())

        inject(nt - 1)
        self.stress_adjoint(A)
        for it in range(nt - 2, -1, -1):
            d = self.s_derivatives(W, I)
            r = {"vz": d["szz_z"] + d["sxz_x"] + d["syz_y"], "vx": d["sxz_z"] + d["sxx_x"] + d["sxy_y"],
                 "vy": d["syz_z"] + d["sxy_x"] + d["syy_y"]}
            g[2][I] += sum(A[k][I] * r[k] for k in self.V) * dt * byc * byc
            for k in self.V:
                W[k][I] -= r[k] * byc * dt
            self.velocity_adjoint(A)
            slot = save.pop()
            for n, k in enumerate(self.V):
                W[k].view(-1)[self.band] = slot[n]
            inject(it)
            for k in ("szz", "sxx", "syy"):
                W[k][src] -= amp[it]
            d = self.v_derivatives(W, I)
            div = d["vz_z"] + d["vx_x"] + d["vy_y"]
            g[0][I] -= (A["szz"][I] + A["sxx"][I] + A["syy"][I]) * div * dt
            xz, yz, xy = d["vx_z"] + d["vz_x"], d["vy_z"] + d["vz_y"], d["vy_x"] + d["vx_y"]
            g[1][I] -= (2.0 * (A["szz"][I] * d["vz_z"] + A["sxx"][I] * d["vx_x"] + A["syy"][I] * d["vy_y"]) + A["sxz"][I] * xz +
                        A["syz"][I] * yz + A["sxy"][I] * xy) * dt
            for k, own, o1, o2 in (("szz", "vz_z", "vx_x", "vy_y"), ("sxx", "vx_x", "vz_z", "vy_y"), ("syy", "vy_y", "vz_z", "vx_x")):
                W[k][I] -= (l2m * d[own] + lam * (d[o1] + d[o2])) * dt
            W["sxz"][I] -= mu * xz * dt
            W["sxy"][I] -= mu * xy * dt
            W["syz"][I] -= mu * yz * dt
            self.stress_adjoint(A)
            for n, k in enumerate(self.S):
                W[k].view(-1)[self.band] = slot[3 + n]
        return misfit, syn, g, light


def _taper(nt, t0, t3, ratio):
    """sin/cos ramps over `ratio` of [t0, t3] at both ends (t0, t3 arrays of one value per trace), squared."""
    t = np.arange(nt)[None] * DT
    t0, t3 = np.asarray(t0, np.float64)[:, None], np.asarray(t3, np.float64)[:, None]
    off = (t3 - t0) * ratio
    up, down = np.sin(math.pi / 2 * (t - t0) / off), np.cos(math.pi / 2 * (t - (t3 - off)) / off)
    w = np.where(t < t0 + off, up, np.where(t < t3 - off, 1.0, down))
    return np.where((t >= t0) & (t < t3), w, 0.0) ** 2


def _exact_wave(case, seed):
    p, kind, nt = case["npml"], case["kind"], case["nt"]
    vel = _velocities(case, seed)
    if kind == "dropin":
        vel = [t.double().requires_grad_(True) for t in vel]
        model = _lame(*(F.pad(t[None, None], (p,) * 6, mode="replicate")[0, 0] for t in vel))
    else:
        model = _lame(*(_pad(t, p) for t in vel))
    X = _Exact(case, [t.detach() for t in model])
    stf = _stf(case).astype(np.float64) * _taper(nt, [0.0], [nt * DT], 0.001)[0]
    rec = torch.from_numpy((_receivers(case) + p).astype(np.int64)).to(DEV)
    src = _sources(case, seed)
    outs = []
    for k, s in enumerate(src):
        at = tuple(i + p for i in s)
        if kind == "synthetic":
            return X.shot(at, stf, rec, None, None, False, False)
        if kind == "dropin":
            w = _windows(case, k)
            fac = _taper(nt, w[0], w[1], 0.005) * w[2].astype(np.float64)[:, None] * float(w[3])
        else:
            fac = _taper(nt, [0.0], [nt * DT], 0.005)
        outs.append(X.shot(at, stf, rec, _recorded(case, seed, s, k), torch.from_numpy(fac).to(DEV), True, case["illum"]))
    if kind == "batch":
        return {"misfits": [o[0] for o in outs], "grads": [tuple(o[2]) for o in outs]}
    if kind == "dropin":
        total = [sum(o[2][i] for o in outs) for i in range(3)]
        g = torch.autograd.grad(model, vel, grad_outputs=total)
        return {"loss": torch.tensor([sum(o[0] for o in outs)], dtype=torch.float64), "vp": g[0], "vs": g[1], "rho": g[2]}
    misfit, syn, g, light = outs[0]
    out = {"misfit": misfit, "syn": syn, "grad": tuple(g)}
    if case["illum"]:
        out["illum"] = light
    return out


def _shifted(x, dims, t, sign=1):
    """x [V][c] moved by tap t of a 3x3x3 window, zero outside."""
    v = F.pad(x.reshape(*dims, -1), (0, 0, 1, 1, 1, 1, 1, 1))
    o = [1 + sign * k for k in (t // 9 - 1, t // 3 % 3 - 1, t % 3 - 1)]
    return v[o[0]:o[0] + dims[0], o[1]:o[1] + dims[1], o[2]:o[2] + dims[2]].reshape(-1, x.shape[1])


def _conv(x, w, dims):
    return sum(_shifted(x, dims, t) @ w[t].T for t in range(27))


def _conv_back(d, x, w, dims):
    """(input gradient, weight gradient) of _conv."""
    return sum(_shifted(d, dims, t, -1) @ w[t] for t in range(27)), torch.stack([d.T @ _shifted(x, dims, t) for t in range(27)])


class _Conv3(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w, dims):
        ctx.save_for_backward(x, w)
        ctx.dims = dims
        return _conv(x, w, dims)

    @staticmethod
    def backward(ctx, d):
        return (*_conv_back(d, *ctx.saved_tensors, ctx.dims), None)


def _exact_net(case, seed):
    sd, dims, feat, target = _net_inputs(case, seed)
    sd = {k: v.to(DEV).double().requires_grad_(case["kind"] == "train") for k, v in sd.items()}
    half = lambda d: tuple(n // 2 for n in d)  # noqa: E731
    layer = lambda n, x, d: torch.relu(_Conv3.apply(x, sd[n + ".w"], d) + sd[n + ".b"])  # noqa: E731

    def pool(x, d):
        h = half(d)
        return x.reshape(h[0], 2, h[1], 2, h[2], 2, -1).mean(dim=(1, 3, 5)).reshape(math.prod(h), -1)

    def up(x, d):
        h, c = half(d), x.shape[1]
        return x.reshape(h[0], 1, h[1], 1, h[2], 1, c).expand(h[0], 2, h[1], 2, h[2], 2, c).reshape(-1, c)

    d2 = half(dims)
    d3 = half(d2)
    x = feat.double()
    e1 = layer("enc1b", layer("enc1a", x, dims), dims)
    e2 = layer("enc2b", layer("enc2a", pool(e1, dims), d2), d2)
    b3 = layer("bot_b", layer("bot_a", pool(e2, d2), d3), d3)
    u2 = layer("dec2b", layer("dec2a", torch.cat([up(b3, d2), e2], 1), d2), d2)
    u1 = layer("dec1b", layer("dec1a", torch.cat([up(u2, dims), e1], 1), dims), dims)
    o = u1 @ sd["head.w"] + sd["head.b"]
    if case["kind"] == "infer":
        return {"update": x[:, 0] * torch.exp(o.clamp(-4.0, 6.0)), "scaling": o.reshape(dims)}
    loss = ((o - target.double()) ** 2).mean()
    loss.backward()
    return {"loss": loss.detach().reshape(1), "grads": {k: v.grad for k, v in sd.items()}}


def exact(case, seed):
    kind = case["kind"]
    if kind == "layer":
        src, w, b, d = (t.double() for t in _layer_inputs(case, seed))
        dims = (case["nz"], case["nx"], case["ny"])
        din, dw = _conv_back(d, src, w, dims)
        return {"out": torch.relu(_conv(src, w, dims) + b), "din": din * (src > 0), "dw": dw, "db": d.sum(0)}
    if kind in ("train", "infer"):
        return _exact_net(case, seed)
    with torch.no_grad() if kind != "dropin" else torch.enable_grad():
        return _exact_wave(case, seed)
