"""The work that a user of this framework has it do, as measurable cases.

``listed`` names the cases, ``draw`` gives more of the same ranges, ``prepare``
makes what a program holds before the call, ``run`` is one pass through the
public entry points, ``work`` the bytes and operations a pass cannot do
without, ``exact`` the same outputs in 64 bits from plain torch.

Kinds of case:

* ``frame``     an interactive frame of the film simulation (GPUDrainageSimulator:
                ten fixed steps, then the thickness and surfactant on the host)
* ``simulate``  a whole simulation of one bubble, host field in, host field out
* ``render``    a large film stepped and rendered spectrally on the device
* ``export``    the images of a film from a moving camera: spectral RGB, the
                LUT-rendered RGBA8 frame and the caustic map, on the host
* ``lut``       the colour tables a renderer builds on start-up
* ``foam``      the films of many bubbles stepped together on the device
* ``cluster``   a foam cluster's contacts and motion
* ``advance``   the learned surrogate stepping a foam of settled films
* ``gradient``  loss and gradient of the surrogate on a host batch
* ``train``     online training windows of the surrogate on a foam
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from soap_bubble_simulation_amd import _lib as L
from soap_bubble_simulation_amd import export
from soap_bubble_simulation_amd import interference
from soap_bubble_simulation_amd.caustics import default_params as caustic_params
from soap_bubble_simulation_amd.cluster import FoamSimulator
from soap_bubble_simulation_amd.config import SimulationConfig
from soap_bubble_simulation_amd.drainage import DrainageContext, DrainageSimulator, GPUDrainageSimulator
from soap_bubble_simulation_amd.foam import FoamBubble, FoamDrainage, foam_params
from soap_bubble_simulation_amd.surrogate import FnoSurrogate

DEV = "cuda"
# Physics of the reference's defaults, used by the 64-bit evaluation.
RHO, GRAV, D_H, D_S = 1000.0, 9.81, 1e-9, 1e-9
N_FILM = 1.33
CAUSTIC_FOCAL = 2e6       # lenses of a film in metres: makes curvature visible


# ---------------------------------------------------------------------------
# The cases.

def listed():
    return [
        # The reference's interactive simulation at its default grid: the
        # smallest call, all latency.
        {"name": "frame_default", "kind": "frame", "nt": 64, "np": 128, "marangoni": False},
        # DrainageSimulator with its default configuration, fronts active.
        {"name": "simulate_default", "kind": "simulate", "nt": 128, "np": 256, "steps": 256, "flags": "tfe"},
        # An odd grid with every transport term and the diagnostics on.
        {"name": "simulate_ragged", "kind": "simulate", "nt": 500, "np": 1003, "steps": 48, "flags": "marangoni"},
        # The benchmark's film: large grid, spectral image of every step.
        {"name": "render_large", "kind": "render", "nt": 2048, "np": 4096, "steps": 8},
        # Still images of a film for export while the camera orbits.
        {"name": "export_frame", "kind": "export", "nt": 512, "np": 1024},
        # Colour tables: the reference's 1024 x 90 table and the renderer's LUT.
        {"name": "lut_tables", "kind": "lut", "nt": 1024, "np": 90},
        # A handful of small bubbles, and a foam that fills the card.
        {"name": "foam_small", "kind": "foam", "bubbles": 24, "lat_lo": 16, "lat_hi": 64, "steps": 64},
        {"name": "foam_large", "kind": "foam", "bubbles": 1024, "lat_lo": 32, "lat_hi": 512, "steps": 32},
        # Foam cluster dynamics with its contact list, at the benchmark's size.
        {"name": "cluster_4096", "kind": "cluster", "bubbles": 4096, "steps": 16},
        # The surrogate: inference on a foam, one gradient, online training.
        {"name": "surrogate_advance", "kind": "advance", "bubbles": 64, "nt": 256, "np": 512, "width": 32,
         "modes": 16, "layers": 4, "windows": 2},
        {"name": "surrogate_gradient", "kind": "gradient", "bubbles": 4, "nt": 128, "np": 512, "width": 32,
         "modes": 16, "layers": 4},
        {"name": "surrogate_train", "kind": "train", "bubbles": 16, "nt": 256, "np": 512, "width": 32,
         "modes": 16, "layers": 4, "windows": 2},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "simulate", "simulate", "render", "export", "lut", "foam", "foam", "cluster",
                       "advance", "gradient", "train"])
    if kind == "frame":
        nt = _log_int(rng, 24, 300)
        return {"kind": kind, "nt": nt, "np": 2 * nt + rng.randrange(0, 3), "marangoni": rng.random() < 0.5}
    if kind == "simulate":
        nt = _log_int(rng, 40, 1200)
        return {"kind": kind, "nt": nt, "np": 2 * nt + rng.randrange(0, 5), "steps": _log_int(rng, 16, 256),
                "flags": rng.choice(["tfe", "marangoni", "wgsl", "diag"])}
    if kind == "render":
        nt = _log_int(rng, 200, 2048)
        return {"kind": kind, "nt": nt, "np": 2 * nt, "steps": rng.randrange(1, 9)}
    if kind == "export":
        nt = _log_int(rng, 90, 1024)
        return {"kind": kind, "nt": nt, "np": 2 * nt + rng.randrange(0, 3)}
    if kind == "lut":
        return {"kind": kind, "nt": _log_int(rng, 64, 4096), "np": _log_int(rng, 16, 256)}
    if kind == "foam":
        lo = rng.choice([16, 24, 32, 48])
        return {"kind": kind, "bubbles": _log_int(rng, 6, 700), "lat_lo": lo,
                "lat_hi": _log_int(rng, lo + 8, 512), "steps": rng.randrange(8, 65)}
    if kind == "cluster":
        return {"kind": kind, "bubbles": _log_int(rng, 40, 10000), "steps": rng.randrange(4, 33)}
    nt, npf = rng.choice([(64, 128), (64, 256), (128, 256), (128, 512), (256, 512)])
    case = {"kind": kind, "bubbles": rng.randrange(2, 13), "nt": nt, "np": npf, "width": rng.choice([16, 32, 32]),
            "modes": rng.choice([8, 16]), "layers": rng.randrange(2, 5)}
    if kind != "gradient":
        case["windows"] = rng.randrange(1, 3)
    return case


# ---------------------------------------------------------------------------
# Inputs, from the seed alone (torch on the GPU, FP64, rounded where the
# entry point takes FP32).

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _film(nt, npf, seed, rel=0.05, noise=0.2, h0=None):
    """A film around h0 (drawn from 300-700 nm): smooth waves and grid noise."""
    g = _gen(seed)
    u = torch.rand(40, generator=g, device=DEV, dtype=torch.float64).cpu()
    if h0 is None:
        h0 = 300e-9 + 400e-9 * float(u[32])
    th = torch.arange(nt, device=DEV, dtype=torch.float64) * (math.pi / (nt - 1))
    ph = torch.arange(npf, device=DEV, dtype=torch.float64) * (2.0 * math.pi / npf)
    f = torch.zeros(nt, npf, device=DEV, dtype=torch.float64)
    for q in range(8):
        m = q % 5
        t = torch.cos((q + 1) * th + 6.28 * float(u[4 * q])) * torch.sin(th) ** m
        f += (float(u[4 * q + 1]) - 0.5) * t[:, None] * torch.cos(m * ph + 6.28 * float(u[4 * q + 2]))[None, :]
    f = f / f.abs().max()
    w = 2.0 * torch.rand(nt, npf, generator=g, device=DEV, dtype=torch.float64) - 1.0
    return h0 * (1.0 + rel * ((1.0 - noise) * f + noise * w))


def _gamma(nt, npf, seed):
    """Surfactant around one half, 10 % waves, as FP32."""
    return (_film(nt, npf, seed + 5003, rel=0.1, noise=0.05, h0=0.5)).float()


def _cmf(seed):
    """Three smooth colour-matching curves over 380-780 nm."""
    rng = np.random.default_rng(seed + 17)
    centre = np.array([610.0, 550.0, 460.0]) + rng.uniform(-15.0, 15.0, 3)
    width = rng.uniform(25.0, 45.0, 3)
    lam = (380.0 + 5.0 * np.arange(81))[:, None]
    return (rng.uniform(0.8, 1.2, 3) * np.exp(-0.5 * ((lam - centre) / width) ** 2)).astype(np.float32)


def _camera(radius, frame):
    a = 0.9 + 0.1 * frame
    return (3.8 * radius * math.cos(a), 1.4 * radius, 3.8 * radius * math.sin(a))


def _cfl(nt, npf, radius, eta, h):
    """Forward-Euler stability limit of the film equation, s."""
    th = np.arange(1, nt - 1) * (math.pi / (nt - 1))
    s = np.abs(np.sin(th))
    dth, dph = math.pi / (nt - 1), 2.0 * math.pi / npf
    lam = (4.0 * max(D_H, D_S) * (1.0 / dth ** 2 + 1.0 / (s * s * dph * dph)) / radius ** 2
           + 3.0 * RHO * GRAV / (3.0 * eta) * s * h * h)
    return 2.0 / float(lam.max())


def _bubbles(case, seed):
    """Bubble descriptions of a foam case; the grids belong to the case."""
    rng = np.random.default_rng(seed + 31)
    n = case["bubbles"]
    if "lat_lo" in case:
        u = np.random.default_rng(n).uniform(math.log(case["lat_lo"]), math.log(case["lat_hi"]), n)
        nt = np.rint(np.exp(u)).astype(int)
        npf = 2 * nt
    else:
        nt, npf = np.full(n, case["nt"]), np.full(n, case["np"])
    radius = np.exp(rng.uniform(math.log(2.5e-3), math.log(25e-3), n))
    h0 = rng.uniform(200e-9, 1000e-9, n)
    eta = rng.uniform(1e-3, 5e-3, n)
    return [dict(n_theta=int(nt[k]), n_phi=int(npf[k]), bubble_radius=float(radius[k]), viscosity=float(eta[k]),
                 h0=float(h0[k])) for k in range(n)]


def _foam_state(bubbles, offsets, seed, rel):
    """Float-float thickness and surfactant of a foam in its layout."""
    total = int(offsets[-1])
    sizes = torch.tensor(np.diff(np.asarray(offsets)), device=DEV)
    h0 = torch.repeat_interleave(torch.tensor([b["h0"] for b in bubbles], device=DEV, dtype=torch.float64), sizes)
    g = _gen(seed + 7)
    h = h0 * (1.0 + rel * (2.0 * torch.rand(total, generator=g, device=DEV, dtype=torch.float64) - 1.0))
    hi = h.float()
    lo = (h - hi.double()).float()
    gam = 0.5 + 0.05 * (2.0 * torch.rand(total, generator=g, device=DEV) - 1.0)
    return hi, lo, gam


def _cluster(case, seed):
    """Positions, radii, velocities and film thicknesses of a cluster (FP32)."""
    n = case["bubbles"]
    box = 0.5 * (n / 4096.0) ** (1.0 / 3.0)
    rng = np.random.default_rng(seed + 41)
    pos = rng.uniform(-box / 2, box / 2, (n, 3)).astype(np.float32)
    r = np.exp(rng.uniform(math.log(2.5e-3), math.log(25e-3), n)).astype(np.float32)
    vel = rng.uniform(-0.02, 0.02, (n, 3)).astype(np.float32)
    th = rng.uniform(200.0, 1000.0, n).astype(np.float32)
    return pos, r, vel, th


def _net_params(case, seed):
    """Surrogate weights with the library's initial distribution, FP32."""
    w, mt, mp, layers = case["width"], 2 * case["modes"], case["modes"], case["layers"]
    rng = np.random.default_rng(seed + 53)
    parts = [rng.standard_normal(8 * w) / math.sqrt(8.0), 0.05 * rng.standard_normal(w)]
    for _ in range(layers):
        parts += [rng.standard_normal(w * w) / math.sqrt(w), 0.05 * rng.standard_normal(w),
                  rng.standard_normal(mt * mp * 2 * w * w) / (w * math.sqrt(2.0 * mt * mp))]
    parts += [0.1 * rng.standard_normal(2 * w) / math.sqrt(w), np.zeros(2)]
    return np.concatenate(parts).astype(np.float32)


def _batch(case, seed):
    shape = (case["bubbles"], case["nt"], case["np"])
    g = _gen(seed + 61)
    x = torch.randn(*shape, 8, generator=g, device=DEV)
    t = 0.5 * torch.randn(*shape, 2, generator=g, device=DEV)
    return x, t


SCALES = (0.05, 1e-4)     # surrogate input and target scales
TRAIN_LR = 1e-4
CONNECTIONS = 8           # contact records held per bubble (about 1.5 are met)
JUDGE_TOL = 1e-3


# ---------------------------------------------------------------------------
# What a program holds, and one pass.

class _Device:
    """A device buffer of the library seen by torch, which keeps the buffer's
    owner alive as long as a tensor refers to it."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (int(ptr), False),
                                         "strides": None, "version": 2}


def _view(owner, ptr, *shape):
    return torch.as_tensor(_Device(owner, ptr.value, shape), device=DEV)


def _flags_params(flags):
    """sf_params and (frozen-pole, transport) options of a simulate case."""
    p = L.Params()
    if flags == "wgsl":
        L.check(L.lib().sf_params_gpu_default(p))
        return p
    L.check(L.lib().sf_params_cpu_default(p))
    if flags == "marangoni":
        p.flags = L.FLAG_MARANGONI | L.FLAG_SURFACTANT | L.FLAG_POLES_AVG_GAMMA | L.FLAG_DIAG
    elif flags == "diag":
        p.flags = L.FLAG_TFE | L.FLAG_SURFACTANT | L.FLAG_DIAG
    return p


def _simulate_dt(case):
    # Marangoni coupling carries the film's Laplacian into the surfactant;
    # the smaller step keeps the grid noise from growing.
    return (0.1 if case["flags"] == "marangoni" else 0.5) * _cfl(case["nt"], case["np"], 0.025, 1e-3, 1e-6)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "frame": 0}
    if kind == "frame":
        nt, npf = case["nt"], case["np"]
        sim = GPUDrainageSimulator(500e-9, npf, nt)
        sim.enabled = True
        if case["marangoni"]:
            sim.set_marangoni_enabled(True)
        sim.ctx.set_fields_f32(_film(nt, npf, seed).float().cpu().numpy(), _gamma(nt, npf, seed).cpu().numpy())
        s["sim"] = sim
    elif kind == "simulate":
        nt, npf = case["nt"], case["np"]
        if case["flags"] == "tfe" and npf == 2 * nt:
            s["sim"] = DrainageSimulator(SimulationConfig(resolution=nt))
        else:
            s["sim"] = DrainageSimulator(params=_flags_params(case["flags"]), n_theta=nt, n_phi=npf,
                                         initial_thickness=500e-9)
        s["h"] = _film(nt, npf, seed).cpu().numpy()
        s["g"] = _gamma(nt, npf, seed).double().cpu().numpy()
        s["dt"] = _simulate_dt(case)
    elif kind in ("render", "export"):
        nt, npf = case["nt"], case["np"]
        p = L.Params()
        L.check(L.lib().sf_params_cpu_default(p))
        p.flags = L.FLAG_TFE | L.FLAG_SURFACTANT | L.FLAG_DIAG
        ctx = DrainageContext(p, nt, npf, 500e-9, 0.5)
        ctx.set_fields(_film(nt, npf, seed, rel=0.1, noise=0.02).cpu().numpy(), _gamma(nt, npf, seed).cpu().numpy())
        s.update(ctx=ctx, radius=p.bubble_radius, cmf=_cmf(seed), dt=_cfl(nt, npf, p.bubble_radius, 1e-3, 1e-6))
        cp = caustic_params()
        cp.focal_length = CAUSTIC_FOCAL
        s["caustic"] = cp
        if kind == "render":
            s["stream"] = torch.cuda.ExternalStream(ctx.stream())
    elif kind == "lut":
        rng = np.random.default_rng(seed)
        s["index"] = float(rng.uniform(1.30, 1.40))
        s["tmax"] = float(rng.uniform(900.0, 1500.0))
    elif kind == "foam":
        bub = _bubbles(case, seed)
        s["foam"] = FoamDrainage(foam_params(), [FoamBubble(**b) for b in bub])
        s["state"] = _foam_state(bub, s["foam"].offsets, seed, 0.05)
        _hold_foam(s)
    elif kind == "cluster":
        pos, r, vel, th = _cluster(case, seed)
        s["sim"] = FoamSimulator(pos, r, vel, th)
        n = case["bubbles"]
        arr = (L.ClusterBubble * n)()
        L.check(L.lib().sf_cluster_get_bubbles(s["sim"].handle, arr))
        s["array"] = arr
        s["out"] = (L.ClusterBubble * n)()
        s["conn"] = (L.ClusterConnection * (CONNECTIONS * n))()
    else:
        cfg = dict(n_theta=case["nt"], n_phi=case["np"], width=case["width"], modes_theta=case["modes"],
                   modes_phi=case["modes"], layers=case["layers"], max_batch=case["bubbles"])
        model = FnoSurrogate(**cfg)
        model.set_params(_net_params(case, seed))
        model.set_scales(*SCALES)
        s["model"] = model
        if kind == "gradient":
            x, t = _batch(case, seed)
            s["x"], s["t"] = x.cpu().numpy(), t.cpu().numpy()
        else:
            bub = _bubbles(case, seed)
            s["foam"] = FoamDrainage(foam_params(), [FoamBubble(**b) for b in bub])
            # a settled film for inference, the training films' grid noise else
            s["state"] = _foam_state(bub, s["foam"].offsets, seed, 2e-4 if kind == "advance" else 0.05)
            _hold_foam(s)
    return s


def _hold_foam(s):
    """The foam in its starting state, and its stream for torch."""
    torch.cuda.current_stream().synchronize()      # the state's arrays come from torch's stream
    st = C.c_void_p()
    L.check(L.lib().sf_foam_stream(s["foam"].handle, C.byref(st)))
    s["stream"] = torch.cuda.ExternalStream(st.value)
    _set_foam(s)


def _set_foam(s):
    hi, lo, g = s["state"]
    L.check(L.lib().sf_foam_set_state(s["foam"].handle, hi.data_ptr(), lo.data_ptr(), g.data_ptr()))


def _foam_out(s):
    """Thickness and surfactant of the foam for a consumer on the device."""
    foam = s["foam"]
    n = foam.length
    hi, lo, g = C.c_void_p(), C.c_void_p(), C.c_void_p()
    L.check(L.lib().sf_foam_device_state(foam.handle, C.byref(hi), C.byref(lo), C.byref(g)))
    with torch.cuda.stream(s["stream"]):
        return {"h": _view(foam, hi, n) + _view(foam, lo, n), "gamma": _view(foam, g, n)}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "frame":
        s["sim"].step(1.0 / 60.0)
        return {"h": s["sim"].current_thickness(), "gamma": s["sim"].concentration()}
    if kind == "simulate":
        sim = s["sim"]
        sim.reset(500e-9)
        sim.ctx.set_fields(s["h"], s["g"])
        sim.step_many(case["steps"], s["dt"])
        h, g = sim.ctx.fields()
        out = {"h": h, "gamma": g}
        if case["flags"] in ("marangoni", "diag"):
            out["mass"], out["dt_cfl"] = sim.ctx.history(case["steps"])
        return out
    if kind == "render":
        ctx, nt, npf = s["ctx"], case["nt"], case["np"]
        cam = L.Camera()
        for k, v in enumerate(_camera(s["radius"], 0)):
            cam.position[k] = v
        L.check(L.lib().sf_drainage_step_spectral(ctx.handle, case["steps"], s["dt"], C.byref(cam), N_FILM,
                                                  L.fptr(s["cmf"].reshape(-1))))
        rgb, hi, lo, g = C.c_void_p(), C.c_void_p(), C.c_void_p(), C.c_void_p()
        L.check(L.lib().sf_spectral_device_rgb(ctx.handle, C.byref(rgb)))
        L.check(L.lib().sf_drainage_device_fields(ctx.handle, C.byref(hi), C.byref(lo), C.byref(g)))
        with torch.cuda.stream(s["stream"]):
            h = _view(ctx, hi, nt, npf) + _view(ctx, lo, nt, npf)
        mass, cfl = ctx.history(case["steps"])
        return {"rgb": _view(ctx, rgb, 3, nt, npf), "h": h, "gamma": _view(ctx, g, nt, npf), "mass": mass,
                "dt_cfl": cfl}
    if kind == "export":
        cam = _camera(s["radius"], s["frame"])
        s["frame"] += 1
        return {"rgb": interference.spectral_rgb(s["ctx"], cam, s["cmf"], N_FILM),
                "frame": export.render_frame(s["ctx"], cam, N_FILM),
                "caustics": s["ctx"].caustics(s["caustic"])}
    if kind == "lut":
        calc = interference.InterferenceCalculator.new(s["index"])
        return {"table": calc.generate_2d_color_lookup_table_array(0.0, s["tmax"], case["nt"], case["np"]),
                "lut": interference.interference_lut_rgba8(s["index"], 1.0)}
    if kind == "foam":
        s["foam"].step(case["steps"])
        return _foam_out(s)
    if kind == "cluster":
        return _run_cluster(s)
    if kind == "gradient":
        loss, grad = s["model"].gradient(s["x"], s["t"])
        return {"loss": loss, "grad": grad}
    _set_foam(s)
    if kind == "advance":
        s["model"].advance_foam(s["foam"], case["windows"], JUDGE_TOL)
        return _foam_out(s)
    losses = s["model"].train_foam(s["foam"], case["windows"], TRAIN_LR)
    return {"losses": losses, "params": s["model"].params()}


def _run_cluster(s):
    lib, h, n = L.lib(), s["sim"].handle, s["case"]["bubbles"]
    L.check(lib.sf_cluster_set_bubbles(h, n, s["array"]))
    m = C.c_int32()
    L.check(lib.sf_cluster_num_connections(h, C.byref(m)))
    if m.value > len(s["conn"]):
        raise ValueError("more contacts than the list holds")
    L.check(lib.sf_cluster_get_connections(h, s["conn"]))
    s["sim"].step_many(s["case"]["steps"], 1e-3)
    L.check(lib.sf_cluster_get_bubbles(h, s["out"]))
    b = np.frombuffer(s["out"], np.float32).reshape(n, 11)
    c = np.frombuffer(s["conn"], np.float32).reshape(-1, 10)
    # what a view of the foam draws (a velocity is its bubble's last move over
    # the step, and where the contact force jumps it flips within rounding)
    return {"position": b[:, 1:4], "connections": m.value, "pairs": np.frombuffer(s["conn"], np.int32).reshape(-1, 10)[:, :2],
            "geometry": c[:, 2:]}


# ---------------------------------------------------------------------------
# Bytes and operations that a pass cannot do without: every input read once,
# every output written once, state between steps held at 4 bytes per field.

def _net_flops(case):
    """Products of one network pass per bubble (truncated DFTs, mixing, W)."""
    t, p, w, mt, mp = case["nt"], case["np"], case["width"], 2 * case["modes"], case["modes"]
    per_layer = t * p * (8.0 * mp * w + 2.0 * w * w) + 16.0 * t * mt * mp * w + 8.0 * mt * mp * w * w
    return case["layers"] * per_layer + t * p * (2.0 * 8 * w + 2.0 * 2 * w)


def _net_weights(case):
    w, mt, mp = case["width"], 2 * case["modes"], case["modes"]
    return 4.0 * (9 * w + case["layers"] * (w * w + w + mt * mp * 2 * w * w) + 2 * w + 2)


def work(case):
    kind = case["kind"]
    if kind in ("frame", "simulate"):
        n = case["nt"] * case["np"]
        steps = 10 if kind == "frame" else case["steps"]
        marangoni = case.get("marangoni") or case.get("flags") == "marangoni"
        return {"bytes": 16.0 * n * steps + 32.0 * n, "flops": (45.0 if marangoni else 35.0) * n * steps}
    if kind == "render":
        n = case["nt"] * case["np"]
        return {"bytes": case["steps"] * (16.0 + 12.0) * n, "flops": case["steps"] * (35.0 + 81 * 10.0) * n}
    if kind == "export":
        n = case["nt"] * case["np"]
        return {"bytes": n * (3 * 8.0 + 12.0 + 4.0 + 4.0), "flops": n * (81 * 10.0 + 40.0 + 45.0)}
    if kind == "lut":
        return {"bytes": 12.0 * case["nt"] * case["np"] + 65536.0,
                "flops": 3 * 40.0 * case["nt"] * case["np"] + 7 * 40.0 * 16384}
    if kind == "foam":
        n = sum(b["n_theta"] * b["n_phi"] for b in _bubbles(case, 0))
        return {"bytes": 16.0 * n * case["steps"] + 20.0 * n, "flops": 35.0 * n * case["steps"]}
    if kind == "cluster":
        n = case["bubbles"]
        return {"bytes": 64.0 * n * case["steps"], "flops": 13.0 * n * n * (case["steps"] + 0.5)}
    n = case["bubbles"] * case["nt"] * case["np"]
    act = 2.0 * case["width"]                          # a layer's activations in 16 bits
    if kind == "gradient":
        return {"bytes": n * (32.0 + 8.0 + 4 * act * case["layers"]) + 2 * _net_weights(case),
                "flops": 3 * case["bubbles"] * _net_flops(case)}
    steps = case["windows"] * (1 if kind == "advance" else 16)
    if kind == "advance":
        return {"bytes": case["windows"] * n * (12.0 + 2 * act * (case["layers"] - 1) + 16.0 + 16.0) + 16.0 * n * steps,
                "flops": case["windows"] * case["bubbles"] * _net_flops(case) + 35.0 * n * steps}
    return {"bytes": case["windows"] * (n * (32.0 + 8.0 + 4 * act * case["layers"]) + 7 * _net_weights(case))
            + 16.0 * n * steps,
            "flops": case["windows"] * 3 * case["bubbles"] * _net_flops(case) + 35.0 * n * steps}


# Largest relative error that another correct implementation at the same
# precision shows: about four times what the 64-bit evaluation was measured
# against the library over the ranges (noted beside each).
TOLERANCE = {
    "frame": {"rel": 1e-6, "max": 1e-5},                      # Γ 1.8e-7
    "simulate": {"rel": 1e-6, "max": 1e-5},                   # Γ 1.7e-7, h 1e-8
    "simulate marangoni": {"rel": 1.4e-5, "max": 3e-4},       # Γ 3.4e-6
    "render": {"rel": 4e-4, "max": 2e-3},                     # RGB 9.8e-5
    "export": {"rel": 4e-4, "max": 2e-3, "differ": 1e-3},     # RGB 9.9e-5; RGBA8 ties
    "lut": {"rel": 5e-5, "max": 2e-3, "differ": 0.0},         # 1.2e-5
    "foam": {"rel": 1e-6, "max": 1e-5},                       # Γ 1.3e-7
    "cluster": {"rel": 4e-5, "max": 2e-2},                    # positions 8.4e-6 (one flipped contact)
    "advance": {"rel": 4e-7, "max": 4e-6},                    # h 2.4e-8, Γ 4.3e-8
    "gradient": {"rel": 2e-2, "max": 0.5},                    # BF16 products: 7e-3
    "train": {"rel": 1.2e-2, "max": 0.9},                     # weights 3e-3 (Adam's step is a sign at first)
}


def tolerance(case):
    kind = case["kind"]
    return dict(TOLERANCE["simulate marangoni" if case.get("flags") == "marangoni" else kind])


# ---------------------------------------------------------------------------
# The same in 64 bits.

class _Film:
    """One bubble's (or a batch of equal bubbles') film equation, FP64."""

    def __init__(self, nt, npf, radius, eta, guard, marangoni=False, transport=True, copy_h=False, avg_g=False,
                 h_crit=10e-9):
        f64 = dict(device=DEV, dtype=torch.float64)
        self.nt, self.np = nt, npf
        self.dth, self.dph = math.pi / (nt - 1), 2.0 * math.pi / npf
        th = torch.arange(1, nt - 1, **f64) * self.dth
        s = torch.sin(th)
        s = torch.where(s.abs() < guard, torch.full_like(s, guard), s)
        self.sin, self.safe, self.cot = torch.sin(th)[:, None], s[:, None], (torch.cos(th) / s)[:, None]
        col = lambda v: torch.as_tensor(v, **f64).reshape(-1, 1, 1)     # noqa: E731  one value per bubble
        self.R, self.c = col(radius), RHO * GRAV / (3.0 * col(eta))
        self.marangoni, self.transport, self.copy_h, self.avg_g, self.crit = (marangoni, transport, copy_h, avg_g,
                                                                             h_crit)

    def lap(self, f):
        c, n, s = f[:, 1:-1], f[:, :-2], f[:, 2:]
        e, w = torch.roll(c, -1, 2), torch.roll(c, 1, 2)
        return ((s - 2.0 * c + n) / self.dth ** 2 + self.cot * (s - n) / (2.0 * self.dth)
                + (e - 2.0 * c + w) / (self.dph ** 2 * self.safe ** 2)) / self.R ** 2

    def step(self, h, g, dt):
        """One explicit step of h and Γ [bubbles][nt][np]."""
        c, cg = h[:, 1:-1], g[:, 1:-1]
        frozen = c < self.crit
        lap = self.lap(h)
        rate = D_H * lap - self.c * c ** 3 * self.sin
        if self.marangoni:
            gt = (g[:, 2:] - g[:, :-2]) / (2.0 * self.dth) / self.R
            gp = (torch.roll(cg, -1, 2) - torch.roll(cg, 1, 2)) / (2.0 * self.dph) / (self.R * self.safe)
            rate = rate + 0.01 * 0.045 * torch.sqrt(gt * gt + gp * gp) * c * c
        hn, gn = h.clone(), g
        hn[:, 1:-1] = torch.where(frozen, c, torch.clamp(c + dt * rate, min=0.0))
        if self.transport:
            grate = D_S * self.lap(g)
            if self.marangoni:
                grate = grate + 0.001 * lap * self.R ** 2 * cg
            gn = g.clone()
            gn[:, 1:-1] = torch.where(frozen, cg, torch.clamp(cg + dt * grate, 0.0, 1.0))
            if self.avg_g:
                gn[:, 0], gn[:, -1] = gn[:, 1].mean(1, keepdim=True), gn[:, -2].mean(1, keepdim=True)
        if not self.copy_h:
            hn[:, 0], hn[:, -1] = hn[:, 1].mean(1, keepdim=True), hn[:, -2].mean(1, keepdim=True)
        return hn, gn

    def mass_cfl(self, h):
        """Film volume and stability limit of one bubble."""
        th = np.arange(self.nt) * self.dth
        lo, hi = np.maximum(th - 0.5 * self.dth, 0.0), np.minimum(th + 0.5 * self.dth, math.pi)
        R = float(self.R)
        area = torch.as_tensor(R * R * (np.cos(lo) - np.cos(hi)) * self.dph, device=DEV)
        D = max(D_H, D_S)
        lam = (4.0 * D * (1.0 / self.dth ** 2 + 1.0 / (self.safe ** 2 * self.dph ** 2)) / R ** 2
               + 3.0 * float(self.c) * self.sin.abs() * h[0, 1:-1] ** 2)
        return float((h[0] * area[:, None]).sum()), 2.0 / float(lam.max())


class _Fronts:
    """Marginal-regeneration fronts (drainage.rs:395-477)."""

    def __init__(self, nt, npf, ratio=0.85, first=0.5, interval=2.0):
        self.th = np.arange(nt) * (math.pi / (nt - 1))
        self.ph = np.arange(npf) * (2.0 * math.pi / npf)
        self.time, self.next, self.interval, self.rate, self.fronts = 0.0, first, interval, (1.0 - ratio) * 0.5, []

    def apply(self, h, dt):
        self.next -= dt
        t = self.time
        if self.next <= 0.0:
            self.fronts.append([abs(math.sin(t * 7.89 + 1.23)) * 2.0 * math.pi, 0.3 + abs(math.sin(t * 3.21)) * 0.4,
                                0.05 + abs(math.cos(t * 5.67)) * 0.05, 0.0])
            self.fronts = self.fronts[-8:]
            self.next = self.interval * (0.5 + abs(math.sin(t * 12.345)))
        for f in self.fronts:
            f[3] = min(f[3] + f[2] * dt, math.pi / 2)
        self.fronts = [f for f in self.fronts if f[3] < math.pi / 2 * 0.95]
        inside = np.zeros((len(self.th), len(self.ph)), bool)
        for centre, width, _, extent in self.fronts:
            d = np.abs(self.ph - centre)
            d = np.where(d > math.pi, 2.0 * math.pi - d, d)
            inside |= (np.abs(self.th - math.pi / 2) <= extent)[:, None] & (d < width / 2.0)[None, :]
        self.time += dt
        if not inside.any():
            return h
        return torch.where(torch.as_tensor(inside, device=DEV), h * (1.0 - self.rate * dt), h)


def _exact_single(case, seed):
    """frame, simulate and render: (h, Γ, mass, cfl) after the pass."""
    nt, npf, kind = case["nt"], case["np"], case["kind"]
    if kind == "frame":
        film = _Film(nt, npf, 0.025, 1e-3, 1e-4, marangoni=case["marangoni"], copy_h=True, h_crit=30e-9)
        h, dt, steps, fronts = _film(nt, npf, seed).float().double(), float(np.float32(1e-3)), 10, None
    elif kind == "simulate":
        f = case["flags"]
        film = _Film(nt, npf, 0.025, 1e-3, 1e-4 if f == "wgsl" else 1e-10, marangoni=f == "marangoni",
                     transport=f != "tfe", copy_h=f == "wgsl", avg_g=f == "marangoni",
                     h_crit=30e-9 if f == "wgsl" else 10e-9)
        h, dt, steps = _film(nt, npf, seed), _simulate_dt(case), case["steps"]
        fronts = _Fronts(nt, npf) if f in ("tfe", "diag") else None
    else:
        film = _Film(nt, npf, 0.025, 1e-3, 1e-10)
        h, dt, steps = _film(nt, npf, seed, rel=0.1, noise=0.02), _cfl(nt, npf, 0.025, 1e-3, 1e-6), case["steps"]
        fronts = _Fronts(nt, npf)
    h, g = h[None], _gamma(nt, npf, seed).double()[None]
    hist = []
    for _ in range(steps):
        h, g = film.step(h, g, dt)
        if fronts:
            h = fronts.apply(h, dt)
        if kind == "render" or case.get("flags") in ("marangoni", "diag"):
            hist.append(film.mass_cfl(h))
    return h[0], g[0], [m for m, _ in hist], [c for _, c in hist]


def _view_terms(nt, npf, radius, cam):
    th = torch.arange(nt, device=DEV, dtype=torch.float64)[:, None] * (math.pi / (nt - 1))
    ph = torch.arange(npf, device=DEV, dtype=torch.float64)[None, :] * (2.0 * math.pi / npf)
    n = (torch.sin(th) * torch.cos(ph), torch.cos(th) + 0.0 * ph, torch.sin(th) * torch.sin(ph))
    v = [cam[k] - radius * n[k] for k in range(3)]
    length = torch.sqrt(v[0] ** 2 + v[1] ** 2 + v[2] ** 2)
    ci = ((v[0] * n[0] + v[1] * n[1] + v[2] * n[2]) / length).abs()
    ct = torch.sqrt(torch.clamp(1.0 - (1.0 - ci * ci) / N_FILM ** 2, min=0.0))
    rs = (ci - N_FILM * ct) / torch.clamp(ci + N_FILM * ct, min=1e-4)
    rp = (N_FILM * ci - ct) / torch.clamp(N_FILM * ci + ct, min=1e-4)
    refl = 0.5 * (rs * rs + rp * rp)
    return ct, 4.0 * refl / torch.clamp(1.0 - refl, min=1e-3) ** 2


def _exact_rgb(h, radius, cam, cmf):
    nt, npf = h.shape
    ct, F = _view_terms(nt, npf, radius, cam)
    opd = 2.0 * N_FILM * h * 1e9 * ct
    rgb = torch.zeros(3, nt, npf, device=DEV, dtype=torch.float64)
    cm = cmf.astype(np.float64)
    for k in range(81):
        fs = F * torch.cos(math.pi * opd / (380.0 + 5.0 * k)) ** 2      # sin(x + pi/2)
        a = fs / (1.0 + fs)
        for c in range(3):
            rgb[c] += float(cm[k, c]) / 81.0 * a
    return rgb


def _exact_caustics(h, focal, intensity=2.0, sharpness=1.5, threshold=0.001):
    up, dn = torch.cat([h[:1], h[:-1]]), torch.cat([h[1:], h[-1:]])
    w, e = (lambda f: torch.roll(f, 1, 1)), (lambda f: torch.roll(f, -1, 1))
    lap = w(h) + e(h) + up + dn - 4.0 * h
    det = (w(h) + e(h) - 2.0 * h) * (up + dn - 2.0 * h) - ((e(dn) - w(dn) - e(up) + w(up)) / 4.0) ** 2
    grad = torch.sqrt(((e(h) - w(h)) / 2.0) ** 2 + ((dn - up) / 2.0) ** 2)
    i = 1.0 / torch.clamp((1.0 + lap * focal).abs(), min=0.01)
    i = i * torch.where(det < -threshold, 1.5, 1.0) * (1.0 + 0.5 * grad)
    return torch.clamp(i ** sharpness * intensity, 0.0, 10.0)


def _exact_table(case, seed):
    rng = np.random.default_rng(seed)
    n, tmax = float(rng.uniform(1.30, 1.40)), float(rng.uniform(900.0, 1500.0))
    f64 = dict(device=DEV, dtype=torch.float64)
    d = torch.arange(case["nt"], **f64)[:, None] * (tmax / max(1, case["nt"] - 1))
    ci = torch.arange(case["np"], **f64)[None, :] / max(1, case["np"] - 1)
    ct = torch.sqrt(1.0 - (1.0 - ci * ci) / (n * n))
    refl = 0.5 * (((ci - n * ct) / (ci + n * ct)) ** 2 + ((n * ci - ct) / (n * ci + ct)) ** 2)
    out = []
    for lam in (650.0, 532.0, 450.0):
        cp = torch.cos(2.0 * math.pi * (2.0 * n * d * ct + lam / 2.0) / lam)
        v = 2.0 * refl * (1.0 - cp) / (1.0 + refl * refl - 2.0 * refl * cp)
        v = torch.where(refl >= 1.0 - 1e-12, torch.ones_like(v), v)      # grazing incidence: total reflection
        out.append(torch.where(d > 0.0, torch.clamp(v, 0.0, 1.0), torch.zeros_like(v)) ** (1.0 / 2.2))
    return torch.stack(out, dim=2)


def _steps_of(bubbles):
    """Each bubble's time step: the limit of its uniform film."""
    return [_cfl(b["n_theta"], b["n_phi"], b["bubble_radius"], b["viscosity"], b["h0"]) for b in bubbles]


def _layout(bubbles):
    """Offsets of the bubbles' fields: each starts at a multiple of 4 cells."""
    offs = [0]
    for b in bubbles:
        offs.append(offs[-1] + (b["n_theta"] * b["n_phi"] + 3) // 4 * 4)
    return np.array(offs, np.int64)


def _exact_foam(case, seed):
    bub = _bubbles(case, seed)
    if len(bub) * case["steps"] > 6000:
        return None
    offs = _layout(bub)
    hi, lo, g = _foam_state(bub, offs, seed, 0.05)
    h, g = hi.double() + lo.double(), g.double()
    for k, (b, dt) in enumerate(zip(bub, _steps_of(bub))):
        nt, npf = b["n_theta"], b["n_phi"]
        cells = slice(int(offs[k]), int(offs[k]) + nt * npf)
        film = _Film(nt, npf, b["bubble_radius"], b["viscosity"], 1e-10)
        hb, gb = h[cells].reshape(1, nt, npf), g[cells].reshape(1, nt, npf)
        for _ in range(case["steps"]):
            hb, gb = film.step(hb, gb, dt)
        h[cells], g[cells] = hb.reshape(-1), gb.reshape(-1)
    return {"h": h, "gamma": g}


def _exact_cluster(case, seed):
    p, r, v, t = (torch.as_tensor(a, device=DEV).double() for a in _cluster(case, seed))
    dt = float(np.float32(1e-3))
    s = r[:, None] + r[None, :]
    mass = torch.clamp(4.0 * math.pi * r * r * t * 1e-9 * 1000.0, min=1e-9)
    weight = 4.0 * math.pi * r * r * t * 1e-9 * 1000.0 * 9.81 - 4.0 / 3.0 * math.pi * r ** 3 * 1.2 * 9.81
    down = torch.tensor([0.0, -1.0, 0.0], device=DEV, dtype=torch.float64)
    for _ in range(case["steps"]):
        d2 = torch.zeros_like(s)
        for k in range(3):
            d2 += (p[None, :, k] - p[:, None, k]) ** 2
        dist = torch.sqrt(d2)
        ok = dist >= 1e-6
        dist = torch.where(ok, dist, torch.ones_like(dist))
        mag = torch.where((dist < 3.0 * s) & (dist > s), 0.001 * r[:, None] * r[None, :] / dist ** 2, 0.0)
        mag = mag - 5.0 * torch.clamp(s - dist, min=0.0) ** 1.5
        mag = mag + torch.where((dist < 1.2 * s) & (dist > 0.95 * s), 2.0 * (1.2 * s - dist), 0.0)
        mag = torch.where(ok, mag / dist, torch.zeros_like(mag))
        f = torch.stack([(mag * (p[None, :, k] - p[:, None, k])).sum(1) for k in range(3)], dim=1)
        f = f + down * torch.clamp(weight, min=0.0)[:, None] - v * (6.0 * math.pi * 0.001 * r)[:, None]
        v = (v + f / mass[:, None] * dt) * float(np.float32(0.8))
        speed = torch.sqrt((v * v).sum(1, keepdim=True))
        v = torch.where(speed > float(np.float32(0.1)), v * (float(np.float32(0.1)) / speed), v)
        p = p + v * dt
    return {"position": p, "connections": None, "pairs": None, "geometry": None}


class _Net:
    """The surrogate network in FP64 (FFT form)."""

    def __init__(self, case, seed):
        w, mt, mp = case["width"], 2 * case["modes"], case["modes"]
        self.case, self.w, self.mt, self.mp = case, w, mt, mp
        self.k = torch.tensor([k if k < mt // 2 else k - mt for k in range(mt)], device=DEV) % case["nt"]
        self.flat = torch.as_tensor(_net_params(case, seed), device=DEV).double()

    def parts(self, flat):
        w, o, out = self.w, 0, []
        sizes = [(8, w), (w,)]
        for _ in range(self.case["layers"]):
            sizes += [(w, w), (w,), (self.mt, self.mp, 2, w, w)]
        for shape in sizes + [(w, 2), (2,)]:
            n = math.prod(shape)
            out.append(flat[o:o + n].reshape(shape))
            o += n
        return out

    def forward(self, flat, x):
        p = self.parts(flat)
        nt, npf, layers = self.case["nt"], self.case["np"], self.case["layers"]
        x = x @ p[0] + p[1]
        for q in range(layers):
            W, b, R = p[2 + 3 * q:5 + 3 * q]
            X = torch.fft.rfft2(x, dim=(1, 2))[:, self.k][:, :, :self.mp]
            Y = torch.einsum("bkmc,kmco->bkmo", X, torch.complex(R[:, :, 0], R[:, :, 1]))
            rows = torch.zeros(x.shape[0], nt, self.mp, self.w, device=DEV, dtype=torch.complex128)
            rows = rows.index_copy(1, self.k, Y)
            full = torch.nn.functional.pad(rows, (0, 0, 0, npf // 2 + 1 - self.mp))
            z = x @ W + b + torch.fft.irfft2(full, s=(nt, npf), dim=(1, 2))
            x = torch.nn.functional.gelu(z, approximate="tanh") if q < layers - 1 else z
        return x @ p[-2] + p[-1]

    def gradient(self, flat, x, t):
        flat = flat.detach().requires_grad_(True)
        loss = ((self.forward(flat, x) - t) ** 2).mean()
        return float(loss.detach()), torch.autograd.grad(loss, flat)[0]


class _Windows:
    """Equal bubbles of a surrogate case and the network's features, FP64."""

    K = 16

    def __init__(self, case, seed, rel):
        self.bub = _bubbles(case, seed)
        nt, npf, n = case["nt"], case["np"], case["bubbles"]
        hi, lo, g = _foam_state(self.bub, _layout(self.bub), seed, rel)
        self.h, self.g = (hi.double() + lo.double()).reshape(n, nt, npf), g.double().reshape(n, nt, npf)
        col = lambda k: torch.tensor([b[k] for b in self.bub], device=DEV, dtype=torch.float64)     # noqa: E731
        self.R, self.eta = col("bubble_radius"), col("viscosity")
        self.dt = torch.tensor(_steps_of(self.bub), device=DEV, dtype=torch.float64)
        self.film = _Film(nt, npf, self.R, self.eta, 1e-10)
        self.sin = torch.sin(torch.arange(nt, device=DEV, dtype=torch.float64) * self.film.dth)

    def plain(self, h, g, steps):
        for _ in range(steps):
            h, g = self.film.step(h, g, self.dt[:, None, None])
        return h, g

    def scale(self, h, prev):
        """h_ref and the increment scale of every bubble."""
        href = h.mean(dim=(1, 2))
        y = href * SCALES[1]
        if prev is not None:
            r = torch.sqrt(((h - prev) ** 2).mean(dim=(1, 2)))
            y = torch.where(r > 1e-6 * y, r, y)
        return href, y

    def features(self, h, g, prev, href, y):
        one = torch.ones_like(h)
        b = lambda v: v[:, None, None]       # noqa: E731
        sink = self.K * self.dt * RHO * GRAV / (3.0 * self.eta) * href ** 2
        diff = self.K * self.dt * D_H / (self.R ** 2 * self.film.dth ** 2)
        lapped = lambda f: torch.nn.functional.pad(     # noqa: E731
            b(self.dt) * D_H * self.film.lap(f), (0, 0, 1, 1))
        d = torch.zeros_like(h) if prev is None else h - prev
        step = lapped(h)
        sunk = b(sink / self.K) * (h / b(href)) ** 3 * b(href) * self.sin[None, :, None]
        step[:, 1:-1] -= sunk[:, 1:-1]
        return torch.stack([(h / b(href) - 1.0) / SCALES[0], (g - 0.5) * 10.0, one * self.sin[None, :, None],
                            one * b(sink) * 1e6, one * b(diff), d / b(y), lapped(d) / b(y), step / b(y)], dim=3)


def _exact_advance(case, seed):
    net, win = _Net(case, seed), _Windows(case, seed, 2e-4)
    h, g, prev, K = win.h, win.g, None, _Windows.K
    for _ in range(case["windows"]):
        href, y = win.scale(h, prev)
        x = win.features(h, g, prev, href, y)
        out = torch.cat([net.forward(net.flat, part) for part in x.split(8)])
        del x
        d = torch.zeros_like(h) if prev is None else h - prev
        near = h + (K - 1) / K * d + out[..., 0] * y[:, None, None]
        prev = h
        h, g = win.plain(near, g, 1)
    return {"h": h.reshape(-1), "gamma": g.reshape(-1)}


def _exact_train(case, seed):
    net, win = _Net(case, seed), _Windows(case, seed, 0.05)
    h, g, prev, K = win.h, win.g, None, _Windows.K
    w = net.flat
    m, v, losses = torch.zeros_like(w), torch.zeros_like(w), []
    for t in range(1, case["windows"] + 1):
        ha, ga = win.plain(h, g, K - 1)
        hb, gb = win.plain(ha, ga, 1)
        href, y = win.scale(h, prev)
        x = win.features(h, g, prev, href, y)
        d = torch.zeros_like(h) if prev is None else h - prev
        target = torch.stack([ha - h - (K - 1) / K * d, hb - h - d], dim=3) / y[:, None, None, None]
        loss, grad = net.gradient(w, x, target)
        losses.append(loss)
        m, v = 0.9 * m + 0.1 * grad, 0.999 * v + 0.001 * grad * grad
        w = w - TRAIN_LR * math.sqrt(1.0 - 0.999 ** t) / (1.0 - 0.9 ** t) * m / (torch.sqrt(v) + 1e-8)
        prev, h, g = h, hb, gb
    return {"losses": torch.tensor(losses, dtype=torch.float64), "params": w}


def exact(case, seed):
    kind = case["kind"]
    if kind == "frame":
        h, g, _, _ = _exact_single(case, seed)
        return {"h": h, "gamma": g}
    if kind == "simulate":
        h, g, mass, cfl = _exact_single(case, seed)
        out = {"h": h, "gamma": g}
        if mass:
            out.update(mass=np.array(mass), dt_cfl=np.array(cfl))
        return out
    if kind == "render":
        h, g, mass, cfl = _exact_single(case, seed)
        return {"rgb": _exact_rgb(h, 0.025, _camera(0.025, 0), _cmf(seed)), "h": h, "gamma": g,
                "mass": np.array(mass), "dt_cfl": np.array(cfl)}
    if kind == "export":
        h = _film(case["nt"], case["np"], seed, rel=0.1, noise=0.02)
        return {"rgb": _exact_rgb(h, 0.025, _camera(0.025, 0), _cmf(seed)), "frame": None,
                "caustics": _exact_caustics(h, CAUSTIC_FOCAL)}
    if kind == "lut":
        return {"table": _exact_table(case, seed), "lut": None}
    if kind == "foam":
        return _exact_foam(case, seed)
    if kind == "cluster":
        return _exact_cluster(case, seed)
    if kind == "gradient":
        x, t = _batch(case, seed)
        loss, grad = _Net(case, seed).gradient(_Net(case, seed).flat, x.double(), t.double())
        return {"loss": loss, "grad": grad}
    return _exact_advance(case, seed) if kind == "advance" else _exact_train(case, seed)
