"""The calls whose speed this repository is measured by.

Each case is one pass through a public entry point, as a program that
reconstructs, trains through or prepares cone-beam scans calls it: whole
reconstructions through the engine (device-resident and from host memory),
training steps of the differentiable form, the stage-level calls on a block of
projections, the Scanco RSQ preprocessing and the 16-bit export.  Sizes are
those of the named workloads (tomokvas_amd.geometry.workloads) and of the
tests, plus odd ones.

listed() gives the named cases, draw() more of the same ranges, prepare() what
a program holds before the call, run() one pass, work() the bytes and
operations a pass cannot do without, exact() its outputs in 64 bits from plain
torch.
"""
from __future__ import annotations

import ctypes as C
import math
import random

import numpy as np
import torch

from tomokvas_amd import _lib, diff, geometry
from tomokvas_amd._hip import hip
from tomokvas_amd.engine import FilteredBackProjection, VolumeSink
from tomokvas_amd.stages import Stages

STORE = {"f32": _lib.F32, "f16": _lib.F16, "bf16": _lib.BF16, "f16p": _lib.F16_PACKED,
         "f64": _lib.F64}
BYTES = {"f32": 4, "f16": 2, "bf16": 2, "f16p": 2, "f64": 8}
RSQ_BH = (-0.8, 0.02)          # beam-hardening line A, B


def _scan(kind, nx, ny, nz, nu, nv, nang, scale, dist, store="f32", filt="ramlak", block=0,
          ang0=0, chunk=0, crop=0, shift=0.0):
    """A scan: volume nx x ny x nz of voxels of `scale` virtual pixels from nang
    projections of nu x nv samples, source at `dist` virtual pixels; block,
    ang0: the projections a stage-level call takes (0: all); chunk: projections
    per chunk of a training step (0: whole); crop: edge of the central cube that
    carries the gradient (0: all); shift: rotation axis off the middle column."""
    return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "nu": nu, "nv": nv, "nang": nang,
            "scale": scale, "dist": dist, "store": store, "filt": filt, "block": block,
            "ang0": ang0, "chunk": chunk, "crop": crop, "shift": shift}


def listed():
    return [
        # one small reconstruction, projections already in device memory: the
        # 128^3 workload, where launches and idle CUs count
        {"name": "fdk-128-f32", **_scan("fdk", 128, 128, 128, 128, 128, 180, 1.0, 2500.0)},
        # odd sizes in every dimension, axis off the middle column, BF16 storage
        {"name": "fdk-ragged-bf16", **_scan("fdk", 203, 190, 157, 300, 219, 251, 1.375, 1100.0,
                                            "bf16", shift=-1.5)},
        # an ordinary laboratory scan: the 512^3 workload, FP16 storage
        {"name": "fdk-512-f16", **_scan("fdk", 512, 512, 512, 1024, 1024, 900, 2.0, 10000.0,
                                        "f16", "shepplogan")},
        # the largest whole reconstruction: 1024^3 from 1200 projections of 1536^2
        {"name": "fdk-1024-f16", **_scan("fdk", 1024, 1024, 1024, 1536, 1536, 1200, 1.5, 10000.0,
                                         "f16", "shepplogan")},
        # the reference program's flow: projections in host memory, slabs back
        # to host memory through the sink
        {"name": "host-256-f32", **_scan("host", 256, 256, 256, 512, 400, 360, 1.75, 5000.0)},
        # one training step with learnable taps, whole stack: the 256^3 workload
        {"name": "train-256-f32", **_scan("train", 256, 256, 256, 256, 256, 360, 1.0, 2500.0)},
        # a training step of a large scan, FP16 storage, 50-projection chunks,
        # loss on the central 128^3
        {"name": "train-512-f16", **_scan("train", 512, 512, 512, 768, 768, 600, 1.5, 10000.0,
                                          "f16", chunk=50, crop=128)},
        # filter and pack of 50 projections of 2048^2: the chunk that precedes a
        # large backprojection
        {"name": "filter-pack-2048-f16", **_scan("filter", 1024, 1024, 64, 2048, 2048, 1800, 2.0,
                                                 10000.0, "f16", "shepplogan", block=50)},
        # backprojection of a block of angles, FP32 storage, odd slice count
        {"name": "backproject-640-f32", **_scan("bp", 640, 640, 321, 1280, 900, 1200, 1.96875,
                                                6400.0, "f32", block=120, ang0=240)},
        # the adjoint alone, dense volume, as an iterative method calls it
        {"name": "forward-384-f32", **_scan("fp", 384, 384, 320, 640, 600, 720, 1.5, 4000.0,
                                            block=90, ang0=100)},
        # one detector block of raw Scanco sinograms to FP32 full-fan sinograms
        {"name": "rsq-248-f32", "kind": "rsq", "sin_x": 1024, "sin_y": 2000, "n": 248, "axis": 21,
         "complete": True, "store": "f32"},
        # range and 16-bit scaling of a reconstructed volume for image export
        {"name": "export-512-u16", "kind": "export", "nx": 512, "ny": 512, "nz": 512},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fdk", "fdk", "fdk", "host", "train", "train", "filter", "bp", "fp", "rsq",
                       "export"])
    if kind == "rsq":
        sx = _logint(rng, 96, 1024)
        return {"kind": "rsq", "sin_x": sx, "sin_y": _logint(rng, 360, 2000),
                "n": _logint(rng, 4, 248), "axis": rng.randrange(0, max(1, sx // 12)),
                "complete": rng.random() < 0.75, "store": rng.choice(["f32", "f32", "f64"])}
    if kind == "export":
        return {"kind": "export", "nx": _logint(rng, 40, 640), "ny": _logint(rng, 40, 640),
                "nz": _logint(rng, 20, 640)}
    store = rng.choice(["f32", "f32", "f16", "f16", "bf16", "f16p"])
    if kind == "train":
        store = rng.choice(["f32", "f32", "f16", "f64"])
        n = _logint(rng, 24, 48 if store == "f64" else 384)
    elif kind in ("filter", "bp", "fp"):
        if kind == "fp":
            store = "f32"
        n = _logint(rng, 48, 512)
    else:
        n = _logint(rng, 32, 512)
    nx, ny = n, max(16, n - rng.choice([0, 0, 0, rng.randrange(1, 14)]))
    nz = max(8, int(n * rng.uniform(0.4, 1.1)))
    scale = rng.choice([1.0, 1.0, 1.5, 2.0, round(rng.uniform(0.75, 2.0) * 64) / 64.0])
    nu = max(32, int(math.ceil(n * scale * rng.uniform(1.0, 1.2))))
    nv = max(24, int(math.ceil(nz * scale * rng.uniform(0.95, 1.3))))
    nang = _logint(rng, max(24, n // 2), max(60, min(900, 3 * n)))
    dist = float(int(nu * math.exp(rng.uniform(math.log(2.5), math.log(20.0)))))
    c = _scan(kind, nx, ny, nz, nu, nv, nang, scale, dist, store,
              rng.choice(["ramlak", "shepplogan"]), shift=rng.choice([0.0, 0.0, 0.5, -1.5, 2.25]))
    if kind in ("filter", "bp", "fp"):
        c["block"] = max(8, min(nang, _logint(rng, 16, 160)))
        c["ang0"] = rng.randrange(0, nang - c["block"] + 1)
    if kind == "train":
        c["chunk"] = rng.choice([0, 0, 24, 50]) if store != "f64" else 0
        c["crop"] = rng.choice([0, 0, max(8, n // 4)])
    return c


# ---------------------------------------------------------------- inputs
def _tau(c):
    return float(np.float32(0.05 / (c["nu"] / 128.0)))


def _dbeta(c):
    return float(np.float32(2.0 * math.pi / c["nang"]))


def _centre(c):
    return (c["nu"] - 1) / 2.0 + c["shift"], (c["nv"] - 1) / 2.0


def _p(c):
    p = 2
    while p < c["nu"]:
        p *= 2
    return 2 * p


def _angles(c):
    """First projection and number of projections of the call."""
    return (c["ang0"], c["block"]) if c["block"] else (0, c["nang"])


def _projections(c, seed):
    """Line integrals through a body and six inclusions (spheres) with counting
    noise of 1e5 photons: float32 [nv][n][nu] on the GPU."""
    rng = random.Random(seed * 7919 + 13)
    gen = torch.Generator(device="cuda").manual_seed(seed * 104729 + 7)
    nu, nv, d = c["nu"], c["nv"], c["dist"]
    a0, n = _angles(c)
    half = 0.5 * c["nx"] * c["scale"]
    halfz = 0.5 * c["nz"] * c["scale"]
    balls = [(0.0, 0.0, 0.0, 0.85 * half, 1.2)]
    for _ in range(6):
        r, t = 0.55 * half * math.sqrt(rng.random()), rng.uniform(0, 2 * math.pi)
        balls.append((r * math.cos(t), r * math.sin(t), rng.uniform(-0.6, 0.6) * halfz,
                      rng.uniform(0.06, 0.25) * half, rng.choice([-0.25, 0.3, 0.6])))
    cx, cz = _centre(c)
    du = (torch.arange(nu, device="cuda", dtype=torch.float32) - cx)[None, None, :]
    dv = (torch.arange(nv, device="cuda", dtype=torch.float32) - cz)[:, None, None]
    inv2 = 1.0 / (du * du + dv * dv + d * d)
    out = torch.empty((nv, n, nu), device="cuda")
    step = max(1, int(4e7 // (nu * nv)))
    for k0 in range(0, n, step):
        k1 = min(n, k0 + step)
        b = (torch.arange(a0 + k0, a0 + k1, device="cuda", dtype=torch.float64)
             * _dbeta(c)).float()[None, :, None]
        cb, sb = torch.cos(b), torch.sin(b)
        p = torch.zeros((nv, k1 - k0, nu), device="cuda")
        for x, y, z, r, w in balls:
            mag = d / (d - (x * cb + y * sb))
            ot = du / mag - (y * cb - x * sb)
            oz = dv / mag - z
            h = ot * ot + oz * oz - (ot * du + oz * dv).square() * inv2
            p += w * torch.sqrt(torch.clamp(1.0 - h / (r * r), min=0.0))
        p += torch.randn(p.shape, device="cuda", generator=gen) * torch.exp(0.5 * p) * 0.00316
        out[:, k0:k1] = p
    return out


def _volume(c, seed):
    """A smooth field plus noise, float32 [nz][ny][nx]."""
    gen = torch.Generator(device="cuda").manual_seed(seed * 15485863 + 3)
    v = torch.randn((c["nz"], c["ny"], c["nx"]), device="cuda", generator=gen) * 0.1
    z = torch.linspace(-1, 1, c["nz"], device="cuda")[:, None, None]
    y = torch.linspace(-1, 1, c["ny"], device="cuda")[None, :, None]
    x = torch.linspace(-1, 1, c["nx"], device="cuda")[None, None, :]
    ph = random.Random(seed).uniform(0, 3)
    return v + torch.cos(3 * x + ph) * torch.cos(2 * y) * torch.cos(2 * z - ph)


def _gradient(c, seed):
    """What the next layer hands back: a volume, zero outside the crop."""
    v = _volume(c, seed)
    if c["crop"]:
        g = torch.zeros_like(v)
        s = [slice(max(0, (m - c["crop"]) // 2), (m - c["crop"]) // 2 + c["crop"])
             for m in (c["nz"], c["ny"], c["nx"])]
        s = [slice(q.start, max(q.stop, q.start + 1)) for q in s]
        g[s[0], s[1], s[2]] = v[s[0], s[1], s[2]]
        return g
    return v


def _taps(c, seed):
    """p spatial taps: the Ram-Lak response of the detector, slightly retrained."""
    nu, p, tau = c["nu"], _p(c), _tau(c)
    n = np.arange(nu) - nu // 2
    odd = -1.0 / (np.maximum(n * n, 1) * math.pi ** 2 * tau * tau)
    t = np.zeros(p)
    t[:nu] = np.where(n == 0, 1.0 / (4 * tau * tau), np.where(n % 2 == 0, 0.0, odd)) / 2
    h = np.real(np.fft.ifft(tau * np.abs(np.fft.fft(t))))
    return h * (1.0 + 0.02 * np.random.RandomState(seed % (1 << 31)).randn(p))


def _rsq_raw(c, seed):
    """Raw sinograms [n][sin_y + 2][sin_x] of 16-bit counts: a dark row, a flat
    row, the projections (held in int16, the same bits)."""
    gen = torch.Generator(device="cuda").manual_seed(seed * 49979687 + 5)
    n, sy, sx = c["n"], c["sin_y"], c["sin_x"]
    raw = torch.empty((n, sy + 2, sx), device="cuda", dtype=torch.int16)
    col = torch.arange(sx, device="cuda", dtype=torch.float32)
    for k in range(n):
        dark = torch.randint(180, 260, (sx,), device="cuda", generator=gen).float()
        flat = 52000 + 4000 * torch.rand(sx, device="cuda", generator=gen)
        att = 2.5 * torch.sqrt(torch.clamp(1 - (col / (0.9 * sx)) ** 2, min=0.0))
        i = dark + (flat - dark) * torch.exp(-att * (1 + 0.1 * torch.rand(
            (sy, sx), device="cuda", generator=gen)))
        raw[k] = torch.cat([dark[None], flat[None], i]).to(torch.int32).to(torch.int16)
    return raw


# ---------------------------------------------------------------- what a program holds
class _DeviceArray:
    """A device buffer of the engine as torch sees it; keeps the engine, which
    owns the buffer, for as long as a tensor over it lives."""

    def __init__(self, fbp, ptr, shape):
        self.fbp = fbp
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "version": 2,
                                         "data": (ptr, False), "strides": None}


def _engine(c, sink=None, storage=True):
    cx, cz = _centre(c)
    g = geometry.ScanGeometry(Nu=c["nu"], Nv=c["nv"], Nang=c["nang"], tau=_tau(c), D=c["dist"],
                              Nx=c["nx"], Ny=c["ny"], Nz=c["nz"], scale=c["scale"], cX=cx, cZ=cz,
                              B=16, dbeta=_dbeta(c))
    fbp = FilteredBackProjection(0)
    g.apply(fbp, None, sink)
    if storage and c["store"] != "f64":
        _lib.check(fbp.SetStorage(STORE[c["store"]]), "SetStorage")
    kind = _lib.FILTER_SHEPPLOGAN if c["filt"] == "shepplogan" else _lib.FILTER_RAMLAK
    _lib.check(fbp.SetFilter(kind), "SetFilter")
    return fbp


def prepare(case, seed):
    c, s = case, {"case": case}
    if c["kind"] == "rsq":
        p = _lib.RsqParams()
        L = _lib.load()
        _lib.check(L.fdk_rsq_default_params(C.byref(p)), "fdk_rsq_default_params")
        p.sin_x, p.sin_y, p.axis_move = c["sin_x"], c["sin_y"], c["axis"]
        p.distance, p.delta_fi = 5.0 * c["sin_x"], 2 * math.pi / c["sin_y"]
        p.complete, p.invert = int(c["complete"]), 1
        w = 2 * c["sin_x"] - 1 - 2 * c["axis"] if c["complete"] else c["sin_x"] - c["axis"]
        dt = torch.float64 if c["store"] == "f64" else torch.float32
        s.update(L=L, p=p, raw=_rsq_raw(c, seed),
                 out=torch.empty((c["n"], c["sin_y"], w), device="cuda", dtype=dt))
        return s
    if c["kind"] == "export":
        s.update(L=_lib.load(), vol=_volume(c, seed), mm=(C.c_double * 2)())
        return s
    if c["kind"] == "host":
        sink = VolumeSink(c["nx"], c["ny"], c["nz"], 16)
        s.update(fbp=_engine(c, sink), sink=sink, proj=_projections(c, seed).cpu().numpy())
        return s
    if c["kind"] == "fdk":
        fbp = _engine(c)
        _lib.check(fbp.Initialize(), "Initialize")
        proj = _projections(c, seed)
        torch.cuda.synchronize()
        assert hip().hipMemcpy(C.c_void_p(fbp.device_sinogram_ptr()), C.c_void_p(proj.data_ptr()),
                               proj.numel() * 4, 3) == 0
        shape = (c["nz"], c["ny"], c["nx"])
        s.update(fbp=fbp, vol=torch.as_tensor(_DeviceArray(fbp, fbp.device_volume_ptr(),
                                                           shape), device="cuda"))
        return s
    st = Stages(_engine(c, storage=False))
    s.update(st=st)
    if c["kind"] == "train":
        dt = torch.float64 if c["store"] == "f64" else torch.float32
        s.update(proj=_projections(c, seed).to(dt), grad=_gradient(c, seed).to(dt),
                 taps=_taps(c, seed))
    elif c["kind"] == "filter":
        s.update(proj=_projections(c, seed))
    elif c["kind"] == "fp":
        s.update(vol=_volume(c, seed))
    else:
        y = _projections(c, seed)
        m = torch.zeros(y.shape[1], dtype=torch.int32, device="cuda")
        st.filter(y, weight=True, maxabs=m)
        stack, scales = st.pack(y, STORE[c["store"]], m)
        torch.cuda.synchronize()
        s.update(stack=stack, scales=scales)
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "fdk":
        _lib.check(s["fbp"].CalculateReconstruction(), "CalculateReconstruction")
        return s["vol"]
    if kind == "host":
        _lib.check(s["fbp"].ReconstructHost(s["proj"]), "ReconstructHost")
        return s["sink"].volume
    if kind == "train":
        st, store = s["st"], STORE[c["store"]]
        diff.set_taps(st, s["taps"])
        vol = diff.forward(st, s["proj"], storage=store, chunk=c["chunk"] or None)
        gproj, dh = diff.backward(st, s["proj"], s["grad"], chunk=c["chunk"] or None)
        return {"vol": vol, "proj_grad": gproj,
                "taps_grad": torch.from_numpy(dh).to(gproj.device, gproj.dtype)}
    if kind == "filter":
        st, store = s["st"], STORE[c["store"]]
        y = s["proj"].clone()
        m = torch.zeros(y.shape[1], dtype=torch.int32, device=y.device)
        st.filter(y, weight=True, maxabs=m)
        stack, scales = st.pack(y, store, m)
        return {"filtered": y, "stack": _samples(st, c, stack), "scales": scales}
    if kind == "bp":
        return s["st"].backproject(s["stack"], STORE[c["store"]], s["scales"], c["ang0"],
                                   c["block"])
    if kind == "fp":
        return s["st"].forward_project(s["vol"], c["ang0"], c["block"])
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    if kind == "rsq":
        _lib.check(s["L"].fdk_rsq_process(C.byref(s["p"]), RSQ_BH[0], RSQ_BH[1],
                                          s["raw"].data_ptr(), c["n"], STORE[c["store"]],
                                          s["out"].data_ptr(), stream), "fdk_rsq_process")
        return s["out"]
    v = s["vol"]
    _lib.check(s["L"].fdk_volume_minmax(v.data_ptr(), v.numel(), s["mm"], stream), "minmax")
    u = torch.empty(v.shape, dtype=torch.int16, device=v.device)
    _lib.check(s["L"].fdk_volume_to_u16(v.data_ptr(), v.numel(), s["mm"][0], s["mm"][1],
                                        u.data_ptr(), stream), "to_u16")
    return {"min": s["mm"][0], "max": s["mm"][1], "u16": u}


def _samples(st, c, stack):
    """The stored samples [n][nv][nu] of a packed stack (rows are padded)."""
    n, b = _angles(c)[1], BYTES[c["store"]]
    per = st.stack_bytes(STORE[c["store"]], 1) - st.stack_bytes(STORE[c["store"]], 0)
    dt = {"f32": torch.float32, "bf16": torch.bfloat16}.get(c["store"], torch.float16)
    return stack[: per * n].view(dt).view(n, c["nv"], per // (b * c["nv"]))[:, :, : c["nu"]]


# ---------------------------------------------------------------- what a pass needs
def work(case):
    c = case
    if c["kind"] == "rsq":
        raw = c["n"] * (c["sin_y"] + 2) * c["sin_x"]
        w = 2 * c["sin_x"] - 1 - 2 * c["axis"] if c["complete"] else c["sin_x"] - c["axis"]
        out = c["n"] * c["sin_y"] * w
        return {"bytes": 2 * raw + BYTES[c["store"]] * out, "flops": 40.0 * raw + 6.0 * out}
    if c["kind"] == "export":
        n = c["nx"] * c["ny"] * c["nz"]
        return {"bytes": 8 * n + 2 * n, "flops": 5.0 * n}
    n = _angles(c)[1]
    b = 8 if c["store"] == "f64" else 4
    sino, vol = n * c["nu"] * c["nv"], c["nx"] * c["ny"] * c["nz"]
    # voxels inside the reconstruction cylinder
    r = 0.5 * c["nu"] / c["scale"]
    inside = min(1.0, math.pi * min(r, c["nx"] / 2) * min(r, c["ny"] / 2) / (c["nx"] * c["ny"]))
    # position 2, three lerps 6, weight and sum 2
    bp = 10.0 * vol * inside * n
    p = _p(c)
    filt = sino / c["nu"] * (5.0 * p * math.log2(p) + 3.0 * p)
    if c["kind"] in ("fdk", "host"):
        return {"bytes": 4 * sino + 4 * vol, "flops": bp + filt}
    if c["kind"] == "filter":
        return {"bytes": (4 + 4 + BYTES[c["store"]]) * sino, "flops": filt}
    if c["kind"] == "bp":
        return {"bytes": BYTES[c["store"]] * sino + 4 * vol, "flops": bp}
    if c["kind"] == "fp":
        return {"bytes": 4 * sino + 4 * vol, "flops": bp}
    share = min(1.0, c["crop"] ** 3 / vol / inside) if c["crop"] else 1.0
    return {"bytes": 2 * b * (sino + vol), "flops": bp * (1.0 + share) + 3.0 * filt}


# ---------------------------------------------------------------- the same in 64 bits
def _axes(c):
    f = dict(device="cuda", dtype=torch.float64)
    ax = c["scale"] * (torch.arange(c["nx"], **f) - (c["nx"] - 1) / 2.0)
    ay = c["scale"] * (torch.arange(c["ny"], **f) - (c["ny"] - 1) / 2.0)
    az = c["scale"] * (torch.arange(c["nz"], **f) - (c["nz"] - 1) / 2.0)
    X, Y = ax[None, :].expand(c["ny"], -1), ay[:, None].expand(-1, c["nx"])
    inside = (X * X + Y * Y) < (0.5 * c["nu"]) ** 2
    return X[inside], Y[inside], az, inside


def _project(c, X, Y, k):
    """u, U and the columns that meet the detector at projection k."""
    b = k * _dbeta(c)
    cb, sb = math.cos(b), math.sin(b)
    U = c["dist"] / (c["dist"] - (X * cb + Y * sb))
    u = (Y * cb - X * sb) * U + _centre(c)[0]
    on = (u >= 0) & (u <= c["nu"] - 1)
    iu = u.floor().clamp(0, c["nu"] - 2).long()
    return U, iu, u - iu, on


def _rows(c, U, az):
    v = az[:, None] * U[None, :] + _centre(c)[1]
    on = (v >= 0) & (v <= c["nv"] - 1)
    iv = v.floor().clamp_(0, c["nv"] - 2).long()
    return iv, v - iv, on


def _weight(c):
    cx, cz = _centre(c)
    f = dict(device="cuda", dtype=torch.float64)
    du, dv = torch.arange(c["nu"], **f) - cx, torch.arange(c["nv"], **f) - cz
    d = c["dist"]
    return (d / torch.sqrt(du[None, :] ** 2 + dv[:, None] ** 2 + d * d))[:, None, :]


def _spectrum(c, taps=None):
    p, tau, nu = _p(c), _tau(c), c["nu"]
    if taps is not None:
        return torch.from_numpy(np.fft.rfft(taps)).cuda()
    n = np.arange(nu) - nu // 2
    t = np.zeros(p)
    if c["filt"] == "shepplogan":
        t[:nu] = -2.0 / (math.pi ** 2 * tau * tau * (4.0 * n * n - 1.0)) / 2
    else:
        odd = -1.0 / (np.maximum(n * n, 1) * math.pi ** 2 * tau * tau)
        t[:nu] = np.where(n == 0, 1.0 / (4 * tau * tau), np.where(n % 2 == 0, 0.0, odd)) / 2
    return torch.from_numpy(tau * np.abs(np.fft.rfft(t))).cuda().to(torch.complex128)


def _filtered(c, x, H):
    """Rows of x [nv][n][nu] through the spectrum, inverse transform unnormalised."""
    p, y = _p(c), torch.empty_like(x)
    step = max(1, int(3e7 // (p * c["nv"])))
    for k in range(0, x.shape[1], step):
        f = torch.fft.rfft(x[:, k:k + step], n=p) * H
        y[:, k:k + step] = torch.fft.irfft(f, n=p)[..., : c["nu"]] * p
    return y


def _backprojected(c, q, a0):
    X, Y, az, inside = _axes(c)
    vol = torch.zeros((c["nz"], X.numel()), device="cuda", dtype=torch.float64)
    for k in range(q.shape[1]):
        U, iu, fu, on = _project(c, X, Y, a0 + k)
        w = torch.where(on, U * U, torch.zeros_like(U))
        h = q[:, k, :][:, iu] * (w * (1 - fu)) + q[:, k, :][:, iu + 1] * (w * fu)
        iv, fv, ok = _rows(c, U, az)
        lo = torch.gather(h, 0, iv)
        lo += fv * (torch.gather(h, 0, iv + 1) - lo)
        vol += lo * ok
    out = torch.zeros((c["nz"], c["ny"], c["nx"]), device="cuda", dtype=torch.float64)
    out[:, inside] = vol * (_dbeta(c) / _p(c))
    return out


def _forward_projected(c, x, a0, n):
    """The transpose of _backprojected."""
    X, Y, az, inside = _axes(c)
    x = x.double()[:, inside] * (_dbeta(c) / _p(c))
    used = (x != 0).any(dim=0)
    slices = (x != 0).any(dim=1)
    X, Y, x, az = X[used], Y[used], x[slices][:, used], az[slices]
    out = torch.zeros((c["nv"], n, c["nu"]), device="cuda", dtype=torch.float64)
    at = torch.arange(c["nu"] + 1, device="cuda")
    for k in range(n):
        U, iu, fu, on = _project(c, X, Y, a0 + k)
        iv, fv, ok = _rows(c, U, az)
        xx = x * ok
        g = torch.zeros((c["nv"], X.numel()), device="cuda", dtype=torch.float64)
        g.scatter_add_(0, iv, xx * (1 - fv))
        g.scatter_add_(0, iv + 1, xx * fv)
        g *= torch.where(on, U * U, torch.zeros_like(U))
        order = torch.argsort(iu)
        edge = torch.searchsorted(iu[order], at)
        for w, shift in ((1 - fu, 0), (fu, 1)):
            cs = torch.nn.functional.pad(torch.cumsum((g * w)[:, order], 1), (1, 0))
            seg = cs[:, edge[1:]] - cs[:, edge[:-1]]
            out[:, k, shift:] += seg[:, : c["nu"] - shift]
    return out


def _exact_rsq(c, seed):
    n, sy, sx, am = c["n"], c["sin_y"], c["sin_x"], c["axis"]
    raw = _rsq_raw(c, seed)
    w = 2 * sx - 1 - 2 * am if c["complete"] else sx - am
    out = torch.empty((n, sy, w), device="cuda", dtype=torch.float64)
    c0 = sx - 1 - am
    dfi = 2 * math.pi / sy
    t = torch.arange(-c0, 0, device="cuda", dtype=torch.float64)
    at = torch.atan(t / (5.0 * sx))
    fi = torch.arange(sy, device="cuda", dtype=torch.float64)[:, None] * dfi
    nf = (fi - 2 * at - math.pi) / dfi
    nf = torch.where((nf > sy - 1) | (nf < 0), (fi - 2 * at + math.pi) / dfi, nf)
    ca, fl = nf.ceil(), nf.floor()
    col = (am - t).long()
    for k in range(n):
        r = (raw[k].int() & 0xffff).double()
        v = -(RSQ_BH[0] * torch.log((r[2:] - r[0]) / (r[1] - r[0])) + RSQ_BH[1])
        if not c["complete"]:
            out[k] = v[:, am:]
            continue
        out[k, :, c0:] = v[:, am:]
        A = v[ca.long() % sy, col]
        out[k, :, :c0] = torch.where(ca != fl, A + (v[fl.long() % sy, col] - A) * (ca - nf), A)
    return out


def exact(case, seed):
    c = case
    if c["kind"] == "rsq":
        return _exact_rsq(c, seed)
    if c["kind"] == "export":
        v = _volume(c, seed).double()
        lo, hi = v.min(), v.max()
        u = torch.floor(65535 * (v - lo) / (hi - lo)).to(torch.int32).to(torch.int16)
        return {"min": float(lo), "max": float(hi), "u16": u}
    a0, n = _angles(c)
    vol = c["nx"] * c["ny"] * c["nz"]
    if c["kind"] == "fp":
        return _forward_projected(c, _volume(c, seed), a0, n)
    if vol * n > 1.3e11 and c["kind"] != "filter":   # takes too long
        return None
    x = _projections(c, seed).double()
    x *= _weight(c)
    taps = _taps(c, seed) if c["kind"] == "train" else None
    H = _spectrum(c, taps)
    q = _filtered(c, x, H)
    if c["kind"] == "filter":
        scales = q.abs().amax(dim=(0, 2)) / 8192.0
        if c["store"] not in ("f16", "f16p"):
            scales = torch.ones_like(scales)
        return {"filtered": q, "scales": scales, "stack": (q / scales[None, :, None]).transpose(0, 1)}
    if c["kind"] == "bp":
        del x
        return _backprojected(c, q, a0)
    out = _backprojected(c, q, 0)
    if c["kind"] != "train":
        return out
    del q
    g = _forward_projected(c, _gradient(c, seed), 0, n)
    p = _p(c)
    R = torch.zeros(p // 2 + 1, device="cuda", dtype=torch.complex128)
    step = max(1, int(3e7 // (p * c["nv"])))
    for k in range(0, n, step):
        Q = torch.fft.rfft(x[:, k:k + step], n=p)
        R += (Q.conj() * torch.fft.rfft(g[:, k:k + step], n=p)).sum(dim=(0, 1))
    return {"vol": out, "proj_grad": _filtered(c, g, H.conj()) * _weight(c),
            "taps_grad": torch.fft.irfft(R, n=p) * p}
