"""Performance cases: what a user of this package has it compute, at the sizes it is used at.

A scan's way through the package is: line integrals of a phantom (simulation
only), the cosine weight and ramp filter, FP16/BF16 storage of the views,
and one of the backprojectors -- a plan kept for a geometry, a batch of
scans, ``feldkamp`` as one call, the host-array ``cbct_back`` and its FP64
MATLAB route, and the helical geometries.  Sizes are those of
``mirt_amd.workloads`` (``cpu_small``, ``plain_flat``, ``clinical_arc``,
``clinical_helix``, ``uneven_scans``) or smaller scans on the same detectors;
``draw`` varies them.  Views are smooth objects on source-following tracks
with noise, ramp-filtered where the path takes filtered views.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from mirt_amd import (FdkBatch, FdkPlan, _lib, cbct_back, ct_geom, geom_of, image_geom,
                      quantize_views)
from mirt_amd.cbct_back_helix import helix_operands
from mirt_amd.fdk import feldkamp, weight_filter_views
from mirt_amd.phantom import ellipsoid_proj

DSO, DSD = 541.0, 949.0
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}


# ---------------------------------------------------------------------------
# the cases

def listed():
    arc = dict(arc=True, ns=888, nt=64, ds=1.0239, dt=1.0964, offset_s=1.25)
    flat = dict(arc=False, ns=512, nt=384, na=360, ds=0.8, dt=0.8, offset_s=0.0)
    helix = dict(arc, na=3 * 492, turns=3, pitch=1.0, nx=256, ny=256, nz=192, dx=1.4, dz=0.625)
    return [
        # a test-size scan on a kept plan: launches and latency count
        dict(name="plan_small_f32", op="plan", fmt="f32", math="exact", mask=False, tune=False,
             arc=False, ns=128, nt=96, na=64, ds=1.0, dt=1.0, offset_s=0.0,
             nx=64, ny=64, nz=32, dx=1.0, dz=1.0),
        # a flat-panel scan in the reference's FP32 arithmetic, plan as created
        dict(flat, name="plan_flat_f32", op="plan", fmt="f32", math="exact", mask=False,
             tune=False, nx=256, ny=256, nz=128, dx=0.5, dz=0.5),
        # the clinical arc scan with FP16 views on an autotuned plan (production use)
        dict(arc, name="plan_arc_f16_tuned", op="plan", fmt="f16", math="fast", mask=False,
             tune=True, na=984, nx=512, ny=512, nz=256, dx=0.7, dz=0.625),
        # odd sizes everywhere, a circular mask, BF16 views, plan as created
        dict(name="plan_ragged_bf16", op="plan", fmt="bf16", math="fast", mask=True, tune=False,
             arc=True, ns=731, nt=61, na=491, ds=1.24, dt=1.15, offset_s=1.25,
             nx=251, ny=247, nz=117, dx=1.43, dz=0.9),
        # several scans of uneven size in one execute (a reconstruction server)
        dict(name="batch_uneven_f16", op="batch", fmt="f16", scans=8, scan_seed=4000,
             largest=256),
        # native helical scan on a kept plan, reference arithmetic
        dict(helix, name="plan_helix_f32", op="helix", fmt="f32", math="exact"),
        # rebinned (cone-parallel) helical views with the conjugate-ray weights
        dict(helix, name="cone_par_w3d_f32", op="cone_par", w3d=1),
        # cosine weight and ramp filter of the clinical arc scan on the device
        dict(arc, name="filter_arc_f32", op="filter", window="ramp", na=984),
        # one whole reconstruction call on device views: filter, FP16 storage, plan,
        # backprojection
        dict(arc, name="feldkamp_arc_f16", op="feldkamp", fmt="f16", window="hann", na=492,
             nx=256, ny=256, nz=128, dx=1.4, dz=0.625),
        # the drop-in call on host arrays in MATLAB order
        dict(flat, name="cbct_back_host_flat", op="host", mask=False, nx=256, ny=256, nz=128,
             dx=0.5, dz=0.5),
        # the FP64 MATLAB backprojector on device views
        dict(arc, name="mat_arc_f64", op="mat", mask=False, na=492, nx=256, ny=256, nz=128,
             dx=1.4, dz=0.625),
        # analytic line integrals of a phantom: the input of every simulated study
        dict(flat, name="phantom_flat_f64", op="phantom", nell=20, oversample=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["plan", "plan", "plan", "batch", "helix", "cone_par", "filter", "feldkamp",
                     "host", "mat", "phantom"])
    if op == "batch":
        return dict(op=op, fmt=rng.choice(["f32", "f16", "bf16"]), scans=_log(rng, 2, 10),
                    scan_seed=rng.randrange(1 << 20), largest=rng.choice([128, 192, 256]))
    arc = rng.random() < 0.5
    ns = _log(rng, 64, 1000)
    nt = _log(rng, 24, 80) if arc else _log(rng, 32, 400)
    # a detector 640 to 900 mm wide; on an arc the filter's taps reach twice its fan angle
    npad = 2 ** math.ceil(math.log2(2 * ns - 1))
    width = rng.uniform(400, 900)
    if arc:
        width = min(width, 1.3 * DSD * 2 * ns / npad)
    ds = width / ns
    case = dict(op=op, arc=arc, ns=ns, nt=nt, na=_log(rng, 24, 720), ds=ds,
                dt=ds * rng.uniform(0.8, 1.2) if not arc else rng.uniform(0.6, 1.2),
                offset_s=rng.choice([0.0, 0.25, 1.25]))
    if op == "phantom":
        over = rng.choice([1, 1, 2])
        case["na"] = min(case["na"], 360 // over ** 2)
        return dict(case, nell=_log(rng, 3, 30), oversample=over)
    if op == "filter":
        return dict(case, window=rng.choice(["ramp", "hann", "hanning,0.75"]))
    nx = _log(rng, 24, 320)
    ny = max(8, nx + rng.randrange(-9, 10))
    nz = _log(rng, 12, 200)
    dx = rng.uniform(0.45, 0.7) * width * DSO / DSD / nx
    # the volume's height over that of the detector at the axis
    dz = rng.uniform(0.4, 2.5) * nt * case["dt"] * DSO / DSD / nz
    case.update(nx=nx, ny=ny, nz=nz, dx=dx, dz=dz)
    if op == "plan":
        fmt = rng.choice(["f32", "f32", "f16", "bf16"])
        return dict(case, fmt=fmt, math=rng.choice(["exact", "fast"]) if fmt == "f32" else "fast",
                    mask=rng.random() < 0.5, tune=False)
    if op == "feldkamp":
        return dict(case, fmt=rng.choice(["f32", "f16", "bf16"]),
                    window=rng.choice(["ramp", "hann"]))
    if op in ("host", "mat"):
        return dict(case, mask=rng.random() < 0.5)
    # helices: 2 to 4 turns, the volume as tall as the source's way
    turns = rng.choice([2, 3, 4])
    pitch = rng.choice([0.5, 0.8, 1.0])
    way = turns * pitch * nt * case["dt"] * DSO / DSD
    case.update(na=turns * (2 * (case["na"] // 4) + 12), turns=turns, pitch=pitch, dz=way / nz)
    if op == "helix":
        fmt = rng.choice(["f32", "f32", "f16"])
        return dict(case, fmt=fmt, math="exact" if fmt == "f32" else "fast")
    return dict(case, w3d=rng.choice([0, 1, 1]))


# ---------------------------------------------------------------------------
# geometries and inputs

def _scans(case):
    """The scans of a batch, drawn as the uneven_scans workload draws them."""
    rng = np.random.default_rng(case["scan_seed"])
    out = []
    for _ in range(case["scans"]):
        edge = int(rng.choice([e for e in (128, 192, 256) if e <= case["largest"]]))
        na = int(rng.integers(180, 721))
        ns = int(rng.integers(256, 769))
        nt = int(rng.integers(128, 513))
        out.append(dict(op="plan", fmt=case["fmt"], math="exact", mask=False, arc=False, ns=ns,
                        nt=nt, na=na, ds=640 / ns, dt=320 / nt, offset_s=0.0, nx=edge, ny=edge,
                        nz=edge // 2, dx=200 / edge, dz=200 / edge))
    return out


def _geoms(case):
    helix = dict(pitch=case["pitch"], source_z0="center") if case.get("pitch") else {}
    cg = ct_geom("fan", ns=case["ns"], nt=case["nt"], na=case["na"], ds=case["ds"],
                 dt=case["dt"], offset_s=case["offset_s"], dsd=DSD, dso=DSO,
                 dfs=0.0 if case["arc"] else math.inf, orbit=360 * case.get("turns", 1), **helix)
    if "nx" not in case:
        return cg, None
    mask = None
    if case.get("mask"):
        x = np.arange(case["nx"]) - (case["nx"] - 1) / 2
        y = np.arange(case["ny"]) - (case["ny"] - 1) / 2
        disc = x[:, None] ** 2 + y[None, :] ** 2 <= (0.49 * min(case["nx"], case["ny"])) ** 2
        mask = np.broadcast_to(disc[:, :, None], (case["nx"], case["ny"], case["nz"]))
    ig = image_geom(nx=case["nx"], ny=case["ny"], nz=case["nz"], dx=case["dx"], dz=case["dz"],
                    mask=mask)
    return cg, ig


def _line_integrals(case, seed):
    """(na, ns, nt) FP32 line integrals: smooth blobs whose shadows follow the
    source, and noise."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    rnd = lambda *n: torch.rand(*n, generator=g, device=dev)   # noqa: E731
    ns, nt, na, k = case["ns"], case["nt"], case["na"], 12
    beta = torch.arange(na, device=dev) * (2 * math.pi * case.get("turns", 1) / na)
    r, phi = 0.35 * ns * rnd(k), 2 * math.pi * rnd(k)
    wid, hgt = ns * (0.02 + 0.15 * rnd(k)), nt * (0.1 + 0.4 * rnd(k))
    tc = nt * (0.2 + 0.6 * rnd(k))
    amp = 0.2 + rnd(k)
    s = torch.arange(ns, device=dev)[None, :, None] - ns / 2
    prof = torch.exp(-((s - r * torch.cos(beta[:, None, None] - phi)) / wid) ** 2) * amp
    rows = torch.exp(-((torch.arange(nt, device=dev)[None, :] - tc[:, None]) / hgt[:, None]) ** 2)
    p = (prof.reshape(na * ns, k) @ rows).reshape(na, ns, nt)
    return p.add_(torch.randn(p.shape, generator=g, device=dev), alpha=0.02)


def _filtered(case, seed):
    """(na, ns, nt) FP32 views after a ramp filter along s."""
    p = _line_integrals(case, seed)
    n = 2 ** math.ceil(math.log2(2 * case["ns"] - 1))
    ramp = torch.fft.rfftfreq(n, d=case["ds"], device=p.device)[None, :, None]
    out = torch.empty_like(p)
    for a in range(0, p.shape[0], 128):
        f = torch.fft.rfft(p[a:a + 128], n=n, dim=1)
        out[a:a + 128] = torch.fft.irfft(f.mul_(ramp), n=n, dim=1)[:, :case["ns"]]
    return out


def _ellipsoids(case, seed):
    rng = np.random.default_rng(seed)
    fov = np.array([250.0, 250.0, min(160.0, 0.9 * case["nt"] * case["dt"] * DSO / DSD)])
    rows = []
    for _ in range(case["nell"]):
        rows.append([*(rng.uniform(-0.3, 0.3, 3) * fov), *(rng.uniform(0.05, 0.4, 3) * fov),
                     rng.uniform(0, 180), 0.0, rng.uniform(0.005, 0.02)])
    return np.asarray(rows)


def _stored(p, fmt):
    """The values a plan of format fmt backprojects, FP64: the views themselves, or
    FP16/BF16 with a power-of-two scale per view that brings the largest to [2^14, 2^15)."""
    if fmt == "f32":
        return p.double()
    e = torch.frexp(p.abs().amax(dim=(1, 2)))[1] - 15
    scale = torch.ldexp(torch.ones_like(e, dtype=torch.float64), e)[:, None, None]
    return (p.double() / scale).to(torch.float32).to(DTYPES[fmt]).double() * scale


# ---------------------------------------------------------------------------
# what a program has in hand, and the call

def prepare(case, seed):
    op = case["op"]
    if op == "batch":
        scans = _scans(case)
        batch = FdkBatch([(geom_of(*_geoms(c)), _geoms(c)[0].ar, None) for c in scans],
                         fmt=case["fmt"])
        views = [_filtered(c, seed * 1000 + i) for i, c in enumerate(scans)]
        if case["fmt"] == "f32":
            return dict(op=op, batch=batch, args=(views,))
        stored = [quantize_views(p, case["fmt"]) for p in views]
        return dict(op=op, batch=batch, args=([q for q, _ in stored], [s for _, s in stored]))
    cg, ig = _geoms(case)
    if op in ("plan", "helix"):
        make = FdkPlan.helix_from_geoms if op == "helix" else FdkPlan.from_geoms
        plan = make(cg, ig, fmt=case["fmt"], math_mode=case["math"])
        p = _filtered(case, seed)
        args = (p,) if case["fmt"] == "f32" else quantize_views(p, case["fmt"])
        if case.get("tune"):
            plan.autotune(*args)
        return dict(op="plan", plan=plan, args=args)
    if op == "filter":
        raw = _line_integrals(case, seed).permute(0, 2, 1).contiguous()      # [ns nt na]
        return dict(op=op, cg=cg, proj=raw, window=case["window"])
    if op == "feldkamp":
        raw = _line_integrals(case, seed).permute(0, 2, 1).contiguous()
        return dict(op=op, cg=cg, ig=ig, proj=raw.permute(2, 1, 0), window=case["window"],
                    fmt=case["fmt"])
    if op == "host":
        p = _filtered(case, seed).cpu().numpy()                              # (na, ns, nt)
        return dict(op=op, cg=cg, ig=ig, proj=np.asfortranarray(p.transpose(1, 2, 0)))
    if op == "phantom":
        return dict(op=op, cg=cg, params=_ellipsoids(case, seed), oversample=case["oversample"])
    if op == "cone_par":
        na1_half, dz_per_rad = helix_operands(cg)
        return dict(op=op, geom=geom_of(cg, ig), proj=_filtered(case, seed), beta=cg.ar,
                    zs=np.ascontiguousarray(cg.source_zs), na1_half=na1_half, w3d=case["w3d"],
                    dz_per_rad=dz_per_rad, pitch=case["pitch"],
                    image=torch.empty((ig.ny, ig.nx, ig.nz), device="cuda"))
    assert op == "mat"
    mask = np.asfortranarray(ig.mask_or).astype(np.uint8, order="F")
    return dict(op=op, geom=geom_of(cg, ig), beta=cg.ar, mask=mask,
                proj=_filtered(case, seed).permute(0, 2, 1).contiguous(),    # [ns nt na]
                scale=math.pi / case["na"],
                image=torch.empty((ig.nz, ig.ny, ig.nx), dtype=torch.float64, device="cuda"))


def run(state):
    op = state["op"]
    if op == "plan":
        return state["plan"](*state["args"])
    if op == "batch":
        return state["batch"](*state["args"])
    if op == "filter":
        return weight_filter_views(state["proj"], state["cg"], window=state["window"])
    if op == "feldkamp":
        return feldkamp(state["cg"], state["ig"], state["proj"], window=state["window"],
                        fmt=state["fmt"])
    if op == "host":
        return cbct_back(state["proj"], state["cg"], state["ig"])
    if op == "phantom":
        return ellipsoid_proj(state["cg"], state["params"], oversample=state["oversample"])
    lib = _lib.load()
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    ptr = lambda a: C.c_void_p(a.ctypes.data)                                # noqa: E731
    dev = lambda t: C.c_void_p(t.data_ptr())                                 # noqa: E731
    if op == "cone_par":
        _lib.check(lib.fdkhip_fdk_ts_back_helix_direct(
            C.byref(state["geom"]), dev(state["proj"]), len(state["beta"]), ptr(state["beta"]),
            ptr(state["zs"]), state["na1_half"], 1, state["w3d"], state["dz_per_rad"],
            state["pitch"], None, dev(state["image"]), stream, None))
    else:
        _lib.check(lib.fdkhip_cbct_back_mat_direct(
            C.byref(state["geom"]), dev(state["proj"]), 0, len(state["beta"]),
            ptr(state["beta"]), None, 1, 0.0, ptr(state["mask"]), state["scale"],
            dev(state["image"]), stream, None))
    return state["image"]


# ---------------------------------------------------------------------------
# what a pass cannot do without

def _updates(case):
    """Voxel-view pairs inside the cone and, on a helix, the view's window,
    from a sample of columns and views."""
    nx, ny, nz, na = case["nx"], case["ny"], case["nz"], case["na"]
    x = ((np.linspace(0, nx - 1, min(nx, 48)) - (nx - 1) / 2) * case["dx"])[None, :, None]
    y = ((np.linspace(0, ny - 1, min(ny, 48)) - (ny - 1) / 2) * case["dx"])[:, None, None]
    b = (np.arange(16) * (2 * math.pi / 16))[None, None, :]
    xb, yb = x * np.cos(b) + y * np.sin(b), DSO - (y * np.cos(b) - x * np.sin(b))
    mag = DSD / yb
    s = (DSD * np.arctan2(xb, yb) if case["arc"] else mag * xb) / case["ds"]
    height = np.minimum(case["nt"] * case["dt"] / (mag * case["dz"]), nz)
    if case.get("pitch"):
        turn = case["pitch"] * case["nt"] * case["dt"] * DSO / DSD / case["dz"]
        height = np.minimum(height, turn)
    inside = np.abs(s) <= case["ns"] / 2
    if case.get("mask"):
        inside &= x * x + y * y <= (0.49 * min(nx, ny) * case["dx"]) ** 2
    return float(np.mean(inside * height)) * nx * ny * na


def _pairs(case):
    return case["nx"] * case["ny"] * case["nz"] * case["na"]


def work(case):
    op = case["op"]
    if op == "batch":
        each = [work(c) for c in _scans(case)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    views = case["ns"] * case["nt"] * case["na"]
    npad = 2 ** math.ceil(math.log2(2 * case["ns"] - 1))
    # two complex transforms of npad points for every pair of rows
    filt = case["nt"] * case["na"] * (5 * npad * math.log2(npad) + 2 * npad + case["ns"])
    if op == "filter":
        return {"bytes": 8 * views, "flops": filt}
    if op == "phantom":
        return {"bytes": 8 * views,
                "flops": 60 * views * case["nell"] * case["oversample"] ** 2}
    voxels = case["nx"] * case["ny"] * case["nz"]
    if op == "mat":
        # the MATLAB rules give every voxel of every view a sample
        return {"bytes": 4 * views + 8 * voxels, "flops": 20 * _pairs(case)}
    sample = 4 if op in ("feldkamp", "cone_par", "host") or case["fmt"] == "f32" else 2
    flops = 14 * _updates(case)
    if op == "cone_par" and case["w3d"]:
        flops *= 2
    return {"bytes": sample * views + 4 * voxels,
            "flops": flops + (filt if op == "feldkamp" else 0)}


# ---------------------------------------------------------------------------
# the same in 64 bits

def _sample64(view, sbin, tbin):
    """Bilinear samples of view (ns, nt) at (sbin (m,), tbin (m, k)), 0-based, zero outside."""
    ns, nt = view.shape
    grid = torch.empty(tbin.shape + (2,), dtype=torch.float64, device=view.device)
    grid[..., 0] = tbin * (2 / (nt - 1)) - 1
    grid[..., 1] = (sbin * (2 / (ns - 1)) - 1)[:, None]
    return torch.nn.functional.grid_sample(view[None, None], grid[None], mode="bilinear",
                                           padding_mode="zeros", align_corners=True)[0, 0]


def _columns64(case):
    cg, ig = _geoms(case)
    f = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.float64, device="cuda")  # noqa: E731
    y, x = torch.meshgrid(f(ig.y), f(ig.x), indexing="ij")
    return cg, ig, x.reshape(-1), y.reshape(-1), torch.arange(ig.nz, device="cuda").double()


def _windows64(case, cg, ig):
    """The slices [first, last) of each view of a helix: those between the source
    heights half a turn before and after it."""
    if not case.get("pitch"):
        return [(0, ig.nz)] * cg.na
    half, zs = helix_operands(cg)[0], cg.source_zs
    edge = lambda i: math.ceil(ig.wz + zs[min(max(i, 0), cg.na - 1)] / ig.dz)        # noqa: E731
    return [(max(edge(i - half), 0), min(edge(i + half), ig.nz)) for i in range(cg.na)]


def _back64(case, views):
    """(ny, nx, nz) of views(ia) -> (ns, nt) FP64, the cone-beam sum with zero borders."""
    cg, ig, x, y, iz = _columns64(case)
    acc = torch.zeros((x.numel(), ig.nz), dtype=torch.float64, device="cuda")
    zs = np.broadcast_to(cg.source_zs, (cg.na,))
    for ia, (z0, z1) in enumerate(_windows64(case, cg, ig)):
        if z0 >= z1:
            continue
        c, s = math.cos(cg.ar[ia]), math.sin(cg.ar[ia])
        xb, yb = x * c + y * s, DSO - (y * c - x * s)
        mag = DSD / yb
        ss = DSD * torch.atan2(xb, yb) if case["arc"] else mag * xb
        w2 = DSD ** 2 / (yb ** 2 + xb ** 2) if case["arc"] else mag ** 2
        tbin = torch.outer(mag * (ig.dz / cg.dt), iz[z0:z1] - (ig.wz + zs[ia] / ig.dz)) + cg.wt
        acc[:, z0:z1] += w2[:, None] * _sample64(views(ia), ss / cg.ds + cg.ws, tbin)
    acc *= torch.as_tensor(ig.mask_or.T.reshape(-1, 1).copy(), device="cuda")
    return acc.reshape(ig.ny, ig.nx, ig.nz)


def _cone_par64(case, views):
    """(ny, nx, nz) of cone-parallel views with the w3d weights of the conjugate ray."""
    cg, ig, x, y, iz = _columns64(case)
    acc = torch.zeros((x.numel(), ig.nz), dtype=torch.float64, device="cuda")
    zs, rate = cg.source_zs, helix_operands(cg)[1]
    half = case["nt"] // 2
    table = torch.zeros(half + 1, dtype=torch.float64, device="cuda")
    table[:half] = (torch.arange(half, device="cuda").double() * (ig.wz / DSD)) ** (
        case["w3d"] * case["pitch"])
    look = lambda t: table[(t - cg.wt).abs().clamp(max=half).floor().long()]         # noqa: E731
    for ia, (z0, z1) in enumerate(_windows64(case, cg, ig)):
        if z0 >= z1:
            continue
        c, s = math.cos(cg.ar[ia]), math.sin(cg.ar[ia])
        xb, yb = x * c + y * s, DSO - (y * c - x * s)
        root = torch.sqrt(DSO ** 2 - xb ** 2)
        rise = torch.asin(-xb / DSO) * rate / ig.dz
        k = iz[z0:z1][None, :]
        mag = DSD / (root - (DSO - yb))
        tbin = (mag * ig.dz / cg.dt)[:, None] * (k - (ig.wz + zs[ia] / ig.dz + rise)[:, None]) \
            + cg.wt
        p = _sample64(views(ia), xb / cg.ds + cg.ws, tbin)
        if case["w3d"]:
            mag_c = DSD / (root + (DSO - yb))
            up = tbin >= cg.wt
            zc = torch.where(up, zs[ia] + math.pi * rate, zs[ia] - math.pi * rate)
            tc = (mag_c * ig.dz / cg.dt)[:, None] * (k - (ig.wz + zc / ig.dz - rise[:, None])) \
                + cg.wt
            a, b = look(tc), look(tbin)
            share = torch.nan_to_num(a / (a + b), nan=0.0).clamp(0.001, 0.999)
            p = torch.where((zc >= zs[0]) & (zc <= zs[-1]), 2 * share, 1.0) * p
        acc[:, z0:z1] += p
    return acc.reshape(ig.ny, ig.nx, ig.nz)


def _mat64(case, views):
    """(nz, ny, nx): samples beyond the first and last detector column are 0, rows clamped."""
    cg, ig, x, y, iz = _columns64(case)
    acc = torch.zeros((x.numel(), ig.nz), dtype=torch.float64, device="cuda")
    for ia in range(cg.na):
        c, s = math.cos(cg.ar[ia]), math.sin(cg.ar[ia])
        xb, yb = x * c + y * s, DSO - (y * c - x * s)
        mag = DSD / yb
        ss = DSD * torch.atan2(xb, yb) if case["arc"] else mag * xb
        w2 = DSD ** 2 / (yb ** 2 + xb ** 2) if case["arc"] else mag ** 2
        sbin = ss / cg.ds + cg.ws
        w2 = w2 * ((sbin >= 0) & (sbin <= cg.ns - 1))
        tbin = torch.outer(mag, (iz - ig.wz) * ig.dz) / cg.dt + cg.wt
        acc += w2[:, None] * _sample64(views(ia), sbin, tbin.clamp(0, cg.nt - 1))
    acc *= (math.pi / cg.na) * torch.as_tensor(ig.mask_or.T.reshape(-1, 1).copy(), device="cuda")
    return acc.reshape(ig.ny, ig.nx, ig.nz).permute(2, 0, 1)


def _filter64(case, p):
    """(na, ns, nt): cosine weight, zero-padded ramp filter along s with the window."""
    cg = _geoms(case)[0]
    ns, nt, ds = cg.ns, cg.nt, cg.ds
    f = lambda a: torch.as_tensor(a, dtype=torch.float64, device="cuda")             # noqa: E731
    ss, tt = f(cg.s)[:, None], f(cg.t)[None, :]
    n = 2 ** math.ceil(math.log2(2 * ns - 1))
    nn = np.arange(-(n // 2), n // 2)
    odd = nn % 2 == 1
    h = np.zeros(n)
    h[n // 2] = 1 / (4 * ds ** 2)
    if case["arc"]:
        ww = (DSO / DSD) * torch.cos(ss / DSD) / torch.sqrt(1 + (tt / DSD) ** 2)
        h[odd] = -1 / (math.pi * DSD * np.sin(nn[odd] * ds / DSD)) ** 2
    else:
        ww = DSO / torch.sqrt(DSD ** 2 + ss ** 2 + tt ** 2)
        h[odd] = -1 / (math.pi * nn[odd] * ds) ** 2
    k = np.arange(n) - n // 2
    if case["window"] == "hann":
        win = 0.5 * (1 + np.cos(2 * math.pi * k / n))
    elif case["window"].startswith("hanning,"):
        w = math.floor(float(case["window"][8:]) * n + 0.5)
        win = 0.5 * (1 + np.cos(2 * math.pi * k / w)) * (np.abs(k) < w / 2)
    else:
        win = np.ones(n)
    resp = ds * np.real(np.fft.fft(np.fft.fftshift(h))) * np.fft.fftshift(win)
    resp = f(resp[:n // 2 + 1])[None, :, None]
    out = torch.empty(p.shape, dtype=torch.float64, device="cuda")
    for a in range(0, p.shape[0], 64):
        q = torch.fft.rfft(p[a:a + 64].double() * ww, n=n, dim=1)
        out[a:a + 64] = torch.fft.irfft(q * resp, n=n, dim=1)[:, :ns]
    return out


def _phantom64(case, params):
    """(ns, nt, na) line integrals of the ellipsoids."""
    cg = _geoms(case)[0]
    f = lambda a: torch.as_tensor(a, dtype=torch.float64, device="cuda")             # noqa: E731
    no = case["oversample"]
    off = [(2 * j - (no - 1)) / (2 * no) for j in range(no)]
    out = torch.zeros((cg.na, cg.nt, cg.ns), dtype=torch.float64, device="cuda")
    for dj in off:
        for di in off:
            ss, tt = (f(cg.s) + di * cg.ds)[None, None, :], (f(cg.t) + dj * cg.dt)[None, :, None]
            if case["arc"]:
                e1, e2 = DSD * torch.sin(ss / DSD), -DSD * torch.cos(ss / DSD)
                polar = -torch.asin(tt / torch.sqrt(e1 ** 2 + e2 ** 2 + tt ** 2))
                az = -torch.atan(e1 / e2)
                uu, vv = torch.sin(az) * DSO, -torch.cos(az) * DSO * torch.sin(polar)
            else:
                r = torch.sqrt(DSD ** 2 + ss ** 2)
                uu, polar, az = DSO * ss / r, -torch.atan(tt / r), torch.atan(ss / DSD)
                vv = DSO * tt / torch.sqrt(r ** 2 + tt ** 2) * DSD / r
            cp, sp = torch.cos(polar), torch.sin(polar)
            for a in range(0, cg.na, 30):
                phi = f(cg.ar[a:a + 30])[:, None, None] + az
                for cx, cy, cz, rx, ry, rz, deg, _, val in params:
                    rot = phi - math.radians(deg)
                    ca, sa = torch.cos(rot), torch.sin(rot)
                    du = uu - (cx * torch.cos(phi) + cy * torch.sin(phi))
                    dv = vv - ((cx * torch.sin(phi) - cy * torch.cos(phi)) * sp + cz * cp)
                    p1, p2, p3 = du * ca + dv * sa * sp, du * sa - dv * ca * sp, dv * cp
                    e1, e2, e3 = -sa * cp, ca * cp, sp
                    qa = (e1 / rx) ** 2 + (e2 / ry) ** 2 + (e3 / rz) ** 2
                    qb = p1 * e1 / rx ** 2 + p2 * e2 / ry ** 2 + p3 * e3 / rz ** 2
                    qc = (p1 / rx) ** 2 + (p2 / ry) ** 2 + (p3 / rz) ** 2 - 1
                    out[a:a + 30] += 2 * val * torch.sqrt((qb ** 2 - qa * qc).clamp(min=0)) / qa
    return (out / no ** 2).permute(2, 1, 0)


def exact(case, seed):
    op = case["op"]
    if op == "batch":
        return [exact(c, seed * 1000 + i) for i, c in enumerate(_scans(case))]
    if op == "phantom":
        return _phantom64(case, _ellipsoids(case, seed))
    if op == "filter":
        return _filter64(case, _line_integrals(case, seed))
    if op == "feldkamp":
        p = _filter64(case, _line_integrals(case, seed))
        return _back64(case, lambda ia: p[ia]).permute(1, 0, 2) * (math.pi / case["na"])
    p = _filtered(case, seed)
    if op == "mat":
        return _mat64(case, lambda ia: p[ia].double())
    if op == "cone_par":
        return _cone_par64(case, lambda ia: p[ia].double())
    if op == "host":
        img = _back64(case, lambda ia: p[ia].double()).permute(1, 0, 2)
        return (img * (math.pi / case["na"])).cpu().numpy()
    p = _stored(p, case["fmt"])
    return _back64(case, lambda ia: p[ia])
