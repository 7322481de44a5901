"""What is timed when the framework's speed is measured: the indexing path and its stages as a user's
program calls them, over the range of sizes, pixel types and options that they are used with.

A case is a dict of plain values; its "kind" names the call:

  scan          Solver.set_patterns and Solver.index on a scan in host memory (default settings)
  batch         Engine.run_batch on patterns on the GPU: filters, coefficients, correlation,
                refinement, records
  prep          zb_prep_work: the pattern filters and the normalization
  coefficients  zb_sh_coefficients: patterns onto the sphere and into harmonics
  refine        zb_refine_order and zb_refine_phases: orientations refined and scored
  fit           fit.fit6: patterns' poses fitted over the detector's shift and the orientation

listed() are the cases timed, draw(rng) makes others of the same ranges, prepare(case, seed) what a
program has in hand before the call, run(state) one pass, work(case) the bytes and operations a
pass cannot do without, exact(case, seed) the same outputs in 64 bits where they have such a value.
"""
import math
import os

import numpy as np
import torch

from zebsdsolve_amd import Solver, engine, fit, rot
from zebsdsolve_amd import _native as nat

GOLDEN = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tests", "golden")
MASTERS = {"ni": os.path.join(GOLDEN, "Ni_master_20kV.npz"), "gan": os.path.join(GOLDEN, "GaN_master_20kV.npz")}
PC = (0.50, 0.50, 0.55)
TILT = 70.0
# the master's point group: fold of the axis c, inversion (only even degrees), a 2-fold axis along y
FOLD = {"ni": 4, "gan": 2}
EVEN = {"ni": True, "gan": False}
Y2 = {"ni": True, "gan": False}
RAW = {"u8": torch.uint8, "u16": torch.uint16, "f32": torch.float32}
RAW_BYTES = {"u8": 1, "u16": 2, "f32": 4}
NO_FILTERS = {"static_background": "none", "dynamic_background": "none"}
FILTERS = {
    # what a scan gets by default: the dynamic background subtracted
    "dynamic": {"static_background": "none"},
    "none": NO_FILTERS,
    # the contrast chain: background divided out, CLAHE, band pass
    "contrast": {"static_background": "none", "dynamic_background": "divide", "clahe": True, "bandpass": True},
}


def listed():
    return [
        # a live view during set-up of the microscope: the few patterns of the last frame, again and again
        {"name": "live view", "kind": "batch", "n": 3, "h": 60, "w": 60, "pixel": "u8", "phases": "ni", "L": 64, "iters": 8, "filters": "dynamic",
         "precision": "fp32"},
        # a whole small map from host memory with every setting at its default: static and dynamic
        # backgrounds, calibration against chance, acceptance, results on the host
        {"name": "scan", "kind": "scan", "rows": 71, "cols": 85, "h": 60, "w": 60, "pixel": "u8", "phases": "ni", "L": 64, "iters": 8},
        # the headline workload's chunk: patterns already normalized by the detector's software
        {"name": "chunk", "kind": "batch", "n": 4500, "h": 60, "w": 60, "pixel": "f32", "phases": "ni", "L": 64, "iters": 5, "filters": "none",
         "precision": "fp32"},
        # a dual-phase chunk: every pattern against both masters
        {"name": "two phases", "kind": "batch", "n": 2501, "h": 60, "w": 60, "pixel": "u8", "phases": "ni,gan", "L": 64, "iters": 5,
         "filters": "none", "precision": "fp32"},
        # the precision form's patterns: fine detector, high bandwidth
        {"name": "fine", "kind": "batch", "n": 1200, "h": 120, "w": 120, "pixel": "u16", "phases": "ni", "L": 96, "iters": 8, "filters": "dynamic",
         "precision": "fp32"},
        # the same with the 16-bit products
        {"name": "fine, 16-bit products", "kind": "batch", "n": 1200, "h": 120, "w": 120, "pixel": "f32", "phases": "ni", "L": 96, "iters": 8,
         "filters": "none", "precision": "bf16"},
        # the filters alone: a chunk as the camera sends it, an odd count
        {"name": "filters", "kind": "prep", "n": 5003, "h": 60, "w": 60, "pixel": "u8", "filters": "dynamic"},
        # large frames (the blur goes by boxes, the images through global memory)
        {"name": "filters, large frames", "kind": "prep", "n": 160, "h": 240, "w": 320, "pixel": "u16", "filters": "dynamic"},
        # the contrast chain on odd frames
        {"name": "filters, contrast", "kind": "prep", "n": 1001, "h": 75, "w": 83, "pixel": "f32", "filters": "contrast"},
        # harmonics for a caller's own search (invariants, dictionaries): odd frames, ragged count
        {"name": "coefficients", "kind": "coefficients", "n": 3001, "h": 60, "w": 80, "L": 64},
        # a few large frames refined from a known neighbourhood
        {"name": "refine, large frames", "kind": "refine", "n": 40, "h": 240, "w": 320, "phases": "ni", "iters": 8},
        # the pattern-centre fit of a map's patterns
        {"name": "fit", "kind": "fit", "n": 4000, "h": 80, "w": 80, "iters": 20},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["scan", "batch", "batch", "batch", "prep", "prep", "coefficients", "refine", "fit"])
    h = rng.choice([40, 48, 53, 60, 60, 64, 75, 80, 96, 101, 120])
    w = rng.choice([h, h, h + rng.randrange(0, 24)])
    pixel = rng.choice(["u8", "u16", "f32"])
    L = rng.choice([24, 32, 40, 48, 50, 55, 63, 64, 64, 72, 88, 96])
    if kind == "scan":
        c = {"kind": kind, "rows": rng.randrange(4, 60), "cols": rng.randrange(5, 80), "h": min(h, 80), "w": min(w, 90), "pixel": pixel, "phases": "ni",
             "L": min(L, 64), "iters": 8}
    elif kind == "batch":
        ph = rng.choice(["ni", "ni", "ni,gan"])
        if ph != "ni":
            L = min(L, 64)
        prec = rng.choice(["fp32", "fp32", "fp32", "fp16", "bf16"])
        c = {"kind": kind, "n": _log_int(rng, 1, 4500), "h": h, "w": w, "pixel": pixel, "phases": ph, "L": L, "iters": rng.choice([5, 8]),
             "filters": rng.choice(["none", "dynamic"]), "precision": prec}
    elif kind == "prep":
        if rng.random() < 0.35:
            h, w = rng.randrange(121, 241), rng.randrange(121, 321)
        c = {"kind": kind, "n": _log_int(rng, 1, 5000), "h": h, "w": w, "pixel": pixel, "filters": rng.choice(["dynamic", "dynamic", "contrast"])}
    elif kind == "coefficients":
        c = {"kind": kind, "n": _log_int(rng, 1, 3000), "h": h, "w": w, "L": L}
    elif kind == "refine":
        if rng.random() < 0.4:
            h, w = rng.randrange(121, 241), rng.randrange(121, 321)
        c = {"kind": kind, "n": _log_int(rng, 1, 4000), "h": h, "w": w, "phases": rng.choice(["ni", "ni,gan"]), "iters": rng.choice([5, 8])}
    else:
        c = {"kind": kind, "n": _log_int(rng, 8, 4000), "h": min(h, 80), "w": min(w, 80), "iters": 20}
    # at most the pixels and the correlation work of the listed ones
    if "n" in c:
        most = {"prep": 12e6, "refine": 3e6, "batch": 16e6, "coefficients": 14e6, "fit": 25e6}[kind]
        c["n"] = max(1, min(c["n"], int(most / (c["h"] * c["w"]))))
        if kind in ("batch", "coefficients"):
            k = (64.0 / L) ** 3 if L > 64 else 1.0
            c["n"] = max(1, min(c["n"], int((2500 if c.get("phases") == "ni,gan" else 4500) * k)))
    return c


# ── what a program keeps: one engine (or Solver) a configuration ──

_KEPT = {}


def _setup(c):
    return (c["kind"] == "scan", c.get("phases", "ni"), c.get("L", 64), c["h"], c["w"], c.get("precision", "fp32"), c.get("filters", "dynamic"),
            c.get("iters", 8))


def _engine(c):
    key = _setup(c)
    if key not in _KEPT:
        if len(_KEPT) > 24:
            _KEPT.clear()
        if c["kind"] == "scan":
            s = Solver()
            s.configure(bandwidth=c["L"], refine_iters=c["iters"])
            s.set_geometry(pc=PC, sample_tilt_deg=TILT, px_um=70.0 * 60 / c["h"], step_x_um=2.0, step_y_um=2.0)
            for p in c["phases"].split(","):
                s.add_phase(MASTERS[p])
            _KEPT[key] = s
        else:
            e = engine.Engine()
            e.settings.apply(bandwidth=c.get("L", 64), refine_iters=c.get("iters", 8), correlation_precision=c.get("precision", "fp32"),
                             **FILTERS[c.get("filters", "dynamic")])
            e.geo.pc, e.geo.sample_tilt_deg = PC, TILT
            for p in c.get("phases", "ni").split(","):
                e.add_phase(MASTERS[p])
            e.set_patterns(np.zeros((1, 1, c["h"], c["w"]), np.uint8))
            _KEPT[key] = e
    return _KEPT[key]


# ── inputs: patterns of random orientations from the masters, noise, pixel types ──

_SHEETS = {}


def _sheets(phase):
    """The phase's master as stored: [2, side, side] float32 on the GPU, zero mean and unit deviation."""
    if phase not in _SHEETS:
        from zebsdsolve_amd import master
        raw = torch.as_tensor(np.asarray(master.load(MASTERS[phase]).raw, np.float32)).cuda()
        _SHEETS[phase] = (raw - raw.mean()) / raw.std()
    return _SHEETS[phase]


def _frame_vectors():
    a = math.radians(0.0 - TILT)
    s, c = math.sin(a), math.cos(a)
    R = np.array([[-s, 0, c], [0, 1, 0], [-c, 0, -s]])
    return R


def _positions(rng, n, h, w, spread):
    pc = np.asarray(PC)[None] + rng.uniform(-spread, spread, (n, 3))
    v = np.stack([0.5 - pc[:, 1] * h, 0.5 - pc[:, 0] * w, pc[:, 2] * h], 1)
    return v @ _frame_vectors().T


def _square(v):
    """Directions [..., 3] to the equal-area square's coordinates in [-1, 1]."""
    ax, ay = v[..., 0].abs(), v[..., 1].abs()
    xn = torch.sqrt(torch.clamp(math.pi / 2 * (ax * ax + ay * ay) / (1 + v[..., 2].abs()), min=0))
    big, small = torch.maximum(ax, ay), torch.minimum(ax, ay)
    t = 4 / math.pi * xn * torch.atan(small / torch.clamp(big, min=1e-30))
    u, w = torch.where(ax >= ay, xn, t), torch.where(ax >= ay, t, xn)
    k = 1 / math.sqrt(math.pi / 2)
    return torch.where(v[..., 0] < 0, -u, u) * k, torch.where(v[..., 1] < 0, -w, w) * k


def _render(phase, q, t, h, w):
    """Patterns [n, h, w] float32: the master along every pixel's ray turned by q (n, 4)."""
    s = _sheets(phase)
    side = s.shape[-1]
    R = torch.as_tensor(_frame_vectors(), dtype=torch.float32, device="cuda")
    rr, cc = torch.meshgrid(torch.arange(h, device="cuda", dtype=torch.float32), torch.arange(w, device="cuda", dtype=torch.float32), indexing="ij")
    plane = (rr[..., None] * R[:, 0] + cc[..., None] * R[:, 1]).reshape(1, -1, 3)
    out = torch.empty((len(q), h * w), device="cuda")
    step = max(1, (1 << 24) // (h * w))
    for a in range(0, len(q), step):
        qa, ta = (torch.as_tensor(x[a:a + step], dtype=torch.float32, device="cuda") for x in (q, t))
        u = plane + ta[:, None]
        u = u / u.norm(dim=-1, keepdim=True)
        qv = qa[:, None, 1:].expand_as(u)
        tt = 2 * torch.linalg.cross(qv, u)
        v = u + qa[:, None, :1] * tt + torch.linalg.cross(qv, tt)
        x, y = _square(v)
        fj, fi = ((z + 1) * 0.5 * (side - 1) for z in (x, y))
        j, i = (torch.clamp(z.long(), 0, side - 2) for z in (fj, fi))
        o = (v[..., 2] < 0).long() * side * side + i * side + j
        f = s.reshape(-1)
        tj, ti = fj - j, fi - i
        out[a:a + step] = ((f[o] * (1 - tj) + f[o + 1] * tj) * (1 - ti) + (f[o + side] * (1 - tj) + f[o + side + 1] * tj) * ti)
    return out.view(-1, h, w)


def _patterns(c, seed, n, spread):
    """(raw patterns on the GPU, orientations, positions, phases) of n patterns, from the seed alone:
    simulated patterns, for camera pixels with a detector's uneven background, Poisson counts."""
    rng = np.random.default_rng(seed)
    h, w = c["h"], c["w"]
    q = rot.qstd(rng.normal(size=(n, 4)))
    t = _positions(rng, n, h, w, spread)
    names = c.get("phases", "ni").split(",")
    which = (rng.random(n) >= 0.7).astype(np.int64) if len(names) > 1 else np.zeros(n, np.int64)
    sims = torch.empty((n, h, w), device="cuda")
    for k, name in enumerate(names):
        sel = np.flatnonzero(which == k)
        if len(sel):
            sims[torch.from_numpy(sel).cuda()] = _render(name, q[sel], t[sel], h, w)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    pixel = c.get("pixel", "f32")
    sig = torch.clamp(1 + 0.25 * sims, min=0.05)
    if c.get("filters", "none") != "none" or c["kind"] == "scan":
        y, x = torch.meshgrid(torch.linspace(-1, 1, h, device="cuda"), torch.linspace(-1, 1, w, device="cuda"), indexing="ij")
        sig = sig * torch.exp(-0.8 * ((x - 0.1) ** 2 + (y + 0.15) ** 2)) * (0.8 + 0.4 * torch.rand((n, 1, 1), generator=gen, device="cuda"))
    raw = torch.poisson(sig * (100.0 if pixel == "u8" else 400.0), generator=gen)
    if pixel == "u8":
        raw = raw.clamp(0, 255).to(torch.uint8)
    elif pixel == "u16":
        raw = raw.clamp(0, 65535).to(torch.int32).to(torch.uint16)
    return raw.contiguous(), q, t.astype(np.float32), which


def _items(t, n):
    return torch.from_numpy(np.concatenate([t, np.arange(n, dtype=np.float32)[:, None]], 1).astype(np.float32)).cuda()


def _normalized(raw, mask):
    """Zero mean and unit norm under the mask, zero outside (plain torch)."""
    m = _mask(raw.shape[1], raw.shape[2], mask).to(raw.device)
    x = raw.float()
    x = torch.where(m, x - (x * m).sum((1, 2), keepdim=True) / m.sum(), torch.zeros_like(x))
    return (x / x.square().sum((1, 2), keepdim=True).sqrt()).contiguous()


def _mask(h, w, mask):
    r, c = torch.meshgrid(torch.arange(h, dtype=torch.float64), torch.arange(w, dtype=torch.float64), indexing="ij")
    return (r - mask[0]) ** 2 + (c - mask[1]) ** 2 <= mask[2]


def _turned(q, rng, lo, hi):
    """Orientations turned by lo to hi degrees about random axes."""
    ax = rng.normal(size=(len(q), 3))
    ax /= np.linalg.norm(ax, axis=1, keepdims=True)
    return rot.qstd(rot.qmul(rot.so3_exp(ax * np.radians(rng.uniform(lo, hi, (len(q), 1)))), q))


def prepare(case, seed):
    c = dict(case)
    lib = nat.load()
    st = {"case": c, "lib": lib}
    if c["kind"] == "scan":
        n = c["rows"] * c["cols"]
        s = _engine(c)
        raw = _patterns(c, seed, n, 0.0)[0]
        st["solver"] = s
        st["scan"] = raw.cpu().numpy().reshape(c["rows"], c["cols"], c["h"], c["w"])
        if c["pixel"] == "u16":
            st["scan"] = st["scan"].astype(np.uint16)
        if s._e.patterns is None:
            s.set_patterns(st["scan"])
            s.index_cells([0])  # the tables of this geometry
        return st
    e = st["engine"] = _engine(c)
    n = c["n"]
    raw, q, t, which = _patterns(c, seed, n, 0.01)
    if c["kind"] == "batch":
        st["raw"], st["items"] = raw, _items(t, n)
        if not hasattr(e, "_tables_made"):
            e.run_batch(raw[:1], st["items"][:1])
            e._tables_made = True
        return st
    mask = e.mask_tuple()
    if c["kind"] == "prep":
        st["raw"], st["mask"] = raw, (nat.ctypes.c_float * 3)(*mask)
        o = nat.PrepOpts()
        s = e.settings
        o.dynamic = {"none": 0, "subtract": 1, "divide": 2}[s["dynamic_background"]]
        o.dynamic_sigma = float(s["dynamic_sigma"]) * c["w"]
        o.clahe, o.clahe_grid, o.clahe_bins, o.clahe_clip = int(s["clahe"]), int(s["clahe_grid"]), int(s["clahe_bins"]), float(s["clahe_clip"])
        o.bandpass, o.bp_fine, o.bp_coarse = int(s["bandpass"]), float(s["bp_fine"]), float(s["bp_coarse"])
        st["opts"] = o
        need = int(lib.zb_prep_workspace(n, c["h"], c["w"], nat.ctypes.byref(o)))
        st["work"] = torch.empty((max(need, 8),), dtype=torch.uint8, device="cuda")
        st["out"] = torch.empty((n, c["h"], c["w"]), device="cuda")
        return st
    st["frame"] = e.frame()
    st["pats"] = _normalized(raw, mask)
    if c["kind"] == "coefficients":
        b = st["band"] = e.band(c["L"])
        st["items"] = _items(t, n)
        st["alm"] = torch.empty((n, b.host.pairs, 2), device="cuda")
        st["stats"] = torch.empty((n, 4), device="cuda")
        st["work"] = torch.empty((int(lib.zb_sh_workspace(b.c, n)),), dtype=torch.uint8, device="cuda")
        return st
    rng = np.random.default_rng([seed, 1])
    if c["kind"] == "refine":
        st["items"] = _items(t, n)
        st["phases"] = []
        for pi in range(len(e.phases)):
            seeds = torch.zeros((n, 8), device="cuda")
            seeds[:, :4] = torch.from_numpy(_turned(q, rng, 0.3, 1.5).astype(np.float32)).cuda()
            st["phases"].append((e.baked(pi)[1][0], e.grad_half(pi), e.phases[pi].master.side, seeds, torch.empty((n,), dtype=torch.int32, device="cuda")))
        st["records"] = torch.empty((len(e.phases), n, 8), device="cuda")
        st["work"] = torch.empty((nat.REFINE_QUEUE_BYTES,), dtype=torch.uint8, device="cuda")
        o = st["opts"] = nat.RefineOpts()
        o.iters, o.max_step, o.scale0, o.scale_min, o.scale_max, o.nmi_bins, o.stamp = c["iters"], math.radians(2.0), 1.0, 0.02, 1e4, 16, 7
        return st
    # fit: the crystal 0.3 to 1.5 degrees off, the detector up to 0.01 of the pattern's height
    st["field"] = fit.PoseField(e, 0, st["pats"])
    off = rng.uniform(-0.01, 0.01, (n, 3)) * c["h"]
    st["poses"] = torch.from_numpy(np.concatenate([t + off, np.arange(n)[:, None], _turned(q, rng, 0.3, 1.5)], 1).astype(np.float32)).cuda()
    return st


def run(st):
    c, lib = st["case"], st["lib"]
    kind = c["kind"]
    if kind == "scan":
        return st["solver"].set_patterns(st["scan"]).index()
    if kind == "batch":
        # (the last of a record's eight values is the call's running number)
        return st["engine"].run_batch(st["raw"], st["items"])[0][..., :7]
    stream = engine.stream_ptr()
    if kind == "prep":
        nat.check(lib.zb_prep_work(st["raw"].data_ptr(), {"u8": 0, "u16": 1, "f32": 2}[c["pixel"]], c["n"], c["h"], c["w"], st["mask"],
                                   nat.ctypes.byref(st["opts"]), st["work"].data_ptr(), st["work"].numel(), st["out"].data_ptr(), stream), "prep")
        return st["out"]
    if kind == "coefficients":
        nat.check(lib.zb_sh_coefficients(st["band"].c, st["frame"], st["pats"].data_ptr(), st["items"].data_ptr(), c["n"], nat.FLAG_CENTER | nat.FLAG_NORM,
                                         st["work"].data_ptr(), st["work"].numel(), st["alm"].data_ptr(), st["stats"].data_ptr(), stream), "coefficients")
        return {"alm": st["alm"], "stats": st["stats"]}
    if kind == "refine":
        n = c["n"]
        for _, _, _, seeds, order in st["phases"]:
            nat.check(lib.zb_refine_order(st["frame"], st["items"].data_ptr(), seeds.data_ptr(), 8, n, order.data_ptr(), stream), "order")
        arr = (nat.RefinePhase * len(st["phases"]))(*[
            nat.RefinePhase(sh.data_ptr(), gh.data_ptr(), side, seeds.data_ptr(), 8, order.data_ptr(), st["records"][k].data_ptr())
            for k, (sh, gh, side, seeds, order) in enumerate(st["phases"])])
        nat.check(lib.zb_refine_phases(arr, len(arr), st["frame"], st["pats"].data_ptr(), st["items"].data_ptr(), n, st["opts"], 0, st["work"].data_ptr(),
                                       st["work"].numel(), stream), "refine")
        return st["records"]
    poses, ncc, state = fit.fit6(st["field"], st["poses"], iters=c["iters"], tol=1e-5)
    return {"poses": poses, "ncc": ncc, "state": state}


# ── the work a pass cannot do without ──

def _fft_size(L):
    n = 16
    while n < 2 * L - 1:
        n *= 2
    return n


def _masked(h, w):
    r = 0.5 * min(h, w)
    return int(_mask(h, w, (0.5 * (h - 1), 0.5 * (w - 1), r * r)).sum())


def _refine_flops(c, iters):
    # 120 a masked pixel and pass: ray, rotation, map, four texels of four values, 19 sums
    return 120.0 * (iters + 2) * _masked(c["h"], c["w"])


def _sphere_flops(L):
    n = _fft_size(L)
    return 5.0 * 2 * n * math.log2(2 * n) * n / 2 + 4.0 * L * (L + 1) / 2 * n / 2


def _corr(phase, L):
    """(operations a pattern, the master's tables' bytes) of the search: the contraction with the
    master's weights for each (b, m') as one product, the transforms along c and a."""
    n = _fft_size(L)
    nc = n // FOLD[phase]
    rows = n // 4 + 1 if Y2[phase] else n // 2 + 1
    slots = sum(-(-(L - m) // 2) if EVEN[phase] else L - m for m in range(L))
    return 8.0 * slots * nc * rows + 5.0 * (n / 2) * math.log2(n / 2) * rows * nc, 8.0 * slots * nc * rows + 4.0 * rows * n * nc


def _filter_flops(c):
    """Separable sums by the filters' taps: 4 a tap and pixel (rows and columns); from 12 pixels of
    deviation the sums go by boxes, some 60 a pixel."""
    px = c["h"] * c["w"]
    sig = {"none": [], "dynamic": [0.15 * c["w"]], "contrast": [0.15 * c["w"], 1.0, 8.0]}[c.get("filters", "dynamic")]
    return sum(px * (4.0 * (2 * math.ceil(3 * s) + 1) if s < 12 else 60.0) for s in sig) + 6.0 * px + (20.0 * px if c.get("filters") == "contrast" else 0)


def work(case):
    c = dict(case)
    px = c["h"] * c["w"]
    side = {"ni": 501, "gan": 301}
    if c["kind"] in ("scan", "batch"):
        n = c.get("n") or c["rows"] * c["cols"]
        names = c["phases"].split(",")
        f = _sphere_flops(c["L"]) + _filter_flops(c) + len(names) * _refine_flops(c, c["iters"])
        b = n * (px * RAW_BYTES[c["pixel"]] + 16.0 + 32.0 * len(names))
        for p in names:
            f += _corr(p, c["L"])[0]
            b += _corr(p, c["L"])[1] + 12.0 * 2 * side[p] ** 2
        return {"bytes": b, "flops": n * f}
    n = c["n"]
    if c["kind"] == "prep":
        return {"bytes": float(n) * px * (RAW_BYTES[c["pixel"]] + 4), "flops": n * _filter_flops(c)}
    if c["kind"] == "coefficients":
        pairs = c["L"] * (c["L"] + 1) // 2
        return {"bytes": n * (4.0 * px + 16 + 8 * pairs + 16) + 4.0 * pairs * _fft_size(c["L"]) / 2, "flops": n * _sphere_flops(c["L"])}
    if c["kind"] == "refine":
        names = c["phases"].split(",")
        return {"bytes": n * (4.0 * px + 16 + len(names) * 64) + sum(24.0 * 2 * side[p] ** 2 for p in names),
                "flops": float(n) * len(names) * _refine_flops(c, c["iters"])}
    # the fit: the start and about eight of the steps before a pose has converged, 43 sums each
    return {"bytes": n * (4.0 * px + 80) + 16.0 * 2 * side["ni"] ** 2, "flops": n * 9 * 200.0 * _masked(c["h"], c["w"])}


# ── the same in 64 bits ──

def _cells(n, s):
    """Centres and widths of the blur's cells of s pixels, three more each way (those are whole)."""
    k = -(-n // s)
    j = np.arange(-3, k + 3)
    lo = j * s
    hi = np.where((j >= 0) & (lo < n), np.minimum(lo + s, n), lo + s)
    return 0.5 * (lo + hi - 1), hi - lo, k


def _blur_axis(n, sigma):
    """One axis of the Gaussian as two matrices [n, n]: of the values and of the counts."""
    s = int(sigma // 6)
    if s < 2:
        d = np.arange(n)
        r = max(1, math.ceil(3 * sigma))
        g = np.exp(-(d[:, None] - d[None]) ** 2 / (2 * sigma * sigma)) * (abs(d[:, None] - d[None]) <= r)
        return g
    cs = math.sqrt(sigma * sigma - s * s - (s * s - 1) / 12)
    reach = math.ceil(4 * cs)
    mid, wide, k = _cells(n, s)
    box = (np.arange(n)[None] // s == np.arange(k)[:, None]).astype(np.float64)
    inner = mid[3:3 + k]
    j = np.arange(k)
    near = (j[None] >= np.floor((mid[:, None] - reach) / s)) & (j[None] <= np.floor((mid[:, None] + reach) / s))
    coarse = np.exp(-(inner[None] - mid[:, None]) ** 2 / (2 * cs * cs)) * near
    own = np.arange(n) // s
    at = np.arange(k + 6)
    spread = wide[None] * np.exp(-(np.arange(n)[:, None] - mid[None]) ** 2 / (2.0 * s * s)) * (abs(at[None] - 3 - own[:, None]) <= 3)
    return spread @ coarse @ box


def _gauss(x, sigma):
    # each pixel's sum of weights; the counts of the boxes travel with the sums
    gy, gx = (torch.as_tensor(_blur_axis(k, sigma), device=x.device) for k in x.shape[1:])
    one = torch.ones(x.shape[1:], dtype=torch.float64, device=x.device)
    return (gy @ x @ gx.T.contiguous()) / (gy @ one @ gx.T.contiguous())


def _clahe(x, T, B, clip):
    n, h, w = x.shape
    lo, hi = x.amin((1, 2), keepdim=True), x.amax((1, 2), keepdim=True)
    x = (x - lo) / (hi - lo).clamp(min=1e-20)
    ph, pw = -h % T, -w % T
    th, tw = (h + ph) // T, (w + pw) // T
    iy, ix = ((torch.arange(k + p, device=x.device) - p).abs() for k, p in ((h, ph), (w, pw)))
    bins = (x.clamp(0, 1) * (B - 1)).long()[:, iy][:, :, ix]
    tile = (torch.arange(h + ph, device=x.device) // th)[:, None] * T + (torch.arange(w + pw, device=x.device) // tw)[None]
    at = torch.arange(n, device=x.device)[:, None, None] * (T * T * B) + tile[None] * B + bins
    hist = torch.bincount(at.reshape(-1), minlength=n * T * T * B).double().view(n, T * T, B)
    total = float(th * tw)
    cut = hist.clamp(max=max(clip * total / B, 1.0))
    lost = total - cut.sum(-1, keepdim=True)
    rest = torch.floor(lost - B * torch.floor(lost / B))
    cut = cut + (lost - rest) / B + (torch.arange(B, device=x.device) < rest)
    cdf = (cut.cumsum(-1) / total).clamp(0, 1)
    gy, gx = ((torch.arange(k, device=x.device, dtype=torch.float64) + 0.5) / k * (T - 1) for k in (h, w))
    y0, x0 = gy.long(), gx.long()
    fy, fx = (gy - y0)[None, :, None], (gx - x0)[None, None]
    bf = x.clamp(0, 1) * (B - 1)
    b0 = torch.floor(bf).clamp(0, B - 2).long()
    fb = bf - b0

    def table(ty, tx):
        k = torch.arange(n, device=x.device)[:, None, None] * (T * T * B) + (ty.clamp(max=T - 1)[:, None] * T + tx.clamp(max=T - 1)[None])[None] * B + b0
        f = cdf.reshape(-1)
        return f[k] * (1 - fb) + f[k + 1] * fb

    return (table(y0, x0) * (1 - fx) + table(y0, x0 + 1) * fx) * (1 - fy) + (table(y0 + 1, x0) * (1 - fx) + table(y0 + 1, x0 + 1) * fx) * fy


def _exact_prep(st):
    c, o = st["case"], st["opts"]
    x = st["raw"].to(torch.int32).double() if c["pixel"] == "u16" else st["raw"].double()
    if o.dynamic:
        b = _gauss(x, float(o.dynamic_sigma))
        x = x - b if o.dynamic == 1 else x / b.clamp(min=1e-6)
    if o.clahe:
        x = _clahe(x, o.clahe_grid, o.clahe_bins, float(o.clahe_clip))
    if o.bandpass:
        x = (_gauss(x, float(o.bp_fine)) if o.bp_fine > 0.05 else x) - _gauss(x, float(o.bp_coarse))
    m = _mask(c["h"], c["w"], [float(v) for v in st["mask"]]).cuda()
    x = torch.where(m, x - (x * m).sum((1, 2), keepdim=True) / m.sum(), torch.zeros_like(x))
    return x / x.square().sum((1, 2), keepdim=True).sqrt()


def _legendre(L, x):
    """Orthonormal associated Legendre functions (Condon-Shortley) P[l, m] at x, by recurrence in l."""
    s = np.sqrt(1 - x * x)
    P = np.zeros((L, L, len(x)))
    P[0, 0] = math.sqrt(0.25 / math.pi)
    for m in range(L):
        if m:
            P[m, m] = -math.sqrt((2 * m + 1) / (2.0 * m)) * s * P[m - 1, m - 1]
        if m + 1 < L:
            P[m + 1, m] = math.sqrt(2 * m + 3.0) * x * P[m, m]
        for k in range(m + 2, L):
            a = math.sqrt((4.0 * k * k - 1) / (k * k - m * m))
            b = math.sqrt(((k - 1.0) ** 2 - m * m) / (4.0 * (k - 1) ** 2 - 1))
            P[k, m] = a * (x * P[k - 1, m] - b * P[k - 2, m])
    return P


def _exact_coefficients(st):
    c = st["case"]
    L, h, w = c["L"], c["h"], c["w"]
    n = _fft_size(L)
    ct, wq = np.polynomial.legendre.leggauss(n)
    ct, wq = ct[::-1].copy(), wq[::-1].copy()
    P = torch.as_tensor(_legendre(L, ct), device="cuda")
    phi = 2 * math.pi * np.arange(2 * n) / (2 * n)
    sn = np.sqrt(1 - ct * ct)
    d = torch.as_tensor(np.stack([sn[:, None] * np.cos(phi), sn[:, None] * np.sin(phi), np.repeat(ct[:, None], 2 * n, 1)], -1), device="cuda").reshape(-1, 3)
    fr = st["frame"]
    c0, c1, c2 = (torch.tensor(list(v), dtype=torch.float64, device="cuda") for v in (fr.c0, fr.c1, fr.c2))
    mask = [float(v) for v in fr.mask]
    wt = torch.as_tensor(wq, device="cuda")
    alms, stats = [], []
    m = torch.cat([torch.full((L - k,), k) for k in range(L)]).cuda()
    k = torch.where(m == 0, 1.0, 2.0).double()
    nd, p0, p1 = d @ c2, d @ c0, d @ c1
    for a in range(0, c["n"], 32):
        it = st["items"][a:a + 32].double()
        t0, t1, t2 = (it[:, :3] @ v for v in (c0, c1, c2))
        s = t2[:, None] / nd.clamp(min=1e-12)[None]
        r, q = s * p0 - t0[:, None], s * p1 - t1[:, None]
        ok = (nd > 1e-4)[None] & (r >= 0) & (r <= h - 1) & (q >= 0) & (q <= w - 1)
        ok &= (r - mask[0]) ** 2 + (q - mask[1]) ** 2 <= mask[2]
        r, q = (torch.where(ok, v, torch.zeros_like(v)) for v in (r, q))
        i, j = r.long().clamp(max=h - 2), q.long().clamp(max=w - 2)
        f = st["pats"].double().view(c["n"], -1)[it[:, 3].long()] if c["n"] <= 32 else st["pats"].view(c["n"], -1)[it[:, 3].long()].double()
        at = i * w + j
        fi, fj = r - i, q - j
        v = (f.gather(1, at) * (1 - fj) + f.gather(1, at + 1) * fj) * (1 - fi) + (f.gather(1, at + w) * (1 - fj) + f.gather(1, at + w + 1) * fj) * fi
        g = ok.double()
        v = (v * g).view(-1, n, 2 * n)
        g = g.view(-1, n, 2 * n)
        sv, sw = (v.sum(2) @ wt), (g.sum(2) @ wt)
        mean = sv / sw.clamp(min=1e-20)
        F = torch.fft.rfft((v - mean[:, None, None] * g), dim=2)[:, :, :L] * wt[None, :, None] * (2 * math.pi / (2 * n))
        full = torch.stack([torch.einsum("bym,lmy->blm", F.real, P), torch.einsum("bym,lmy->blm", F.imag, P)], -1)
        alm = torch.cat([full[:, mm:, mm] for mm in range(L)], 1)
        nrm = (k[None, :, None] * alm.square()).sum((1, 2)).sqrt()
        alm = alm / nrm[:, None, None]
        alms.append(alm)
        stats.append(torch.stack([sw * math.pi / n, mean, nrm, alm[:, 0, 0]], 1))
    return {"alm": torch.cat(alms), "stats": torch.cat(stats)}


def exact(case, seed):
    """Orientations come from a search for a maximum and from steps that are kept or refused, scores
    from histograms: none of them has a value of its own in 64 bits. The filters and the harmonics do."""
    if case["kind"] == "prep":
        return _exact_prep(prepare(case, seed))
    if case["kind"] == "coefficients":
        return _exact_coefficients(prepare(case, seed))
    return None
