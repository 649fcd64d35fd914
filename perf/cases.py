"""Performance cases: calls a user of ctbangbang_amd makes, over the sizes, scanners and options it ships.

Kinds of case
  volume       a whole reconstruction of device-resident scans: ``Context.reconstruct_dev`` (one scan) or
               ``Context.reconstruct_batch_dev`` (several), from raw readings to the thickened stack in HU
  adaptive     the adaptive raw-data filter of one block's pull (``Context.adaptive_filter_dev``)
  rebin        fan-to-parallel rebinning + ramp filter of one block (``Context.rebin_filter_dev``)
  rows         the ramp filter alone on rows a program already holds (``Context.filter_rows_dev``)
  backproject  weighted backprojection of one 32-slice block (``Context.backproject_dev``)
  finalize     slice thickening + HU, then int16 stored values (``Context.finalize_dev``, ``hu_to_int16_dev``)

Scans are synthetic (the package's analytic phantom with Poisson noise); a stage that starts from filtered
projections gets an analytic sinogram of spheres with noise.  ``exact`` evaluates the same stage in FP64 torch.
"""
import math
import os
import tempfile
import weakref

import numpy as np
import torch

import ctbangbang_amd as cb
from ctbangbang_amd import PhantomParams, scans

# scanner: channels, projections per turn and focal position, filtered row length
SCANNERS = {"definitionas": (736, 1152), "sensation64": (672, 1160), "force": (920, 1400)}
FFS = {"none": (0, 0), "phi": (0, 1), "z": (1, 0), "both": (1, 1)}        # (z, phi)
FILTERS = {"fft32": cb.FILTER_FFT32, "f32": cb.FILTER_F32, "bf16x3": cb.FILTER_BF16X3, "f16x3": cb.FILTER_F16X3}
PI_BP = float(np.float32(3.1415368979))      # the backprojection's and preprocessing's pi constant
PI_RB = float(np.float32(3.1415926535897))   # the rebinning's
MU_WATER = 0.02


def scan(**kw):
    """Scan fields of a case with their usual values."""
    c = {"scanner": "definitionas", "rows": 64, "coll": 0.6, "ffs": "both", "pitch": 0.8, "nx": 512, "fov": 250.0,
         "slices": 40, "thickness": 3.0}
    c.update(kw)
    return c


def listed():
    return [
        # a short routine scan without a flying focal spot: the smallest whole reconstruction, one 32-slice block
        {"name": "volume_256_one_block", "kind": "volume", "scans": 1, "filter": "fft32", "bf16": False,
         "adaptive": False, "threshold": 0.0,
         **scan(rows=16, coll=1.2, ffs="none", pitch=1.0, nx=256, slices=16, thickness=1.0)},
        # the phi+z flying-focal-spot chest-length scan that the benchmark quotes: 512^2, seven blocks, adaptive filter on
        {"name": "volume_512_phi_z", "kind": "volume", "scans": 1, "filter": "fft32", "bf16": False,
         "adaptive": True, "threshold": 0.0, **scan()},
        # preprocessing alone with the per-view threshold (few samples are smoothed)
        {"name": "adaptive_phi_z", "kind": "adaptive", "threshold": 0.0, **scan()},
        # preprocessing by a protocol that prescribes the noise threshold (3e4 of 1e5 photons): the rays through
        # the patient are smoothed
        {"name": "adaptive_fixed_threshold", "kind": "adaptive", "threshold": 1.204,
         **scan(scanner="sensation64", ffs="z", pitch=1.0)},
        # sinogram preparation of one block, plain FP32 form
        {"name": "rebin_filter_phi_z", "kind": "rebin", "filter": "fft32", "bf16": False, **scan()},
        # sinogram preparation of one block, split-precision matrix-core filter and bfloat16 projections
        {"name": "rebin_filter_z_mixed", "kind": "rebin", "filter": "f16x3", "bf16": True,
         **scan(scanner="sensation64", ffs="z", pitch=1.0)},
        # filtering the rows of a single view (interactive use, one projection at a time)
        {"name": "rows_one_view", "kind": "rows", "scanner": "definitionas", "n_rows": 64, "filter": "fft32",
         "bf16": False},
        # rows of the widest shipped scanner, an odd number of them
        {"name": "rows_920_channels", "kind": "rows", "scanner": "force", "n_rows": 45001, "filter": "fft32",
         "bf16": False},
        # the split bfloat16 product on a ragged number of rows
        {"name": "rows_bf16x3", "kind": "rows", "scanner": "definitionas", "n_rows": 30011, "filter": "bf16x3",
         "bf16": False},
        # one block on a small matrix with a 16-row detector (a preview image)
        {"name": "backproject_256_16_rows", "kind": "backproject", "bf16": False,
         **scan(rows=16, coll=1.2, ffs="none", pitch=1.0, nx=256, slices=16, thickness=1.0)},
        # one block of a large matrix from bfloat16 projections
        {"name": "backproject_1024_bf16", "kind": "backproject", "bf16": True,
         **scan(coll=0.5, ffs="z", pitch=0.6, nx=1024, fov=400.0, slices=150, thickness=2.0)},
        # the final stack of a long scan, in HU and as stored values for DICOM
        {"name": "finalize_768_long", "kind": "finalize",
         **scan(nx=768, fov=360.0, pitch=1.0, slices=201, thickness=2.0)},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _draw_scan(rng, volume):
    scanner = rng.choice(sorted(SCANNERS))
    ffs = rng.choice(sorted(FFS))
    rows, coll = rng.choice([(16, 1.2), (32, 0.6), (32, 1.2), (64, 0.5), (64, 0.6)])
    nx = 16 * int(_log_uniform(rng, 8, 33 if volume else 65))            # 128 .. 512 (1024 for one block)
    fov = round(rng.uniform(180.0, min(500.0, 1.2 * nx)) if nx > 150 else 150.0, 1)
    thickness = round(rng.choice([1.0, 2.0, 3.0]) * rng.uniform(0.8, 1.2), 2)
    slices = int(_log_uniform(rng, 5, 60))
    return scan(scanner=scanner, ffs=ffs, rows=rows, coll=coll, pitch=round(rng.uniform(0.5, 1.5), 3), nx=nx, fov=fov,
                slices=slices, thickness=thickness)


def draw(rng):
    kind = rng.choice(["volume", "adaptive", "rebin", "rows", "backproject", "finalize"])
    if kind == "rows":
        mode = rng.choice(["fft32", "fft32", "f16x3", "bf16x3", "f32"])
        return {"kind": kind, "scanner": rng.choice(sorted(SCANNERS)), "filter": mode,
                "n_rows": int(_log_uniform(rng, 16, 60000 if mode != "f32" else 20000)), "bf16": rng.random() < 0.25}
    c = {"kind": kind, **_draw_scan(rng, kind == "volume")}
    if kind == "volume":
        c.update(scans=rng.choice([1, 1, 1, 2]), filter=rng.choice(["fft32", "fft32", "f16x3"]), bf16=False,
                 adaptive=rng.random() < 0.7, threshold=rng.choice([0.0, 0.0, 0.0, 1.204]))
        c["bf16"] = c["filter"] == "f16x3"
        # (within the cost of the largest listed case)
        while work(c)["flops"] > (6e11 if c["bf16"] else 1.2e12) and (c["scans"] > 1 or c["slices"] > 4 or c["bf16"]):
            if c["scans"] > 1:
                c["scans"] = 1
            elif c["slices"] > 4:
                c["slices"] //= 2
            else:
                c.update(filter="fft32", bf16=False)
    elif kind == "adaptive":
        c.update(threshold=rng.choice([0.0, 0.0, 1.204]))
    elif kind == "rebin":
        c.update(filter=rng.choice(["fft32", "fft32", "f16x3", "bf16x3"]), bf16=False)
        c["bf16"] = c["filter"] != "fft32"
        if c["bf16"] and c["rows"] == 64:
            c.update(rows=32, coll=1.2)
    elif kind == "backproject":
        c.update(bf16=rng.random() < 0.3)
    return c


# ---------------------------------------------------------------------------
# planning


def _tokens(c):
    z, phi = FFS[c["ffs"]]
    feed = round(c["pitch"] * c["rows"] * c["coll"], 4)
    margin = 2.6 * feed
    span = (c["slices"] - 1) * c["thickness"] + 2 * c["thickness"]
    turns = int(math.ceil((2 * margin + span + 32 * c["coll"]) / feed))
    t = scans.base_tokens()
    t.update({"Scanner": c["scanner"] + ".scanner", "Nrows": c["rows"], "CollSlicewidth": c["coll"], "Zffs": z,
              "Phiffs": phi, "PitchValue": feed, "Readings": turns * SCANNERS[c["scanner"]][1] * (1 << (z + phi)),
              "Nx": c["nx"], "Ny": c["nx"], "ReconFOV": c["fov"], "SliceThickness": c["thickness"],
              "StartPos": round(margin, 3), "NSlices": c["slices"],
              "EndPos": round(margin, 3) + (c["slices"] - 1) * c["thickness"], "AdaptiveFiltration": 1.0,
              "MuWater": MU_WATER})
    return t


class _Plan:
    """A planned scan: the metadata (block `block` current) and its prm tokens."""

    def __init__(self, c, block=None):
        self.tokens = _tokens(c)
        with tempfile.TemporaryDirectory() as d:
            prm = os.path.join(d, "scan.prm")
            cb.write_prm(prm, self.tokens)
            self.mr = cb.metadata_from_prm(prm)
        self.n_read = int(self.tokens["Readings"])
        self.frame = int(self.mr.cg.n_rows_raw * self.mr.cg.n_channels)
        cb.plan_block(self.mr, int(self.mr.ri.n_blocks) // 2 if block is None else block)
        self.sizes = cb.block_sizes(self.mr)
        weakref.finalize(self, cb.free_metadata, self.mr)

    def phantom(self, seed):
        pp = PhantomParams()
        pp.phantom_seed = 1000 + seed
        pp.noise_seed = 2000 + seed
        pp.n_random = 8
        pp.i0 = 1e5
        pp.scale_mm = 100.0
        pp.z_center = 0.5 * (self.tokens["StartPos"] + self.tokens["EndPos"])
        pp.mu_water = MU_WATER
        return pp

    def updates(self):
        total = 0.0
        for b in range(int(self.mr.ri.n_blocks)):
            cb.plan_block(self.mr, b)
            total += cb.block_sizes(self.mr).voxel_updates_block
        return total


# ---------------------------------------------------------------------------
# inputs

_contexts = weakref.WeakValueDictionary()


class _Handle:
    """The context a program keeps for its calls with one set of options."""

    def __init__(self, options):
        self.ctx = cb.Context(0)
        self.ctx.set_options(**options)


def _handle(**options):
    key = tuple(sorted(options.items()))
    h = _contexts.get(key)
    if h is None:
        h = _contexts[key] = _Handle(options)
    return h


def _floats(n):
    return torch.empty(int(n), dtype=torch.float32, device="cuda:0")


def _raw_pull(plan, h, seed):
    """Readings of the current block's pull, [n_proj_pull][rows][channels]."""
    raw = _floats(plan.sizes.raw_pull)
    h.ctx.synth_scan_dev(plan.mr, plan.phantom(seed), cb.pull_start(plan.mr), int(plan.mr.ri.n_proj_pull), raw)
    h.ctx.synchronize()
    return raw


def _filtered(n_views, n_rows, nos, seed):
    """Filtered projections of a few spheres with noise: second differences of their parallel projections."""
    g = torch.Generator(device="cuda:0").manual_seed(seed)
    r = np.random.RandomState(seed % (1 << 31))
    out = torch.randn((n_views, n_rows, nos), generator=g, device="cuda:0") * 0.02
    v = torch.arange(n_views, device="cuda:0", dtype=torch.float32)[:, None]
    ch = torch.arange(nos, device="cuda:0", dtype=torch.float32)[None, :]
    proj = torch.zeros((n_views, nos), device="cuda:0")
    for _ in range(6):
        rad, amp, ph = 0.05 + 0.15 * r.rand(), 0.3 * r.rand(), 6.28 * r.rand()
        s = (ch - nos / 2) / nos - amp * torch.sin(v * (6.28 / 1152) + ph)
        proj += (0.5 + r.rand()) * torch.sqrt(torch.clamp(rad * rad - s * s, min=0.0))
    sharp = torch.zeros_like(proj)
    sharp[:, 1:-1] = 40.0 * (2 * proj[:, 1:-1] - proj[:, :-2] - proj[:, 2:]) + proj[:, 1:-1]
    rows = 1.0 + 0.1 * torch.sin(torch.arange(n_rows, device="cuda:0", dtype=torch.float32) * 0.3)
    out += sharp[:, None, :] * rows[None, :, None]
    return out.reshape(-1)


def prepare(case, seed):
    k = case["kind"]
    s = {"kind": k, "case": case}
    if k == "volume":
        h = s["handle"] = _handle(filter_mode=FILTERS[case["filter"]], proj_dtype=int(case["bf16"]), mu_water=MU_WATER,
                                  adaptive_filter=int(case["adaptive"]), adaptive_threshold=case["threshold"])
        s["plans"], s["raws"], s["outs"] = [], [], []
        for i in range(case["scans"]):
            # (a batch: scans of uneven length)
            p = _Plan(dict(case, slices=max(3, case["slices"] // (i + 1))))
            raw = _floats(p.n_read * p.frame)
            h.ctx.synth_scan_dev(p.mr, p.phantom(seed + 100 * i), 0, p.n_read, raw)
            s["plans"].append(p)
            s["raws"].append(raw)
            s["outs"].append(_floats(p.sizes.final_stack))
        h.ctx.synchronize()
    elif k == "adaptive":
        p = s["plan"] = _Plan(case)
        s["handle"] = _handle(adaptive_filter=1, adaptive_threshold=case["threshold"])
        s["raw"] = _raw_pull(p, s["handle"], seed)
        s["out"] = torch.empty_like(s["raw"])
    elif k == "rebin":
        p = s["plan"] = _Plan(case)
        s["handle"] = _handle(filter_mode=FILTERS[case["filter"]], proj_dtype=int(case["bf16"]))
        s["raw"] = _raw_pull(p, s["handle"], seed)
        s["out"] = torch.empty(int(p.sizes.rebin), dtype=torch.bfloat16 if case["bf16"] else torch.float32, device="cuda:0")
    elif k == "rows":
        nch = SCANNERS[case["scanner"]][0]
        s["handle"] = _handle(filter_mode=FILTERS[case["filter"]], proj_dtype=int(case["bf16"]))
        s["n"], s["rows"] = 2 * nch, case["n_rows"]
        s["in"], s["taps"] = _row_inputs(case, seed)
        s["out"] = torch.empty(s["n"] * s["rows"], dtype=torch.bfloat16 if case["bf16"] else torch.float32, device="cuda:0")
    elif k == "backproject":
        p = s["plan"] = _Plan(case)
        s["handle"] = _handle(proj_dtype=int(case["bf16"]))
        s["in"] = _bp_input(p, case, seed)
        s["out"] = _floats(p.sizes.image_block)
    elif k == "finalize":
        p = s["plan"] = _Plan(case)
        s["handle"] = _handle(mu_water=MU_WATER)
        g = torch.Generator(device="cuda:0").manual_seed(seed)
        s["in"] = torch.rand(int(p.sizes.image_stack), generator=g, device="cuda:0") * (2 * MU_WATER)
        s["hu"] = _floats(p.sizes.final_stack)
        s["i16"] = torch.empty(int(p.sizes.final_stack), dtype=torch.int16, device="cuda:0")
    return s


def _row_inputs(case, seed):
    """Smooth line integrals with noise, and the scanner's apodised ramp filter."""
    nch = SCANNERS[case["scanner"]][0]
    n = 2 * nch
    g = torch.Generator(device="cuda:0").manual_seed(seed)
    x = torch.linspace(-1, 1, n, device="cuda:0")[None, :]
    width = 0.3 + 0.6 * torch.rand((case["n_rows"], 1), generator=g, device="cuda:0")
    rows = 4.0 * torch.sqrt(torch.clamp(1 - (x / width) ** 2, min=0.0))
    rows += 0.02 * torch.randn((case["n_rows"], n), generator=g, device="cuda:0")
    apod = 0.4 + 0.6 * ((seed % 7) / 6.0)
    taps = torch.from_numpy(cb.ramp_filter(n, 0.35, apod, 0.5 + 0.5 * ((seed % 5) / 4.0))).to("cuda:0")
    return rows.reshape(-1), taps


def _bp_input(p, case, seed):
    mr = p.mr
    x = _filtered(int(p.sizes.n_proj_out), int(mr.cg.n_rows), int(mr.cg.n_channels_oversampled), seed)
    return x.to(torch.bfloat16) if case["bf16"] else x


# ---------------------------------------------------------------------------
# one pass


def run(s):
    k, ctx = s["kind"], s["handle"].ctx
    if k == "volume":
        if len(s["plans"]) == 1:
            p = s["plans"][0]
            ctx.reconstruct_dev(p.mr, s["raws"][0], p.n_read, s["outs"][0])
        else:
            ctx.reconstruct_batch_dev([p.mr for p in s["plans"]], s["raws"], [p.n_read for p in s["plans"]], s["outs"])
        return s["outs"]
    if k == "adaptive":
        ctx.adaptive_filter_dev(s["plan"].mr, s["raw"], s["out"])
        return s["out"]
    if k == "rebin":
        ctx.rebin_filter_dev(s["plan"].mr, s["raw"], s["out"])
        return s["out"]
    if k == "rows":
        ctx.filter_rows_dev(s["taps"], s["n"], s["rows"], s["in"], s["out"])
        return s["out"]
    if k == "backproject":
        ctx.backproject_dev(s["plan"].mr, s["in"], s["out"])
        return s["out"]
    ctx.finalize_dev(s["plan"].mr, s["in"], s["hu"])
    ctx.hu_to_int16_dev(s["hu"], s["hu"].numel(), s["i16"])
    return {"hu": s["hu"], "stored": s["i16"]}


def work(case):
    """Bytes read and written once; 12 FLOP per voxel-update, 5 N log2 N per FFT-filtered row pair's transforms,
    2 n^2 per row of a matrix-product filter."""
    k = case["kind"]

    def filter_flops(n, rows, mode):
        length = 2 * n
        return rows * (5.0 * length * math.log2(length) if mode == "fft32" else 2.0 * n * n)

    if k == "rows":
        n, rows = 2 * SCANNERS[case["scanner"]][0], case["n_rows"]
        return {"bytes": float(rows * n * (4 + (2 if case["bf16"] else 4)) + 8 * n),
                "flops": filter_flops(n, rows, case["filter"])}
    if k == "volume":
        b = f = 0.0
        for i in range(case["scans"]):
            p = _Plan(dict(case, slices=max(3, case["slices"] // (i + 1))))
            lo, hi, used = 1 << 60, 0, 0.0
            n = int(p.mr.cg.n_channels_oversampled)
            for blk in range(int(p.mr.ri.n_blocks)):
                cb.plan_block(p.mr, blk)
                sz = cb.block_sizes(p.mr)
                start = cb.pull_start(p.mr)
                lo, hi = min(lo, max(0, start)), max(hi, min(p.n_read, start + int(p.mr.ri.n_proj_pull)))
                rows = (int(p.mr.cg.n_proj_turn) // 2) * sz.n_half_turns * int(p.mr.cg.n_rows)
                used += filter_flops(n, rows, case["filter"]) + 12.0 * sz.voxel_updates_block
            b += 4.0 * ((hi - lo) * p.frame + p.sizes.final_stack)
            f += used
        return {"bytes": b, "flops": f}
    p = _Plan(case)
    mr, sz = p.mr, p.sizes
    eb = 2 if case.get("bf16") else 4
    if k == "adaptive":
        return {"bytes": 8.0 * sz.raw_pull, "flops": 2.0 * sz.raw_pull}
    if k == "rebin":
        n = int(mr.cg.n_channels_oversampled)
        return {"bytes": 4.0 * sz.raw_pull + eb * float(sz.rebin),
                "flops": 6.0 * sz.rebin + filter_flops(n, sz.rebin // n, case["filter"])}
    if k == "backproject":
        views = (int(mr.cg.n_proj_turn) // 2) * sz.n_half_turns
        return {"bytes": float(eb * views * int(mr.cg.n_rows) * int(mr.cg.n_channels_oversampled) + 4 * sz.image_block),
                "flops": 12.0 * sz.voxel_updates_block}
    return {"bytes": 4.0 * sz.image_stack + 6.0 * sz.final_stack, "flops": 2.0 * sz.image_stack}


# ---------------------------------------------------------------------------
# the same in FP64


def exact(case, seed):
    k = case["kind"]
    if k == "rows":
        rows, taps = _row_inputs(case, seed)
        return _filter64(rows, taps, 2 * SCANNERS[case["scanner"]][0]).reshape(-1)
    if k == "volume":
        if case["scans"] > 1 or case["adaptive"]:
            return None             # (threshold decisions of the adaptive filter differ between FP32 and FP64)
        p = _Plan(case)
        if p.updates() > 1.5e10 or int(p.mr.ri.n_blocks) > 2:
            return None
        h = _handle(adaptive_filter=0)
        raw = _floats(p.n_read * p.frame)
        h.ctx.synth_scan_dev(p.mr, p.phantom(seed), 0, p.n_read, raw)
        h.ctx.synchronize()
        raw = raw.reshape(p.n_read, p.frame)
        taps = torch.from_numpy(cb.load_filter(p.mr)).to("cuda:0")
        blocks = []
        for b in range(int(p.mr.ri.n_blocks)):
            cb.plan_block(p.mr, b)
            s0, n = cb.pull_start(p.mr), int(p.mr.ri.n_proj_pull)
            win = torch.zeros((n, p.frame), device="cuda:0")
            lo, hi = max(s0, 0), min(s0 + n, p.n_read)
            win[lo - s0:hi - s0] = raw[lo:hi]
            reb = _rebin64(p.mr, win.reshape(-1))
            flt = _filter64(reb.reshape(-1), taps, int(p.mr.cg.n_channels_oversampled))
            blocks.append(_backproject64(p.mr, flt.reshape(reb.shape)))
        return [_finalize64(p.mr, torch.cat(blocks)).reshape(-1)]
    p = _Plan(case)
    if k == "adaptive":
        return _adaptive64(p.mr, _raw_pull(p, _handle(adaptive_filter=1), seed), case["threshold"])
    if k == "rebin":
        reb = _rebin64(p.mr, _raw_pull(p, _handle(adaptive_filter=1), seed))
        taps = torch.from_numpy(cb.load_filter(p.mr)).to("cuda:0")
        return _filter64(reb.reshape(-1), taps, int(p.mr.cg.n_channels_oversampled)).reshape(-1)
    if k == "backproject":
        if p.sizes.voxel_updates_block > 6.5e10:
            return None
        mr = p.mr
        x = _bp_input(p, case, seed).to(torch.float64)
        return _backproject64(mr, x.reshape(-1, int(mr.cg.n_rows), int(mr.cg.n_channels_oversampled))).reshape(-1)
    g = torch.Generator(device="cuda:0").manual_seed(seed)
    x = torch.rand(int(p.sizes.image_stack), generator=g, device="cuda:0") * (2 * MU_WATER)
    nxy = int(p.mr.rp.nx * p.mr.rp.ny)
    return {"hu": _finalize64(p.mr, x.reshape(-1, nxy)).reshape(-1), "stored": None}


def _filter64(rows, taps, n):
    """y[l] = sum_k taps[n + l - k] x[k] by a zero-padded FP64 FFT."""
    length = 4 * n
    spec = torch.fft.rfft(taps.double(), n=length)
    x = rows.reshape(-1, n)
    out = torch.empty(x.shape, dtype=torch.float64, device=x.device)
    for i in range(0, x.shape[0], 16384):
        y = torch.fft.irfft(torch.fft.rfft(x[i:i + 16384].double(), n=length) * spec, n=length)
        out[i:i + 16384] = y[:, n:2 * n]
    return out


def _maps64(mr):
    """Radial index and azimuthal offset per output channel and focal-spot set: (kind, bidx, aoff)."""
    cg = mr.cg
    nch, nos, n_ffs = int(cg.n_channels), int(cg.n_channels_oversampled), int(mr.ri.n_ffs)
    cc, db, rf, sdd = (float(v) for v in (cg.central_channel, cg.fan_angle_increment, cg.r_f, cg.src_to_det))
    turns = float(cg.n_proj_ffs) / (2 * PI_RB)
    da = sdd * rf * db / (4 * (sdd - rf))
    dr = sdd * float(mr.rp.coll_slicewidth) / (4 * (sdd - rf) * math.tan(float(cg.anode_angle)))

    def angle(x1, x2, y1, y2):
        return np.arcsin((x1 * y2 - x2 * y1) / (np.hypot(x1, x2) * np.hypot(y1, y2)))

    def beta_rk(a, r, ch):
        b0 = (ch - cc) * db
        return angle(-(rf + r), -a, -(sdd * np.cos(b0) + r), -(sdd * np.sin(b0) + a))

    def lookup(beta, lut):
        lo = np.argmax(lut[None, :] >= beta[:, None], axis=1)
        lo = np.where((lut[None, :] >= beta[:, None]).any(axis=1), lo, len(lut) - 1)
        lo = np.maximum(lo, 1)
        return lo - 1.0 + (beta - lut[lo - 1]) / (lut[lo] - lut[lo - 1])

    ch, c = np.arange(nch, dtype=np.float64), np.arange(nos, dtype=np.float64)
    if n_ffs == 1:
        beta = np.arcsin((c - 2 * cc) * (db / 2))
        return 0, [beta / db + cc], [beta * float(cg.n_proj_turn) / (2 * PI_RB)]
    if n_ffs == 2 and mr.rp.z_ffs == 1:
        bi, ao = [], []
        for fs, r in enumerate((-dr, dr)):
            beta = np.arcsin((c - 2 * cc) * (db / 2) * rf / (rf + r))
            bi.append(lookup(beta, beta_rk(0.0, r, ch)))
            ao.append((beta * turns + angle(rf, 0.0, rf + r, 0.0) * turns + fs) / 2)
        return 1, bi, ao
    spots = [(da, 0.0), (-da, 0.0)] if n_ffs == 2 else [(da, -dr), (-da, -dr), (da, dr), (-da, dr)]
    bi, ao = [], []
    for pr in range(len(spots) // 2):
        lut, off = np.empty(nos), np.empty(nos)
        for h in range(2):
            a, r = spots[2 * pr + h]
            lut[h::2] = beta_rk(a, r, ch)
            off[h::2] = (lut[h::2] * turns + angle(rf, 0.0, rf + r, a) * turns + 2 * pr + h) / n_ffs
        rfr = rf if n_ffs == 2 else rf + (-dr if pr == 0 else dr)
        beta = np.arcsin((c - 2 * cc) * (db / 2) * rf / rfr)
        bi.append(lookup(beta, lut))
        ao.append(off)
    return (2 if n_ffs == 2 else 3), bi, ao


def _rebin64(mr, raw):
    cg = mr.cg
    nch, nos, nrr, n_rows = (int(v) for v in (cg.n_channels, cg.n_channels_oversampled, cg.n_rows_raw, cg.n_rows))
    n_ffs, n_proj, add = int(mr.ri.n_ffs), int(mr.ri.n_proj_pull) // int(mr.ri.n_ffs), int(cg.add_projections)
    n_out = n_proj - 2 * add
    kind, bidx, aoff = _maps64(mr)
    raw = raw.reshape(n_proj, n_ffs, nrr, nch)
    dev = raw.device
    proj = torch.arange(n_out, device=dev, dtype=torch.float64)[:, None] + add

    def taps(x, n):
        x = x.clamp(0, n - 1)
        i0 = x.floor()
        return i0.long(), (i0.long() + 1).clamp(max=n - 1), x - i0

    def azimuthal(spot, ch, off):
        """Raw samples of channels ch (spots spot) interpolated at proj - off: [view][channel][row]."""
        p0, p1, f = taps(proj - off[None, :], n_proj)
        sp, chb = spot.expand_as(p0), ch.expand_as(p0)
        out = torch.empty((n_out, ch.numel(), nrr), dtype=torch.float64, device=dev)
        for v in range(0, n_out, 128):
            e = slice(v, v + 128)
            u0 = raw[p0[e], sp[e], :, chb[e]].double()
            out[e] = u0 + f[e][..., None] * (raw[p1[e], sp[e], :, chb[e]].double() - u0)
        return out

    res = torch.empty((n_out, n_rows, nos), dtype=torch.float64, device=dev)
    for st in range(len(bidx)):
        by = torch.from_numpy(bidx[st]).to(dev)
        ao = torch.from_numpy(aoff[st]).to(dev)
        if kind <= 1:
            c0, c1, fc = taps(by, nch)
            spot = torch.full_like(c0, st if kind == 1 else 0)
            lo, hi = azimuthal(spot, c0, ao), azimuthal(spot, c1, ao)
        else:
            m0, m1, fc = taps(by, nos)
            lo = azimuthal(2 * st + (m0 & 1), m0 >> 1, ao[m0])
            hi = azimuthal(2 * st + (m1 & 1), m1 >> 1, ao[m1])
        val = (lo + fc[None, :, None] * (hi - lo)).permute(0, 2, 1)
        if kind in (0, 2):
            res[:] = val
        else:
            res[:, (st ^ (1 if cg.reverse_row_interleave else 0))::2] = val
    return res


def _adaptive64(mr, raw, fixed):
    """Per-view threshold (or the fixed one), then 5x5x5 triangle smoothing (peak one past the middle) above it."""
    cg = mr.cg
    n, nrr, nch = int(mr.ri.n_proj_pull), int(cg.n_rows_raw), int(cg.n_channels)
    x = raw.reshape(n, nrr, nch)
    npf = int(cg.n_proj_ffs)
    if fixed > 0:
        thr = torch.full((n,), float(np.float32(fixed)), dtype=torch.float64, device=x.device)
    else:
        def odd(frac):
            w = int(math.ceil(frac * npf))
            return w + (1 - w % 2)

        sup = x.reshape(n, -1).amax(1).double().clamp(min=0)
        n_avg, n_range = odd(18.0 / 360.0), odd(0.5)
        idx = torch.arange(n, device=x.device)
        sm = torch.zeros(n, dtype=torch.float64, device=x.device)
        for i in range(n_avg):
            sm += sup[(idx - n_avg // 2 + i).clamp(0, n - 1)] / n_avg
        win_idx = idx[:, None] - n_range // 2 + torch.arange(n_range, device=x.device)[None, :]
        inside = (win_idx >= 0) & (win_idx < n)
        win = sm[win_idx.clamp(0, n - 1)]
        hi = torch.where(inside, win, torch.zeros_like(win)).amax(1)
        lo = torch.where(inside, win, torch.full_like(win, 1e4)).amin(1)
        win = torch.where(inside, win, torch.full_like(win, -1.0))
        ecc = ((1 - lo / hi - 0.3) / 0.2).clamp(0, 1)
        lhs = 0.03 * float(mr.rp.adaptive_filtration_s) * ecc
        lower, upper, thr = lo.clone(), hi.clone(), (hi + lo) / 2

        def rhs_of(t):
            return (win > t[:, None]).sum(1).double() / (PI_BP * npf)

        rhs = rhs_of(thr)
        for _ in range(20):
            go = ((lhs - rhs).abs() / lhs > 0.01) & (rhs != lhs)
            if not bool(go.any()):
                break
            lower = torch.where(go & (rhs > lhs), thr, lower)
            upper = torch.where(go & (rhs < lhs), thr, upper)
            thr = torch.where(go, (lower + upper) / 2, thr)
            rhs = torch.where(go, rhs_of(thr), rhs)
    out = torch.empty(x.shape, dtype=torch.float64, device=x.device)
    tri = [3 - abs(i - 3) for i in range(5)]
    step = 256
    for p0 in range(0, n, step):
        a, b = max(0, p0 - 2), min(n, p0 + step + 2)
        m = min(n, p0 + step) - p0
        blk = torch.zeros((step + 4, nrr + 4, nch + 4), dtype=torch.float64, device=x.device)
        blk[a - p0 + 2:b - p0 + 2, 2:-2, 2:-2] = x[a:b].double()
        one = torch.zeros_like(blk)
        one[a - p0 + 2:b - p0 + 2, 2:-2, 2:-2] = 1.0
        val = torch.zeros((m, nrr, nch), dtype=torch.float64, device=x.device)
        norm = torch.zeros_like(val)
        for k in range(5):
            for j in range(5):
                for i in range(5):
                    t = float(tri[i] + tri[j] + tri[k] + 1)
                    val += t * blk[k:k + m, j:j + nrr, i:i + nch]
                    norm += t * one[k:k + m, j:j + nrr, i:i + nch]
        c = x[p0:p0 + m].double()
        out[p0:p0 + m] = torch.where(c > thr[p0:p0 + m, None, None], val / norm, c)
    return out.reshape(-1)


def _backproject64(mr, reb):
    """One 32-slice block: Stierstorfer weights, bilinear taps with a zero border, per-angle normalisation."""
    cg, rp = mr.cg, mr.rp
    nx, ny, nos, n_rows = int(rp.nx), int(rp.ny), int(cg.n_channels_oversampled), int(cg.n_rows)
    npt = int(cg.n_proj_turn)
    half, td = npt // 2, int(cg.table_direction)
    n_ht = (int(mr.ri.n_proj_pull) // int(mr.ri.n_ffs) - 2 * int(cg.add_projections)) // half
    f32 = np.float32
    # the start angle is a float32 number of degrees
    t0 = f32(mr.tube_angles[0]) + f32(cb.pull_start(mr) + int(cg.add_projections_ffs)) * f32(360.0) / f32(int(cg.n_proj_ffs))
    start = float(f32(math.fmod(float(t0), 360.0) * float(f32(PI_BP)) / 180.0))
    rf, zr, coll, fov = float(cg.r_f), float(cg.z_rot), float(rp.coll_slicewidth), float(rp.recon_fov)
    ds = rf * float(cg.fan_angle_increment) / 2
    tanc = math.tan(float(cg.theta_cone) / 2)
    hr = (n_rows - 1) / 2.0
    dev = reb.device
    flip = 1.0 if td == -1 else -1.0
    x = (flip * fov / nx * (torch.arange(nx, device=dev, dtype=torch.float64) - (nx - 1) / 2) + float(rp.x_origin))[:, None]
    y = (fov / ny * (torch.arange(ny, device=dev, dtype=torch.float64) - (ny - 1) / 2) + float(rp.y_origin))[None, :]
    z = torch.arange(32, device=dev, dtype=torch.float64)[:, None, None] * coll
    img = torch.zeros((32, nx, ny), dtype=torch.float64, device=dev)
    # samples with a border of zeros on the channel axis
    pad = torch.zeros((n_rows + 1, nos + 2), dtype=torch.float64, device=dev)
    wide = nos + 2
    for i in range(half):
        st, ht = torch.zeros_like(img), torch.zeros_like(img)
        for k in range(n_ht):
            dth = 2 * PI_BP / npt * i + k * PI_BP
            sn, cs = math.sin(start + dth), math.cos(start + dth)
            phat = x * sn - y * cs
            pl = phat / ds + 2 * float(cg.central_channel)
            lhat = torch.sqrt(rf * rf - phat * phat) - x * cs - y * sn
            g = -td / (lhat * tanc)
            dz = zr / (2 * PI_BP) * torch.asin(phat / rf) + (zr / 2 - zr * dth / (2 * PI_BP))
            q = g * (dz + z)
            aq = q.abs()
            w = torch.where(aq < 0.6, torch.ones_like(aq), torch.cos(PI_BP / 2 * ((aq - 0.6) / 0.4)) ** 2)
            w = torch.where(aq < 1.0, w, torch.zeros_like(w))
            row = ((q + 1) * hr).clamp(0, n_rows - 1)
            r0 = row.floor()
            fr = row - r0
            c0 = pl.floor()
            fc = pl - c0
            ok = (c0 >= -1) & (c0 <= nos - 1)
            ci = torch.where(ok, c0 + 1, torch.zeros_like(c0)).long()
            pad[:n_rows, 1:-1] = reb[i + k * half]
            flat = pad.reshape(-1)
            at = r0.long() * wide + ci
            top = flat[at]
            top += fc * (flat[at + 1] - top)
            bot = flat[at + wide]
            bot += fc * (flat[at + wide + 1] - bot)
            val = torch.where(ok, top + fr * (bot - top), torch.zeros_like(top))
            st += w * val
            ht += w
        img += torch.where(ht > 0, st / ht, torch.zeros_like(st))
    inside = torch.sqrt(x * x + y * y) < float(rp.acq_fov) / 2
    return torch.where(inside, img * (2 * PI_BP / npt), torch.zeros_like(img)).reshape(32, nx * ny)


def _finalize64(mr, image):
    """Triangle-weighted thickening of the raw slices (blocks stored in table order), then HU."""
    rp, ri = mr.rp, mr.ri
    nb, n_raw = int(ri.n_slices_block), int(ri.n_slices_block * ri.n_blocks)
    d = rp.end_pos - rp.start_pos
    rdir = 1 if d >= 0 else -1
    tdir = 1 if mr.table_positions[1000] - mr.table_positions[0] >= 0 else -1
    loc = [float(np.float32(ri.recon_start_pos + np.float32(rdir * i) * np.float32(rp.coll_slicewidth))) for i in range(n_raw)]
    out = []
    for kf in range(int(cb.n_slices_final(mr))):
        at = float(np.float32(rp.start_pos + np.float32(rdir * kf) * np.float32(rp.slice_thickness)))
        w = [max(0.0, 1 - abs(v - at) / rp.slice_thickness) for v in loc]
        total = sum(w)
        acc = torch.zeros(image.shape[1], dtype=torch.float64, device=image.device)
        for i, wi in enumerate(w):
            if wi:
                b, zz = divmod(i, nb)
                acc += wi / total * image[b * nb + (nb - 1 - zz) if rdir != tdir else i].double()
        mu = float(np.float32(MU_WATER))
        out.append(1000.0 * (acc - mu) / mu)
    return torch.stack(out)
