"""The workloads whose speed this library is developed against.

listed() are the calls that users of the library make, from a refocused target
chip to the realistic full scene: back-projection on the nearest, linear and
sinc8 interpolators, on complex64 and bf16x2 profiles, planned and unplanned,
alone and batched; range compression; omega-K image formation; and the echo
generator.  draw() gives further cases of the same ranges.  prepare() makes a
case's inputs on the GPU and keeps what a program keeps between calls (a
context, a plan, the output buffers); run() is one call; work() the bytes and
floating-point operations that the call cannot do without; exact() the result
in 64-bit torch, written from the definitions in include/sarbp.h.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from sar_cambrianaccelerationcard_amd import device as D
from sar_cambrianaccelerationcard_amd import native

C_LIGHT = 299792458.0
FC = 9.6e9                        # X band
BANDWIDTH, PULSE_WIDTH, FS_RAW = 150e6, 2e-6, 200e6
DR = C_LIGHT / (2 * 4 * FS_RAW)   # 4-times upsampled range bin
SPEED, PRF, ALTITUDE, GROUND_RANGE = 150.0, 1000.0, 3000.0, 4000.0
MOST_PIXEL_PULSES = 4096 * 4096 * 4096
EXACT_PIXEL_PULSES = 6e9          # above it the 64-bit sum takes too long

# The radar of the omega-K path's reference scene (omegak.radarsat_scene).
WK = dict(c=299790000.0, f0=5.3e9, fs=32.317e6, prf=1256.98, kr=-7.2135e11, vr=7062.0, f_nc=-6900.0)
WK_R0 = 988647.462


def listed():
    return [
        # The smallest call: one target chip around a known point, planned from
        # the grid alone; launch latency and the host's share count.
        dict(name="chip_smallest", kind="bp", nx=128, ny=128, pulses=128, samples=2048, spacing=0.5,
             interp="sinc8", dtype="c64", precision="ref", planned=False),
        # The small scene of configs/config0.json, as the quick-look user runs
        # it: linear interpolation, no plan.
        dict(name="scene_small_linear", kind="bp", nx=512, ny=512, pulses=512, samples=2048, spacing=0.5,
             interp="linear", dtype="c64", precision="ref", planned=False),
        # Refocusing a small region with the full aperture (odd sizes): few
        # pixels, every pulse, from a plan.
        dict(name="chip_long_aperture", kind="bp", nx=257, ny=251, pulses=4096, samples=8192, spacing=0.25,
             interp="sinc8", dtype="c64", precision="ref", planned=True),
        # The realistic scene of configs/config1.json: the library's headline.
        dict(name="scene_realistic", kind="bp", nx=4096, ny=4096, pulses=4096, samples=8192, spacing=0.25,
             interp="sinc8", dtype="c64", precision="ref", planned=True),
        # The reference-compatible synchronous entry point (nearest bin, 1 m
        # pixels, its own geometry), at a ragged image size.
        dict(name="dropin_nearest", kind="dropin", na=1000, nr=900, pulses=1024, samples=8192),
        # A medium scene with profiles stored as bf16 pairs to halve their
        # memory; ragged tiles on both edges.
        dict(name="scene_bf16", kind="bp", nx=1537, ny=1409, pulses=2048, samples=8192, spacing=0.5,
             interp="sinc8", dtype="bf16x2", precision="ref", planned=True),
        # Wide-area browse image: pixels too coarse for the FP32 differential,
        # so the library runs its double-float arithmetic.
        dict(name="scene_coarse", kind="bp", nx=1024, ny=768, pulses=2048, samples=8192, spacing=1.6,
             interp="sinc8", dtype="c64", precision="ref", planned=True),
        # Uneven jobs of the size mix of configs/config3.json in one batched
        # call, as a processing queue submits them.
        dict(name="batch_mixed", kind="batch", jobs=16, side_min=256, side_max=2048, mix=20260031),
        # Range compression of the realistic scene's raw echoes.
        dict(name="range_compress", kind="range", pulses=4096, n_raw=2448, upsample=4, crop=0, n_out=8192,
             dtype="c64"),
        # omega-K at the reference scene's size (power-of-two padded azimuth).
        dict(name="omega_k_scene", kind="wk", na_in=3072, nr_in=2048, window="floor", range_ref="r0"),
        # omega-K of a crop: odd lengths, no power of two on either axis.
        dict(name="omega_k_crop", kind="wk", na_in=701, nr_in=613, window="floor", range_ref="centre"),
        # Raw echoes of a point-target scene by the reference-compatible
        # generator.
        dict(name="echo_targets", kind="echo", pulses=2048, samples=2448, targets=64),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["bp", "bp", "bp", "bp", "dropin", "batch", "range", "wk", "echo"])
    if kind == "bp":
        nx, ny = _log(rng, 64, 4096), _log(rng, 64, 4096)
        pulses = max(64, min(_log(rng, 64, 4096), MOST_PIXEL_PULSES // (nx * ny)))
        coarse = rng.random() < 0.2
        spacing = round(rng.uniform(1.5, 2.0) if coarse else rng.uniform(0.25, 1.0), 3)
        return dict(kind="bp", nx=nx, ny=ny, pulses=pulses, samples=rng.randint(2048, 8192), spacing=spacing,
                    interp=rng.choice(["sinc8", "sinc8", "linear", "nearest"]),
                    dtype=rng.choice(["c64", "c64", "bf16x2"]), precision="ref", planned=rng.random() < 0.6)
    if kind == "dropin":
        return dict(kind="dropin", na=_log(rng, 96, 2048), nr=_log(rng, 80, 2048), pulses=_log(rng, 128, 2048),
                    samples=8192)
    if kind == "batch":
        return dict(kind="batch", jobs=rng.randint(2, 12), side_min=256, side_max=rng.choice([512, 1024, 2048]),
                    mix=rng.randint(1, 1 << 30))
    if kind == "range":
        n_raw, upsample = _log(rng, 60, 6000), rng.choice([1, 2, 3, 4, 4, 8])
        nf = _fft_size(n_raw)
        n_out = rng.randint(max(1, upsample * n_raw // 2), upsample * n_raw)
        return dict(kind="range", pulses=_log(rng, 64, 4096), n_raw=n_raw, upsample=upsample,
                    crop=rng.randint(0, min(64, upsample * nf - n_out)), n_out=n_out,
                    dtype=rng.choice(["c64", "c64", "bf16x2"]))
    if kind == "wk":
        na_in = rng.choice([768, 1536, 3072]) if rng.random() < 0.4 else _log(rng, 96, 3000)
        return dict(kind="wk", na_in=na_in, nr_in=_log(rng, 96, 2048), window=rng.choice(["floor", "centered"]),
                    range_ref=rng.choice(["r0", "centre"]))
    return dict(kind="echo", pulses=_log(rng, 128, 4096), samples=_log(rng, 300, 4096), targets=_log(rng, 5, 128))


# ---- inputs -------------------------------------------------------------------

_context = None


def _ctx():
    """The one context that a program keeps for all its calls."""
    global _context
    if _context is None:
        _context = native.Context(0)
    return _context


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _noise(shape, gen):
    return torch.view_as_complex(torch.randn((*shape, 2), dtype=torch.float32, device="cuda", generator=gen))


def _track(pulses, seed):
    """Straight track with smooth cross-track and vertical deviations (0.5 m)."""
    rng = np.random.default_rng(int(seed) & 0x7FFFFFFF)
    pos = np.zeros((pulses, 3))
    pos[:, 0] = SPEED * (np.arange(pulses) - 0.5 * (pulses - 1)) / PRF
    pos[:, 2] = ALTITUDE
    k = 200
    for ax in (1, 2):
        w = np.convolve(rng.standard_normal(pulses + k), np.ones(k) / k, mode="valid")[:pulses]
        w -= w.mean()
        pos[:, ax] += 0.5 * w / max(w.std(), 1e-12)
    return pos


def _profiles(pos, targets, r0, dr, samples, fc, bandwidth, gen):
    """Range-compressed, upsampled profiles [pulses][samples] complex64: point
    targets over band-limited clutter and noise."""
    pulses = pos.shape[0]
    # clutter and noise occupy the chirp's share of the upsampled band
    nf = 1 << (samples - 1).bit_length()
    band = max(8, int(nf * min(1.0, dr * 2.0 * bandwidth / C_LIGHT)))
    prof = torch.empty((pulses, samples), dtype=torch.complex64, device="cuda")
    step = max(1, (1 << 24) // nf)
    for m in range(0, pulses, step):
        n = min(step, pulses - m)
        z = torch.zeros((n, nf), dtype=torch.complex64, device="cuda")
        z[:, :band] = _noise((n, band), gen)
        prof[m:m + n] = torch.fft.ifft(z, dim=1)[:, :samples] * (0.3 * nf / math.sqrt(band))
    p = torch.from_numpy(pos).cuda()
    rows = torch.arange(pulses, device="cuda")[:, None]
    k = torch.arange(-24, 25, device="cuda")[None, :]
    for t in torch.from_numpy(targets).cuda():
        r = torch.linalg.vector_norm(p - t[:3], dim=1)
        u = (r - r0) / dr
        idx = torch.floor(u).long()[:, None] + k
        rev = 2.0 * fc * r / C_LIGHT
        rev = -2.0 * math.pi * (rev - torch.floor(rev))
        amp = torch.sinc((u[:, None] - idx) * (2.0 * bandwidth * dr / C_LIGHT)) * t[3]
        v = torch.polar(amp.abs(), rev[:, None] + torch.where(amp < 0, math.pi, 0.0)).to(torch.complex64)
        ok = (idx >= 0) & (idx < samples)
        idx = idx.clamp(0, samples - 1)
        # a target's samples of one pulse are distinct where `ok`; clamped ones
        # put back what is there
        old = prof[rows, idx]
        r_ok, i_ok = rows.expand_as(idx)[ok], idx[ok]
        prof[r_ok, i_ok] = (old + v)[ok]
    return prof


def _bf16x2(prof):
    """complex64 -> int32 words, bf16 re in the low half, rounded to nearest even."""
    w = torch.view_as_real(prof).to(torch.bfloat16).view(torch.int16).to(torch.int32) & 0xFFFF
    return (w[..., 0] | (w[..., 1] << 16)).contiguous()


def _grid(nx, ny, spacing):
    return ([-(nx // 2) * spacing, GROUND_RANGE - (ny // 2) * spacing, 0.0], [spacing, 0.0, 0.0],
            [0.0, spacing, 0.0], nx, ny)


def _targets(origin, ux, uy, nx, ny, seed, n=12):
    rng = np.random.default_rng((int(seed) & 0x7FFFFFFF) + 17)
    ix, iy = rng.uniform(0.1, 0.9, n) * nx, rng.uniform(0.1, 0.9, n) * ny
    t = np.empty((n, 4))
    t[:, :3] = np.asarray(origin) + ix[:, None] * np.asarray(ux) + iy[:, None] * np.asarray(uy)
    t[:, 3] = rng.uniform(3.0, 8.0, n)
    return t


def _bp_inputs(case, seed):
    grid = _grid(case["nx"], case["ny"], case["spacing"])
    pos = _track(case["pulses"], seed)
    r0 = math.hypot(GROUND_RANGE, ALTITUDE) - 0.5 * case["samples"] * DR
    prof = _profiles(pos, _targets(*grid, seed), r0, DR, case["samples"], FC, BANDWIDTH,
                     _gen(seed))
    if case["dtype"] == "bf16x2":
        prof = _bf16x2(prof)
    return grid, pos, r0, prof


def _mix(case, seed):
    """The jobs of a batched case: sizes from its `mix`, data from the seed."""
    rng = np.random.default_rng(case["mix"])
    jobs = []
    for i in range(case["jobs"]):
        side = int(round(math.exp(rng.uniform(math.log(case["side_min"]), math.log(case["side_max"])))))
        jobs.append(dict(nx=side, ny=side, spacing=float(rng.uniform(0.25, 1.0)),
                         pulses=int(rng.integers(512, 4097)), samples=int(rng.integers(2048, 8193)),
                         interp="sinc8", dtype="c64", precision="ref", seed=int(seed) * 1009 + i))
    return jobs


def _dropin_params(case):
    p = native.SarParams.reference_defaults()
    p.H, p.Rg0, p.La = 3000.0, 5000.0, 60.0
    p.Mslow, p.Nfast = case["pulses"], case["samples"]
    return p


def _dropin_geometry(p, na, nr):
    """Positions and grid of the reference host driver (include/sarbp.h)."""
    m = np.arange(p.Mslow, dtype=np.float64)
    ta = -p.La / (2 * p.vr) + (p.La / p.vr) * m / (p.Mslow - 1)
    pos = np.stack([np.float64(p.vr) * ta, np.zeros(p.Mslow), np.full(p.Mslow, np.float64(p.H))], 1)
    grid = ([p.Az0 - na // 2, p.Rg0 - nr // 2, 0.0], [0.0, 1.0, 0.0], [1.0, 0.0, 0.0], nr, na)
    return pos, grid


def _dropin_inputs(case, seed):
    p = _dropin_params(case)
    pos, grid = _dropin_geometry(p, case["na"], case["nr"])
    prof = _profiles(pos, _targets(*grid, seed), 0.0, float(p.c) / (2 * float(p.Fr)), case["samples"], float(p.fc),
                     float(p.Br), _gen(seed))
    return p, pos, grid, prof


def _fft_size(n_raw):
    return 1 << (n_raw + math.ceil(PULSE_WIDTH * FS_RAW) - 1).bit_length()


def _range_radar(case):
    return dict(c=C_LIGHT, bandwidth=BANDWIDTH, pulse_width=PULSE_WIDTH, fs=FS_RAW, t0=3.2e-5,
                n_raw=case["n_raw"], upsample=case["upsample"], crop_offset=case["crop"], n_out=case["n_out"])


def _range_inputs(case, seed):
    """Raw echoes: overlapping chirps of a few scatterers per pulse, over noise."""
    gen = _gen(seed)
    raw = _noise((case["pulses"], case["n_raw"]), gen)
    t = torch.arange(case["n_raw"], device="cuda", dtype=torch.float32)[None, :] / FS_RAW
    for _ in range(4):
        delay = torch.rand((case["pulses"], 1), device="cuda", generator=gen) * (case["n_raw"] / FS_RAW)
        tau = t - delay
        ph = math.pi * BANDWIDTH / PULSE_WIDTH * (tau - 0.5 * PULSE_WIDTH) ** 2
        raw += torch.where((tau > 0) & (tau < PULSE_WIDTH), torch.polar(torch.full_like(ph, 2.0), ph), 0)
    return raw


def _wk_params(case):
    _, nr = native.wk_padded_size(case["na_in"], case["nr_in"])
    window = 0.5 * WK["c"] * nr / WK["fs"]
    r0 = max(1, round(WK_R0 / window)) * window
    if case["range_ref"] == "centre":
        pad = (nr - case["nr_in"]) // 2
        r0 += 0.5 * WK["c"] * pad / WK["fs"]
    return native.make_wk_params(**WK, r0=r0, taps=6, window=case["window"], range_ref=case["range_ref"])


def _wk_inputs(case, seed):
    """Raw echoes: range chirps of scatterers with quadratic azimuth phase, over
    noise."""
    gen = _gen(seed)
    na, nr = case["na_in"], case["nr_in"]
    echo = _noise((na, nr), gen)
    m = torch.arange(na, device="cuda", dtype=torch.float64)[:, None]
    n = torch.arange(nr, device="cuda", dtype=torch.float64)[None, :]
    rng = np.random.default_rng((int(seed) & 0x7FFFFFFF) + 3)
    lam = WK["c"] / WK["f0"]
    rate = 2.0 * WK["vr"] ** 2 / (lam * WK_R0)
    for _ in range(6):
        m0, n0 = rng.uniform(0, na), rng.uniform(0, nr)
        tau, eta = (n - n0) / WK["fs"], (m - m0) / WK["prf"]
        rev = 0.5 * WK["kr"] * tau ** 2 - 0.5 * rate * eta ** 2 + WK["f_nc"] * eta
        v = torch.polar(torch.full_like(rev, 3.0), 2.0 * math.pi * (rev - torch.floor(rev)))
        echo += torch.where(tau.abs() < 20e-6, v, 0).to(torch.complex64)
    return echo


def _echo_inputs(case, seed):
    rng = np.random.default_rng(int(seed) & 0x7FFFFFFF)
    p = native.SarParams.reference_defaults()
    p.La, p.H, p.Ntarget = 80.0, 3000.0, case["targets"]
    n = case["targets"]
    pt = np.stack([rng.uniform(-40, 40, n), rng.uniform(7000, 7600, n), rng.uniform(0.2, 2.0, n)], 1)
    t0 = np.float32(2 * math.hypot(7000.0, p.H) / p.c - 30 / p.Fr)
    tr = (t0 + np.arange(case["samples"], dtype=np.float32) / np.float32(p.Fr)).astype(np.float32)
    ta = np.linspace(-0.3, 0.3, case["pulses"]).astype(np.float32)
    return pt.astype(np.float32), ta, tr, p


def prepare(case, seed):
    kind, ctx = case["kind"], _ctx()
    if kind == "bp":
        grid, pos, r0, prof = _bp_inputs(case, seed)
        params = native.make_params(c=C_LIGHT, fc=FC, r0=r0, dr=DR, n_pulses=case["pulses"],
                                    n_samples=case["samples"], interp=case["interp"], precision=case["precision"],
                                    dtype=case["dtype"])
        ng = native.make_grid(*grid)
        return dict(kind=kind, ctx=ctx, prof=prof, pos=torch.from_numpy(pos).cuda(), grid=ng, params=params,
                    plan=ctx.plan(pos, ng, params) if case["planned"] else None,
                    img=torch.empty((case["ny"], case["nx"]), dtype=torch.complex64, device="cuda"))
    if kind == "dropin":
        p, _, _, prof = _dropin_inputs(case, seed)
        return dict(kind=kind, lib=native.load(), prof=prof, p=p, na=case["na"], nr=case["nr"],
                    img=torch.empty((case["na"], case["nr"]), dtype=torch.complex64, device="cuda"))
    if kind == "batch":
        jobs, keep, imgs = [], [], []
        for spec in _mix(case, seed):
            grid, pos, r0, prof = _bp_inputs(spec, spec["seed"])
            d_pos = torch.from_numpy(pos).cuda()
            img = torch.empty((spec["ny"], spec["nx"]), dtype=torch.complex64, device="cuda")
            j = native.Job()
            j.d_profiles, j.d_pos, j.h_pos, j.d_image = prof.data_ptr(), d_pos.data_ptr(), pos.ctypes.data, img.data_ptr()
            j.grid = native.make_grid(*grid)
            j.params = native.make_params(c=C_LIGHT, fc=FC, r0=r0, dr=DR, n_pulses=spec["pulses"],
                                          n_samples=spec["samples"], interp=spec["interp"])
            jobs.append(j)
            keep.append((prof, d_pos, pos))
            imgs.append(img)
        return dict(kind=kind, ctx=ctx, jobs=jobs, keep=keep, imgs=imgs)
    if kind == "range":
        out = torch.empty((case["pulses"], case["n_out"]), device="cuda",
                          dtype=torch.complex64 if case["dtype"] == "c64" else torch.int32)
        return dict(kind=kind, ctx=ctx, raw=_range_inputs(case, seed), out=out, n=case["pulses"],
                    rp=D.range_params(_range_radar(case), case["dtype"]))
    if kind == "wk":
        size = native.wk_padded_size(case["na_in"], case["nr_in"])
        return dict(kind=kind, ctx=ctx, echo=_wk_inputs(case, seed), wp=_wk_params(case),
                    img=torch.empty(size, dtype=torch.complex64, device="cuda"))
    pt, ta, tr, p = _echo_inputs(case, seed)
    return dict(kind=kind, pt=pt, ta=ta, tr=tr, p=p)


def run(state):
    kind = state["kind"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "bp":
        args = state["prof"].data_ptr(), state["pos"].data_ptr()
        if state["plan"] is not None:
            state["plan"].execute(*args, state["img"].data_ptr(), stream)
        else:
            state["ctx"].backproject(*args, state["grid"], state["params"], state["img"].data_ptr(), stream)
        return state["img"]
    if kind == "dropin":
        native.check(state["lib"].sarbp_launch_backprojection(
            C.c_void_p(state["prof"].data_ptr()), C.c_void_p(state["img"].data_ptr()), state["p"], state["na"],
            state["nr"]), "sarbp_launch_backprojection")
        return state["img"]
    if kind == "batch":
        state["ctx"].backproject_batch(state["jobs"], stream)
        return state["imgs"]
    if kind == "range":
        state["ctx"].range_compress(state["raw"].data_ptr(), state["n"], state["rp"], state["out"].data_ptr(), stream)
        return state["out"]
    if kind == "wk":
        echo = state["echo"]
        state["ctx"].omega_k(echo.data_ptr(), echo.shape[0], echo.shape[1], state["wp"], state["img"].data_ptr(),
                             stream)
        return state["img"]
    return D.generate_echo(state["pt"], state["ta"], state["tr"], state["p"])


# ---- work ---------------------------------------------------------------------

def _bp_work(nx, ny, pulses, samples, interp, dtype):
    # per pixel and pulse: the range (3 differences, 3 squares, 2 sums, a root),
    # the bin (2), the phase (2), its sine and cosine (2), the rotation and the
    # sum (8), and the taps (a complex multiply-add each)
    taps = {"nearest": 0, "linear": 2, "sinc8": 8}[interp]
    w = float(nx) * ny * pulses
    return {"bytes": pulses * samples * (8 if dtype == "c64" else 4) + pulses * 24 + nx * ny * 8,
            "flops": w * (23 + 4 * taps)}


def _fft_flops(n):
    return 5.0 * n * math.log2(max(n, 2))


def work(case):
    kind = case["kind"]
    if kind == "bp":
        return _bp_work(case["nx"], case["ny"], case["pulses"], case["samples"], case["interp"], case["dtype"])
    if kind == "dropin":
        return _bp_work(case["nr"], case["na"], case["pulses"], case["samples"], "nearest", "c64")
    if kind == "batch":
        w = [_bp_work(j["nx"], j["ny"], j["pulses"], j["samples"], "sinc8", "c64") for j in _mix(case, 0)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    if kind == "range":
        nf, up = _fft_size(case["n_raw"]), case["upsample"]
        return {"bytes": case["pulses"] * (8 * case["n_raw"] + (8 if case["dtype"] == "c64" else 4) * case["n_out"]),
                "flops": case["pulses"] * (_fft_flops(nf) + 6 * nf + up * _fft_flops(nf) + 6 * (up - 1) * nf)}
    if kind == "wk":
        na_in, nr_in = case["na_in"], case["nr_in"]
        na, nr = native.wk_padded_size(na_in, nr_in)
        # two 2-D transforms, the reference function (a root, a sine, a cosine,
        # a complex product), 6 taps
        return {"bytes": 8 * na_in * nr_in + 8 * na * nr,
                "flops": nr_in * _fft_flops(na) + nr * _fft_flops(na) + 2 * na * _fft_flops(nr) + na * nr * (16 + 24)}
    return {"bytes": 8 * case["pulses"] * case["samples"] + 4 * (case["pulses"] + case["samples"]) + 12 * case["targets"],
            # the delay gate of every target at every sample (2); the ranges
            # once per pulse and target
            "flops": 2.0 * case["pulses"] * case["samples"] * case["targets"] + 12.0 * case["pulses"] * case["targets"]}


# ---- 64-bit results -------------------------------------------------------------

def _kernel8(x, beta=6.0):
    """8-tap Kaiser-windowed sinc."""
    t = x / 4.0
    w = torch.special.i0(beta * torch.sqrt(torch.clamp(1.0 - t * t, min=0.0))) / float(np.i0(beta))
    return torch.where(x.abs() < 4.0, torch.sinc(x) * w, 0.0)


def _exact_bp(prof, pos, grid, r0, dr, fc, c, interp):
    origin, ux, uy, nx, ny = grid
    dev = prof.device
    if prof.dtype == torch.int32:
        prof = torch.complex((prof << 16).view(torch.float32), (prof & -65536).view(torch.float32))
    pulses, samples = prof.shape
    o, a, b = (torch.tensor(v, dtype=torch.float64, device=dev) for v in (origin, ux, uy))
    p = torch.from_numpy(pos).to(dev)
    img = torch.zeros(ny * nx, dtype=torch.complex128, device=dev)
    per = max(1, min(nx * ny, 1 << 20))
    for i0 in range(0, nx * ny, per):
        i = torch.arange(i0, min(i0 + per, nx * ny), device=dev)
        px = o + (i % nx).double()[:, None] * a + (i // nx).double()[:, None] * b
        step = max(1, (1 << 23) // len(i))
        for m0 in range(0, pulses, step):
            q = p[m0:m0 + step]
            r = torch.sqrt(sum((px[None, :, k] - q[:, k, None]) ** 2 for k in range(3)))
            u = (r - r0) / dr
            s = prof[m0:m0 + step]

            def tap(j):
                ok = (j >= 0) & (j < samples)
                v = torch.gather(s, 1, j.clamp(0, samples - 1).long())
                return torch.where(ok, v, 0)

            if interp == "nearest":
                v = tap(torch.floor(u + 0.5)).to(torch.complex128)
            else:
                f0 = torch.floor(u)
                f = u - f0
                if interp == "linear":
                    v = tap(f0) * (1.0 - f) + tap(f0 + 1) * f
                else:
                    v = sum(tap(f0 - 3 + t) * _kernel8(f + 3 - t) for t in range(8))
            rev = 2.0 * fc * r / c
            rev = 2.0 * math.pi * (rev - torch.floor(rev))
            img[i] += (v * torch.polar(torch.ones_like(rev), rev)).sum(0)
    return img.reshape(ny, nx)


def _exact_range(case, seed):
    rd = _range_radar(case)
    raw = _range_inputs(case, seed)
    nf, up = _fft_size(case["n_raw"]), case["upsample"]
    n = torch.arange(nf, device="cuda", dtype=torch.float64)
    t = n / rd["fs"]
    rev = 0.5 * rd["bandwidth"] / rd["pulse_width"] * (t - 0.5 * rd["pulse_width"]) ** 2
    h = torch.polar(torch.ones_like(rev), 2.0 * math.pi * (rev - torch.floor(rev)))
    h = torch.where((t > 0) & (t < rd["pulse_width"]) & (n < case["n_raw"]), h, 0)
    hc = torch.conj(torch.fft.fft(h))
    half, nu = (nf + 1) // 2, up * nf
    out = torch.empty((case["pulses"], case["n_out"]), dtype=torch.complex128, device="cuda")
    step = max(1, (1 << 23) // nu)
    for m in range(0, case["pulses"], step):
        y = torch.fft.fft(raw[m:m + step].to(torch.complex128), n=nf, dim=1) * hc
        z = torch.zeros((y.shape[0], nu), dtype=torch.complex128, device="cuda")
        z[:, :half] = y[:, :half]
        z[:, half + nu - nf:] = y[:, half:]
        out[m:m + step] = (torch.fft.ifft(z, dim=1) * up)[:, case["crop"]:case["crop"] + case["n_out"]]
    return out


def _exact_wk(case, seed):
    echo, wp = _wk_inputs(case, seed).to(torch.complex128), _wk_params(case)
    na_in, nr_in = echo.shape
    na, nr = native.wk_padded_size(na_in, nr_in)
    pa, pr = (na - na_in) // 2, (nr - nr_in) // 2

    def ramp(n):
        k = torch.arange(n, device="cuda") + (n + 1) // 2
        return torch.where(k >= n, k - n, k).double() - 0.5 * n

    def unit(rev):
        return torch.polar(torch.ones_like(rev), 2.0 * math.pi * (rev - torch.round(rev)))

    x = torch.zeros((na, nr), dtype=torch.complex128, device="cuda")
    x[pa:pa + na_in, pr:pr + nr_in] = echo
    ta = (torch.arange(na, device="cuda").double() - 0.5 * na) / wp.prf
    x = x * unit(-wp.f_nc * ta)[:, None]
    fr, fa = ramp(nr) * (wp.fs / nr), wp.f_nc + ramp(na) * (wp.prf / na)
    z = torch.fft.fft(torch.fft.fft(x, dim=0), dim=1)
    kk, h = wp.c * wp.c / (4.0 * wp.vr * wp.vr), nr // 2
    f = (wp.f0 + fr)[None, :]
    s = torch.sqrt(torch.clamp(f * f - kk * (fa * fa)[:, None], min=0.0))
    centre = wp.range_ref == native.WK_RANGE_REF_CENTRE
    if centre:
        ts = 2.0 * wp.r0 / wp.c - pr / wp.fs
        z = z * unit((ts + h / wp.fs) * s + (0.5 / wp.kr * fr - ts) * fr)
    else:
        z = z * unit(2.0 * wp.r0 / wp.c * s + 0.5 / wp.kr * fr * fr)
    cen = torch.arange(nr, device="cuda").double()[None, :] - (s - f) * (nr / wp.fs)
    fl = torch.floor(cen)
    y, half = torch.zeros_like(z), wp.taps // 2
    if wp.window == native.STOLT_FLOOR:
        for p in range(-half, half):
            idx = torch.clamp(fl + p, 0, nr - 1)
            y = y + torch.gather(z, 1, idx.long()) * torch.sinc(cen - idx)
    else:
        for q in range(-half, half + 2):
            idx, d = fl + q, cen - (fl + q)
            ok = (d.abs() <= half) & (idx >= 0) & (idx <= nr - 1)
            y = y + torch.where(ok, torch.gather(z, 1, idx.clamp(0, nr - 1).long()) * torch.sinc(d), 0)
    if centre:
        y = y * unit(-fr * (h / wp.fs))
    return torch.fft.ifft(torch.fft.ifft(y, dim=1), dim=0)


def _exact_echo(case, seed):
    pt, ta, tr, p = _echo_inputs(case, seed)
    ta, tr = (torch.from_numpy(v).cuda().double() for v in (ta, tr))
    out = torch.zeros((len(ta), len(tr)), dtype=torch.complex128, device="cuda")
    for x, y, sigma in pt.astype(np.float64):
        az = ta * float(p.vr) - x
        r = torch.sqrt(az * az + y * y + float(p.H) * float(p.H))
        t = tr[None, :] - (2.0 * r / float(p.c))[:, None]
        rev = 0.5 * float(p.Kr) * t * t - (2.0 * r / float(p.lambda_))[:, None]
        v = torch.polar(torch.full_like(rev, sigma), 2.0 * math.pi * (rev - torch.round(rev)))
        out += torch.where((t > 0) & (t < float(p.Tr)) & (az.abs() < float(p.La) / 2)[:, None], v, 0)
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "bp":
        if case["nx"] * case["ny"] * case["pulses"] > EXACT_PIXEL_PULSES:
            return None
        grid, pos, r0, prof = _bp_inputs(case, seed)
        return _exact_bp(prof, pos, grid, r0, DR, FC, C_LIGHT, case["interp"])
    if kind == "dropin":
        if case["na"] * case["nr"] * case["pulses"] > EXACT_PIXEL_PULSES:
            return None
        p, pos, grid, prof = _dropin_inputs(case, seed)
        return _exact_bp(prof, pos, grid, 0.0, float(p.c) / (2 * float(p.Fr)), float(p.fc), float(p.c), "nearest")
    if kind == "batch":
        specs = _mix(case, seed)
        if sum(j["nx"] * j["ny"] * j["pulses"] for j in specs) > EXACT_PIXEL_PULSES:
            return None
        out = []
        for j in specs:
            grid, pos, r0, prof = _bp_inputs(j, j["seed"])
            out.append(_exact_bp(prof, pos, grid, r0, DR, FC, C_LIGHT, "sinc8"))
        return out
    if kind == "range":
        # bf16 words are compared as they are
        return _exact_range(case, seed) if case["dtype"] == "c64" else None
    if kind == "wk":
        return _exact_wk(case, seed)
    return _exact_echo(case, seed)
