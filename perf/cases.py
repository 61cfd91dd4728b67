"""Workloads of the SSB engine, for timing and for checking its results.

Each case is one call (or the few calls that belong together) that a user of
this package makes: reconstructing a scan that lies on the GPU, opening a
session on it, re-evaluating a prepared scan, evaluating aberration trials,
loading compressed frames, training the aberration initializer.  ``listed``
names the cases, ``draw`` gives further ones of the same ranges, ``prepare``
builds what the user's program holds before the call, ``run`` makes the call,
``work`` counts what it cannot do without, and ``exact`` gives the results in
64 bits from plain torch and NumPy.

Inputs are simulated 4D-STEM scans: a smoothed-noise phase object, an
aberrated probe, Poisson counts at a stated dose.  Lengths are in Angstrom,
300 kV, scan steps at half the Nyquist step of the bright-field disk.
"""
from __future__ import annotations

import math

import numpy as np
import torch

WAVELENGTH = 0.019687489006849          # 300 kV, Angstrom
SEMIANGLE = 20.0                        # mrad
TARGETS = (128, 256, 512, 1024)         # supported square scans
BYTES = {"uint8": 1, "uint16": 2, "uint32": 4, "int16": 2, "int32": 4, "float32": 4}


# --------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # The smallest scan in use: 64 x 64 positions, detector 64 x 64, padded
        # to 128 x 128 in the call.  Launches and latency count.
        _recon("recon_s64_d64", 64, 64, 64, 64, 16, "uint16", dose=1e4),
        # An odd-sized region of interest of a binned detector, padded to 256 x 256.
        _recon("recon_s203x178_d93x96", 203, 178, 93, 96, 11, "uint16", c12=40.0),
        # The benchmark scan.
        _recon("recon_s256_d128", 256, 256, 128, 128, 16, "uint16"),
        # The large scan: 8.6 GB of raw frames, rotated axes.
        _recon("recon_s512_d128", 512, 512, 128, 128, 16, "uint16", c10=350.0, rot=3.0, dose=1e4),
        # Frames that stay float32 (gain-corrected by a float32 gain map).
        _recon("recon_s128_d128_f32", 128, 128, 128, 128, 16, "float32", gain=True),
        # A whole session: constructor, object and loss, close.
        dict(_base("session_s256_d128", "session", 256, 256, 128, 128, 16), compute_loss=True),
        # A prepared scan re-evaluated at other aberrations, as in interactive tuning.
        _base("object_s256", "object", 256, 256, 128, 128, 16, c12=30.0),
        # One batch of a fit's refinement: defocus, C30 and rotation differ per trial.
        dict(_base("loss_s256_t16_c30", "loss", 256, 256, 128, 128, 16), trials=16, c30_range=2e5, rotations=True),
        # A slice of a (C10, C12, phi12) grid search at the smallest scan.
        dict(_base("loss_s128_t64_quad", "loss", 128, 128, 64, 64, 16), trials=64, c30_range=0.0, rotations=False),
        # The batched search: 512 trials in one launch.
        dict(_base("search_s256_t512", "search", 256, 256, 128, 128, 16), trials=512),
        # Loading: 16,384 bitshuffle-LZ4 chunks of one 192 x 192 frame, binned by 2.
        dict(name="load_f16384_d192_bin2", kind="load", frames=16384, det_rows=192, det_cols=192, radius=24,
             dose=2e4, bin=2, masked=True, dtype="uint32"),
        # One optimisation step of the learned initializer at its training batch.
        dict(name="train_b256", kind="train", batch=256),
    ]


def draw(rng) -> dict:
    """One more case of the listed ranges (sizes over their logarithm)."""
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["recon"] * 4 + ["session", "object", "object", "loss", "loss", "search", "load", "load", "train"])
    if kind == "train":
        return {"kind": "train", "batch": log(32, 400)}
    if kind == "load":
        rows, cols = rng.randint(40, 256), rng.randint(40, 256)
        return {"kind": "load", "frames": max(16, min(log(200, 40000), int(6e8) // (rows * cols))), "det_rows": rows,
                "det_cols": cols, "radius": max(4, min(rows, cols) // rng.randint(5, 9)),
                "dose": round(10 ** rng.uniform(3.5, 4.8)), "bin": rng.choice([1, 2, 2, 3, 4]),
                "masked": rng.random() < 0.5, "dtype": rng.choice(["uint32", "uint32", "uint16"])}
    while True:
        rows = log(40, 700)
        cols = max(33, min(760, int(rows * rng.uniform(0.75, 1.3))))
        det_rows, det_cols = log(32, 200), 0
        det_cols = max(32, min(200, int(det_rows * rng.uniform(0.85, 1.18))))
        radius = max(4, min(24, int(min(det_rows, det_cols) * rng.uniform(0.09, 0.26))))
        dtype = rng.choice(["uint16"] * 5 + ["uint8", "float32", "int32"]) if kind == "recon" else "uint16"
        n = _target(rows, cols)
        nbf = math.pi * radius * radius
        if n * n * det_rows * det_cols * BYTES[dtype] > 8.5e9 or nbf * n * n > 2.0e8:
            continue
        if kind != "recon" and nbf * n * n > 5.5e7:
            continue
        break
    ab = dict(c10=round(rng.uniform(-500, 500), 1), c12=round(rng.choice([0.0, rng.uniform(5, 80)]), 1),
              rot=round(rng.uniform(-5, 5), 2), dose=round(10 ** rng.uniform(4.0, 5.0)))
    if kind == "recon":
        case = _recon("", rows, cols, det_rows, det_cols, radius, dtype, gain=rng.random() < 0.2, **ab)
    else:
        case = _base("", kind, rows, cols, det_rows, det_cols, radius, **ab)
    if kind == "session":
        case["compute_loss"] = rng.random() < 0.7
    if kind == "loss":
        case["trials"] = max(1, min(log(2, 64), int(16 * 5.3e7 / (nbf * n * n))))
        case["c30_range"] = rng.choice([0.0, 2e5])
        case["rotations"] = case["c30_range"] > 0 or rng.random() < 0.5
    if kind == "search":
        case["trials"] = max(8, min(log(8, 512), int(512 * 5.3e7 / (nbf * n * n))))
    case.pop("name")
    return case


def _base(name, kind, rows, cols, det_rows, det_cols, radius, c10=200.0, c12=0.0, rot=0.0, dose=5e4) -> dict:
    return dict(name=name, kind=kind, rows=rows, cols=cols, det_rows=det_rows, det_cols=det_cols, radius=radius,
                c10=c10, c12=c12, rot=rot, dose=dose)


def _recon(name, rows, cols, det_rows, det_cols, radius, dtype, gain=False, **ab) -> dict:
    return dict(_base(name, "recon", rows, cols, det_rows, det_cols, radius, **ab), dtype=dtype, gain=gain)


def _target(rows: int, cols: int) -> int:
    longest = max(rows, cols)
    return next((t for t in TARGETS if longest <= t), TARGETS[-1])


def _ang(case) -> float:
    """Detector sampling in mrad per pixel of a disk of ``radius`` pixels."""
    return SEMIANGLE / case["radius"]


def _step(case) -> float:
    """Scan step: half the Nyquist step of the bright-field disk."""
    return WAVELENGTH / (4.0 * SEMIANGLE * 1e-3)


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------

def _simulate(case: dict, seed: int, frames: int | None = None) -> torch.Tensor:
    """Counts ``[rows, cols, det_rows, det_cols]`` (or ``[frames, ...]``) of a
    phase object under a probe with the case's defocus."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 7919 + 17)
    det_rows, det_cols, radius = case["det_rows"], case["det_cols"], case["radius"]
    if frames is None:
        rows, cols = case["rows"], case["cols"]
    else:
        cols = max(1, int(math.sqrt(frames)))
        rows = -(-frames // cols)
    n = -(-max(det_rows, det_cols) // 16) * 16           # detector window that transforms fast
    pixel = WAVELENGTH / (n * SEMIANGLE * 1e-3 / radius)  # object pixel, Angstrom
    step_px = _step(case) / pixel
    size = max(n, -(-int(max(rows, cols) * step_px) // 32) * 32)
    f = torch.fft.fftfreq(size, device=dev)
    smooth = torch.exp(-2 * math.pi ** 2 * 4.0 * (f[:, None] ** 2 + f[None, :] ** 2))
    phase = torch.fft.ifft2(torch.fft.fft2(torch.randn((size, size), device=dev, generator=gen)) * smooth).real
    phase = phase * (0.1 / phase.std())
    obj = torch.exp(1j * phase.to(torch.complex64))

    k = torch.fft.fftfreq(n, device=dev, dtype=torch.float64) / pixel
    k2 = k[:, None] ** 2 + k[None, :] ** 2
    semi, ang = SEMIANGLE * 1e-3, SEMIANGLE * 1e-3 / radius
    aperture = ((semi - k2.sqrt() * WAVELENGTH) / ang + 0.5).clamp(0, 1)
    probe_f = aperture * torch.exp(-1j * math.pi * WAVELENGTH * k2 * case.get("c10", 200.0))
    norm = float((probe_f.abs() ** 2).sum())
    probe_f = probe_f.to(torch.complex64)
    kk = torch.fft.fftfreq(n, device=dev, dtype=torch.float32)
    win = torch.arange(n, device=dev) - n // 2

    t = math.radians(case.get("rot", 0.0))
    ct, st = math.cos(t), math.sin(t)
    ri = (torch.arange(rows * cols, device=dev) // cols).to(torch.float64) * step_px
    ci = (torch.arange(rows * cols, device=dev) % cols).to(torch.float64) * step_px
    pos_r, pos_c = ri * ct + ci * st, ci * ct - ri * st
    total = rows * cols if frames is None else frames
    dtype = getattr(torch, case["dtype"]) if case["kind"] == "recon" else torch.uint16
    top = {torch.uint8: 255}.get(dtype, 65535)
    out = torch.empty((total, det_rows, det_cols), dtype=dtype, device=dev)
    r0, c0 = n // 2 - det_rows // 2, n // 2 - det_cols // 2
    batch = max(1, (1 << 26) // (n * n))
    for s in range(0, total, batch):
        e = min(total, s + batch)
        br, bc = pos_r[s:e].floor(), pos_c[s:e].floor()
        fr, fc = (pos_r[s:e] - br).float(), (pos_c[s:e] - bc).float()
        ramp = (torch.polar(torch.ones((e - s, n), device=dev), -2 * math.pi * fr[:, None] * kk)[:, :, None]
                * torch.polar(torch.ones((e - s, n), device=dev), -2 * math.pi * fc[:, None] * kk)[:, None, :])
        probe = torch.fft.fftshift(torch.fft.ifft2(probe_f * ramp), dim=(-2, -1))
        del ramp
        pr = (br.long()[:, None] + win) % size
        pc = (bc.long()[:, None] + win) % size
        wave = torch.fft.fft2(probe * obj[pr[:, :, None], pc[:, None, :]])
        del probe
        inten = torch.fft.fftshift(wave.real ** 2 + wave.imag ** 2, dim=(-2, -1))
        inten = inten[:, r0:r0 + det_rows, c0:c0 + det_cols] * (case["dose"] / norm)
        counts = torch.poisson(inten, generator=gen).clamp_(0, top)
        out[s:e] = counts.to(dtype) if dtype in (torch.float32, torch.int32) else counts.to(torch.int32).to(dtype)
    return out if frames is not None else out.reshape(rows, cols, det_rows, det_cols)


def _gain(case: dict, seed: int):
    if not case.get("gain"):
        return None
    rng = np.random.default_rng(seed + 101)
    return torch.tensor(rng.uniform(0.9, 1.1, (case["det_rows"], case["det_cols"])), dtype=torch.float32, device="cuda")


def _trials(case: dict, seed: int):
    """Aberration vectors and rotations of the case's trials."""
    rng = np.random.default_rng(seed + 202)
    t = case["trials"]
    mags, angles = np.zeros((t, 14)), np.zeros((t, 14))
    mags[:, 0] = rng.uniform(-500, 500, t).astype(np.float32)
    if case["kind"] == "search" or case["c30_range"] > 0:
        c30 = case.get("c30_range", 2e5)
        mags[:, 4] = rng.uniform(-c30, c30, t).astype(np.float32)
    else:
        mags[:, 1] = rng.uniform(0, 60, t).astype(np.float32)
        angles[:, 1] = rng.uniform(-1.5, 1.5, t).astype(np.float32)
    turn = case["kind"] == "search" or case["rotations"]
    rot = np.radians(rng.uniform(-5, 5, t)) if turn else None
    return mags, angles, rot


def _engine(case: dict, gain=None):
    from quantem.gpu_amd.ssb.compute.hip.engine import HipSSBEngine, PlanSpec, SSBPlan
    n, ang, step = _target(case["rows"], case["cols"]), _ang(case) * 1e-3, _step(case)
    spec = PlanSpec(n, case["det_rows"], case["det_cols"], case["det_rows"] * case["det_cols"], WAVELENGTH,
                    SEMIANGLE * 1e-3, ang, ang, step, step)
    eng = HipSSBEngine(SSBPlan(spec, device=torch.device("cuda", torch.cuda.current_device())))
    if gain is not None:
        eng.set_detector_gain(gain)
    return eng


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "load":
        return _prepare_load(case, seed)
    if kind == "train":
        return _prepare_train(case, seed)
    data = _simulate(case, seed)
    if kind == "session":
        return {"case": case, "data": data}
    gain = _gain(case, seed)
    eng = _engine(case, gain)
    n = eng.n
    if kind == "recon":
        return {"case": case, "data": data, "engine": eng,
                "object": torch.empty((n, n), dtype=torch.complex64, device=data.device),
                "phase": torch.empty((n, n), dtype=torch.float32, device=data.device)}
    from quantem.gpu_amd.ssb.compute.hip.engine import normalize_scan
    data = normalize_scan(data)
    eng.mean_dp(data)
    eng.select_bf(0.0, None)
    eng.prepare_g(data)
    eng.cache_rotation(math.radians(case["rot"]))
    state = {"case": case, "engine": eng}
    if kind == "object":
        state["phase"] = torch.empty((n, n), dtype=torch.float32, device=data.device)
    else:
        state["trials"] = _trials(case, seed)
    if kind == "search":
        from quantem.gpu_amd.ssb.compute.hip.trials import TrialBatch
        state["batch"] = TrialBatch([eng], case["trials"])
    return state


def _prepare_load(case: dict, seed: int) -> dict:
    """Compressed chunks of the case's frames: 64 simulated frames, each stored
    many times over, in a shuffled order."""
    from quantem.gpu_amd.ssb.compute.hip.bslz4 import Bslz4Chunks, encode_u16
    distinct = min(64, case["frames"])
    frames = _simulate(case, seed, frames=distinct).cpu().numpy()
    chunks = [np.frombuffer(encode_u16(f), dtype=np.uint8) for f in frames]
    rng = np.random.default_rng(seed + 303)
    order = rng.integers(0, distinct, case["frames"])
    sizes = np.array([chunks[i].size for i in order], dtype=np.int64)
    buf = np.concatenate([chunks[i] for i in order])
    shape = (case["det_rows"], case["det_cols"])
    mask = (rng.random(shape) < 1e-3) if case["masked"] else None
    return {"case": case, "chunks": Bslz4Chunks((buf, sizes), (1,) + shape),
            "mask": None if mask is None else torch.tensor(mask.astype(np.uint8), device="cuda"),
            "frames": torch.empty((case["frames"],) + shape, dtype=torch.uint16, device="cuda")}


def _weights(seed: int) -> dict:
    rng = np.random.default_rng(seed + 404)
    shapes = [(32, 144), (64, 288), (64, 576), (64, 576), (256, 256), (3, 256)]
    out = {}
    for i, (o, k) in enumerate(shapes):
        out[f"w{i}"] = (rng.standard_normal((o, k)) * math.sqrt(2.0 / k)).astype(np.float32)
        out[f"b{i}"] = (rng.standard_normal(o) * 0.05).astype(np.float32)
    out["b5"] += np.float32(0.75)                 # early in training: predictions off by a common amount
    return out


def _train_inputs(case: dict, seed: int):
    """Feature maps as the initializer sees them: per scan frequency a
    magnitude in [0, 1] and a phase over pi, zero outside the bright-field
    disk of each 32 x 32 window; targets of order one."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed * 31 + 5)
    b = case["batch"]
    x = torch.rand((b, 32, 32, 16), device="cuda", generator=gen)
    x[..., 1::2] = x[..., 1::2] * 2 - 1
    d = torch.arange(32, device="cuda").float() - 16
    x *= ((d[:, None] ** 2 + d[None, :] ** 2) <= 256.0)[None, :, :, None]
    target = torch.rand((b, 3), device="cuda", generator=gen) * 2 - 1
    return x, target


def _prepare_train(case: dict, seed: int) -> dict:
    from quantem.gpu_amd.ssb.learned import LearnedInit
    net = LearnedInit(seed=1)
    net.load_state_dict(_weights(seed))
    x, target = _train_inputs(case, seed)
    return {"case": case, "net": net, "x": x, "target": target}


# --------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------

def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "recon":
        from quantem.gpu_amd.ssb.compute.hip.engine import normalize_scan
        state["engine"].recon_u16(normalize_scan(state["data"]), case["c10"], case["c12"], 0.3,
                                  math.radians(case["rot"]), obj_out=state["object"], phase_out=state["phase"])
        return {"object": state["object"], "phase": state["phase"]}
    if kind == "session":
        from quantem.gpu_amd.ssb.compute.hip.backend import HipSSBBackend
        ssb = HipSSBBackend(state["data"], semiangle=SEMIANGLE, scan_sampling=_step(case), det_sampling=_ang(case),
                            voltage_kV=300.0, aberrations={"C10": case["c10"], "C12": case["c12"], "phi12": 0.3},
                            rotation_angle_deg=case["rot"])
        result = ssb.result(compute_loss=case["compute_loss"])
        ssb.close()
        return {"object": result.object_wave, "loss": result.loss}
    if kind == "object":
        obj = state["engine"].reconstruct_object(case["c10"], case["c12"], 0.3, phase_out=state["phase"])
        return {"object": obj, "phase": state["phase"]}
    if kind == "loss":
        return state["engine"].batch_phase_loss(*state["trials"])
    if kind == "search":
        state["batch"].set(*state["trials"])
        return state["batch"].phase_variance()
    if kind == "load":
        from quantem.gpu_amd.ssb.compute.hip.binning import bin_frames
        frames = state["chunks"].decode(state["frames"])
        counts = frames.view(torch.int16)         # the same bits: torch computes little on uint16 and uint32
        if case["bin"] == 1:
            return {"frames": counts}
        binned = bin_frames(frames, case["bin"], pixel_mask=state["mask"], dtype=getattr(torch, case["dtype"]))
        return {"frames": counts, "binned": binned.view(torch.int16 if case["dtype"] == "uint16" else torch.int32)}
    net = state["net"]
    loss, grads = net.loss_and_grad(state["x"], state["target"])
    net.apply(grads, 1e-4)
    return {"loss": loss, "grads": grads}


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------

def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "train":
        macs = 16 * 16 * 32 * 144 + 8 * 8 * 64 * 288 + 4 * 4 * 64 * 576 + 2 * 2 * 64 * 576 + 256 * 256 + 256 * 3
        params = 32 * 144 + 64 * 288 + 2 * 64 * 576 + 256 * 256 + 3 * 256 + 32 + 3 * 64 + 256 + 3
        # weights, gradients and the two moments are read and the first three written
        return {"bytes": case["batch"] * 32 * 32 * 16 * 4 + params * 4 * 8, "flops": 6.0 * macs * case["batch"]}
    if kind == "load":
        pixels = case["frames"] * case["det_rows"] * case["det_cols"]
        b = case["bin"]
        binned = case["frames"] * (case["det_rows"] // b) * (case["det_cols"] // b)
        out = 0 if b == 1 else binned * BYTES[case["dtype"]]
        return {"bytes": 2.0 * pixels * 1.06 + out, "flops": 0 if b == 1 else pixels}
    n = _target(case["rows"], case["cols"])
    nbf = math.pi * case["radius"] ** 2
    half = nbf * n * (n // 2 + 1)                 # stored Fourier samples
    fft = 2.5 * nbf * n * n * math.log2(n * n)    # one real transform of every image
    overlap = 30.0 * half                         # overlap factor, product and compensated sum
    raw = case["rows"] * case["cols"] * case["det_rows"] * case["det_cols"] * BYTES[case.get("dtype", "uint16")]
    out = 12.0 * n * n
    if kind == "recon":
        return {"bytes": raw + out, "flops": fft + overlap}
    if kind == "session":
        return {"bytes": raw + out, "flops": fft + overlap + (2 * fft + 2 * overlap if case["compute_loss"] else 0)}
    if kind == "object":
        return {"bytes": 8.0 * half + out, "flops": overlap}
    if kind == "loss":
        return {"bytes": 8.0 * half + 4 * case["trials"], "flops": case["trials"] * (2 * fft + 2 * overlap)}
    return {"bytes": 8.0 * half + 4 * case["trials"], "flops": 2 * overlap * case["trials"]}


# --------------------------------------------------------------------------
# The results in 64 bits
# --------------------------------------------------------------------------

def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "load":
        return None                               # integers
    if kind == "train":
        return _exact_train(case, seed)
    data = _simulate(case, seed)
    geom = _exact_geometry(case, data, _gain(case, seed))
    if kind in ("recon", "object"):
        obj = _exact_object(geom, case["c10"], case["c12"], 0.3)
        return {"object": obj, "phase": torch.angle(obj)}
    if kind == "session":
        obj = _exact_object(geom, case["c10"], case["c12"], 0.3)
        loss = None
        if case["compute_loss"]:
            mags, angles = np.zeros(14), np.zeros(14)
            mags[:2], angles[1] = (case["c10"], case["c12"]), 0.3
            loss = _exact_loss(geom, mags, angles)
        return {"object": obj, "loss": loss}
    mags, angles, rot = _trials(case, seed)
    if case["trials"] * geom["kr"].numel() * geom["n"] ** 2 > (1.2e9 if kind == "loss" else 4.0e9):
        return None                               # over the time this may take
    got = []
    for t in range(case["trials"]):
        g = geom if rot is None else _rotated(geom, float(rot[t]))
        if kind == "loss":
            got.append(_exact_loss(g, mags[t], angles[t]))
        else:
            ph = torch.angle(_exact_object_full(g, mags[t], angles[t]))
            got.append(float((ph - ph.mean()).square().mean()))
    v = torch.tensor(got, dtype=torch.float64)
    return v if kind == "loss" else v[None]


def _as_float(x: torch.Tensor) -> torch.Tensor:
    if x.dtype == torch.uint16:
        return (x.view(torch.int16).to(torch.int32) & 0xFFFF).float()
    return x.float()


def _frame_sum(data: torch.Tensor) -> torch.Tensor:
    """Per-pixel sums over the scan, in 64 bits."""
    flat = data.reshape(-1, data.shape[-2] * data.shape[-1])
    total = 0
    for s in range(0, flat.shape[0], 4096):
        part = flat[s:s + 4096]
        if part.dtype == torch.uint16:
            part = part.view(torch.int16).to(torch.int32) & 0xFFFF
        total = total + part.to(torch.float64).sum(0)   # counts and their sums are below 2^53
    return total.reshape(data.shape[-2], data.shape[-1])


def _exact_geometry(case: dict, data: torch.Tensor, gain) -> dict:
    """Bright-field pixels, their Fourier images and detector coordinates."""
    rows, cols = data.shape[:2]
    n = _target(rows, cols)
    frames = rows * cols
    total = _frame_sum(data)
    mean_src = total / frames
    top, left = (n - min(rows, n)) // 2, (n - min(cols, n)) // 2
    pad = mean_src if data.dtype == torch.float32 else mean_src.trunc()
    pad = pad.float() if data.dtype == torch.float32 else pad
    total = total + pad.double() * (n * n - frames)
    mean = total.float() / torch.tensor(float(n * n), device=data.device)
    if gain is not None:
        mean = mean * gain
    m64 = mean.double()
    probe = m64 > m64.mean() + m64.std(unbiased=False)
    pr, pc = torch.nonzero(probe, as_tuple=True)
    count = int(probe.sum())
    cr = np.float32(np.float32(int(pr.sum())) / np.float32(count))
    cc = np.float32(np.float32(int(pc.sum())) / np.float32(count))
    rr = (torch.arange(mean.shape[0], device=data.device).float() - float(cr)) ** 2
    qq = (torch.arange(mean.shape[1], device=data.device).float() - float(cc)) ** 2
    keep = (mean > 0) & ((rr[:, None] + qq[None, :]) <= float(np.float32(count / math.pi)))
    r, c = torch.nonzero(keep, as_tuple=True)
    images = torch.empty((r.numel(), n, n), dtype=torch.float32, device=data.device)
    images[:] = pad.float()[r, c][:, None, None]
    flat = data.reshape(frames, -1)
    idx = r * data.shape[-1] + c
    for s in range(0, r.numel(), 256):
        cols_ = flat[:, idx[s:s + 256]] if flat.dtype != torch.uint16 else flat.view(torch.int16)[:, idx[s:s + 256]]
        cols_ = _as_float(cols_.view(torch.uint16) if flat.dtype == torch.uint16 else cols_)
        images[s:s + 256, top:top + rows, left:left + cols] = cols_.t().reshape(-1, rows, cols)
    if gain is not None:
        images *= gain[r, c][:, None, None]
    recip = _ang(case) * 1e-3 / WAVELENGTH
    geom = {"n": n, "images": images, "ang": _ang(case) * 1e-3, "dr": (r.double() - float(cr)) * recip,
            "dc": (c.double() - float(cc)) * recip, "dc_value": images.double().sum((1, 2)).mean(),
            "q": torch.fft.fftfreq(n, _step(case), dtype=torch.float64, device=data.device)}
    return _rotated(geom, math.radians(case["rot"]))


def _rotated(geom: dict, angle: float) -> dict:
    ct, st = math.cos(-angle), math.sin(-angle)
    return dict(geom, kr=geom["dr"] * ct + geom["dc"] * st, kc=geom["dc"] * ct - geom["dr"] * st)


_ORDER = np.array([1, 1, 2, 2, 3, 3, 3, 4, 4, 4, 5, 5, 5, 5])
_FOLD = np.array([0, 2, 1, 3, 0, 2, 4, 1, 3, 5, 0, 2, 4, 6])


def _probe(geom: dict, x, y, mags, angles):
    """Soft aperture times exp(-i chi) at the frequencies (x, y)."""
    r2 = x * x + y * y
    alpha = r2.sqrt() * WAVELENGTH
    semi = SEMIANGLE * 1e-3
    aperture = torch.where(r2 > 0, ((semi - alpha) / geom["ang"] + 0.5).clamp(0, 1), torch.ones_like(r2))
    chi = torch.zeros_like(r2)
    phi = None
    for i in range(14):
        if mags[i] == 0.0:
            continue
        o, m = int(_ORDER[i]), int(_FOLD[i])
        term = alpha ** (o + 1) * (float(mags[i]) / (o + 1))
        if m:
            phi = torch.atan2(y, x) if phi is None else phi
            term = term * torch.cos(m * (phi - float(angles[i])))
        chi = chi + term
    return torch.polar(aperture, -2 * math.pi / WAVELENGTH * chi)


def _corrected(geom: dict, b0: int, b1: int, mags, angles):
    """Fourier images times the conjugate normalised overlap factor."""
    kr, kc = geom["kr"][b0:b1, None, None], geom["kc"][b0:b1, None, None]
    q = geom["q"]
    x, y = q[None, :, None], q[None, None, :]
    pk = _probe(geom, kr, kc, mags, angles)
    factor = (_probe(geom, x - kr, y - kc, mags, angles) * pk.conj()
              - _probe(geom, x + kr, y + kc, mags, angles).conj() * pk)
    mag = factor.abs()
    scale = torch.where(mag * mag > 1e-16, 1.0 / mag, torch.full_like(mag, 1e8))
    return torch.fft.fft2(geom["images"][b0:b1].double()) * (factor * scale).conj()


def _chunk(geom: dict) -> int:
    return max(1, (1 << 24) // (geom["n"] ** 2))


def _exact_object_full(geom: dict, mags, angles) -> torch.Tensor:
    total, nb, step = 0, geom["kr"].numel(), _chunk(geom)
    for b in range(0, nb, step):
        total = total + _corrected(geom, b, min(nb, b + step), mags, angles).sum(0)
    total = total / nb
    total[0, 0] = geom["dc_value"]
    return torch.fft.ifft2(total)


def _exact_object(geom: dict, c10: float, c12: float, phi12: float) -> torch.Tensor:
    mags, angles = np.zeros(14), np.zeros(14)
    mags[:2], angles[1] = (c10, c12), phi12
    return _exact_object_full(geom, mags, angles)


def _exact_loss(geom: dict, mags, angles) -> float:
    nb, step = geom["kr"].numel(), _chunk(geom)
    s1 = s2 = 0
    for b in range(0, nb, step):
        c = _corrected(geom, b, min(nb, b + step), mags, angles)
        c[:, 0, 0] = geom["dc_value"]
        ph = torch.angle(torch.fft.ifft2(c))
        s1, s2 = s1 + ph.sum(0), s2 + ph.square().sum(0)
    return float((s2 / nb - (s1 / nb) ** 2).mean())


def _exact_train(case: dict, seed: int) -> dict:
    """Loss and gradients of the network without any rounding to 16 bits."""
    params = {k: torch.tensor(v, dtype=torch.float64, device="cuda", requires_grad=True)
              for k, v in _weights(seed).items()}
    x, target = _train_inputs(case, seed)
    h = x.double()
    for i in range(6):
        w, b = params[f"w{i}"], params[f"b{i}"]
        if i < 4:
            bn, s, _, cin = h.shape
            padded = torch.nn.functional.pad(h, (0, 0, 1, 1, 1, 1))
            taps = [padded[:, dy:dy + s:2, dx:dx + s:2, :] for dy in range(3) for dx in range(3)]
            h = torch.cat(taps, dim=-1) @ w.t() + b
        else:
            h = h.reshape(h.shape[0], -1) @ w.t() + b
        h = torch.relu(h) if i < 5 else h
    loss = (h - target.double()).square().mean()
    names = [k for i in range(6) for k in (f"w{i}", f"b{i}")]
    grads = dict(zip(names, torch.autograd.grad(loss, [params[k] for k in names])))
    return {"loss": loss.detach().reshape(1), "grads": [(grads[f"w{i}"], grads[f"b{i}"]) for i in range(6)]}
