"""The work that a user of this framework has it do, as measurable cases.

Each case is one pass through the public entry points on inputs made from a seed: the forward projector (a
resident and a freshly uploaded phantom, a two-term and a measured-like attenuation table, a voxel grid on and off
the whole-centimetre planes), its differentiable form, the dual-energy decomposition's gradient, the MLEM + TV
iteration, FDK (plan, half-fan plan, one-shot calls) and the batched launch.  `listed()` holds the sizes of the
repository's own workloads and ragged and small ones beside them; `draw()` gives others of the same ranges.
`exact()` restates the computation in 64 bits with torch alone.
"""
from __future__ import annotations

import math

import numpy as np
import torch

PITCH, PITCH_ISO, SAD, PIXNUM = 0.05, 0.032509752, 100.0, 800.0
NMAT = 6
# density fractions (H, C, N, O, P, Ca; g/cc) of the phantoms' tissues: air, water, fat, muscle, lung, bone, marrow
TISSUES = ((0.0, 0.0, 0.001, 0.0, 0.0, 0.0), (0.111, 0.0, 0.0, 0.888, 0.0, 0.0), (0.108, 0.568, 0.007, 0.264, 0.0, 0.0),
           (0.107, 0.150, 0.036, 0.753, 0.002, 0.0), (0.027, 0.027, 0.008, 0.193, 0.0, 0.0),
           (0.065, 0.298, 0.081, 0.835, 0.198, 0.433), (0.107, 0.580, 0.015, 0.302, 0.001, 0.0))


# --------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # the headline: one phantom resident on the GPU, a full half-fan scan of it (0.5 mm / 1 mm voxels, 115 mm
        # panel offset, 91 energy bins)
        dict(name="forward_full_scan", kind="forward", N=512, Nz=128, s=0.05, t=0.1, nA=360, H=400, W=400, shift=1.15,
             table="two_term", upload=False),
        # the shipped 36-angle example: a new phantom is uploaded and projected with a table of measured rank (no
        # low-rank form, so the six elemental maps themselves are traversed)
        dict(name="forward_measured_table", kind="forward", N=512, Nz=64, s=0.05, t=0.1, nA=36, H=400, W=400, shift=0.0,
             table="measured", upload=True),
        # a phantom on a clinical CT grid (0.9766 mm pixels: the whole-cm planes fall inside voxels), ragged sizes
        dict(name="forward_ct_grid", kind="forward", N=320, Nz=77, s=0.09765625, t=0.125, nA=120, H=300, W=324,
             shift=0.4, table="two_term", upload=True),
        # a quick look at a coarse phantom (2 mm voxels): latency and launches
        dict(name="forward_preview", kind="forward", N=96, Nz=25, s=0.2, t=0.2, nA=12, H=72, W=80, shift=0.0,
             table="two_term", upload=True),
        # one gradient step of a reconstruction through the differentiable projector (forward and backward)
        dict(name="gradient", kind="gradient", N=256, Nz=64, s=0.1, t=0.1, nA=90, H=256, W=256, table="two_term",
             form="autograd"),
        # the smallest gradient a fit runs on, with a measured-rank table
        dict(name="gradient_small", kind="gradient", N=64, Nz=20, s=0.5, t=0.4, nA=24, H=60, W=52, table="measured",
             form="loss"),
        # one problem of a dual-energy decomposition iteration: new maps, both spectra's loss and its gradient
        dict(name="dual_energy", kind="dual", N=512, Nz=64, s=0.05, t=0.1, nA=360, H=400, W=400),
        # one iteration of the MLEM + TV loop
        dict(name="mlem_tv", kind="mlem", N=256, Nz=64, s=0.1, t=0.1, nA=360, H=400, W=400),
        # reconstruction of a full scan with a plan kept for the geometry
        dict(name="fdk_plan", kind="fdk", nA=360, H=400, W=400, R=270, Z=128, step=0.1, scale=0.1, shift=0.0,
             half_fan=False, alpha=0.5),
        # the same for the offset panel: weighted and padded inside the filter
        dict(name="fdk_half_fan", kind="fdk", nA=360, H=400, W=400, R=270, Z=128, step=0.1, scale=0.1, shift=11.5,
             half_fan=True, alpha=0.5),
        # the one-shot calls, as the drop-in program makes them, on the 36-projection example
        dict(name="fdk_one_shot", kind="fdk_once", nA=36, H=400, W=400, R=270, Z=64, step=0.1, scale=0.1),
        # a batch of uneven phantoms, each projected and reconstructed in one launch sequence
        dict(name="batch", kind="batch", N=512, s=0.05, t=0.1, slices="64,100,161", nA=180, H=400, W=400, R=270,
             Z=100),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: the kinds as often as they are listed, sizes over their whole range."""
    kind = rng.choice(("forward", "forward", "forward", "gradient", "gradient", "dual", "mlem", "fdk", "fdk",
                       "fdk_once", "batch"))
    H = _log_int(rng, 48, 400)
    W = max(48, min(400, int(H * rng.uniform(0.7, 1.5))))
    if kind in ("fdk", "fdk_once"):
        half = kind == "fdk" and rng.random() < 0.4
        c = dict(kind=kind, nA=_log_int(rng, 24, 360), H=H, W=W, R=_log_int(rng, 64, 270), Z=_log_int(rng, 16, 128),
                 step=rng.choice((0.1, 0.15, 0.2)), scale=rng.choice((0.07, 0.1, 0.125)))
        if kind == "fdk":
            c.update(shift=round(rng.uniform(4.0, 11.5), 2) if half else 0.0, half_fan=half,
                     alpha=rng.choice((0.5, 0.5, 1.0)))
        return c
    N = _log_int(rng, 64, 512)
    if rng.random() < 0.7:  # planes on voxel boundaries
        s = min((0.05, 0.1, 0.2, 0.25, 0.5), key=lambda v: abs(v * N - 26.0))
    else:  # a field of view divided by the grid
        s = round(rng.uniform(24.0, 32.0) / N, 5)
    t = rng.choice((0.05, 0.1, 0.125, 0.2, 0.3)) if N > 128 else rng.choice((0.2, 0.25, 0.4, 0.5))
    c = dict(kind=kind, N=N, Nz=_log_int(rng, 12, 128), s=s, t=t, nA=_log_int(rng, 8, 360), H=H, W=W)
    if kind == "forward":
        c.update(shift=round(rng.choice((0.0, rng.uniform(0.2, 1.15))), 3), table=rng.choice(("two_term", "measured")),
                 upload=rng.random() < 0.6)
    elif kind == "gradient":
        c.update(table=rng.choice(("two_term", "measured")), form=rng.choice(("autograd", "loss")))
    elif kind == "batch":
        c.pop("Nz")
        c.update(slices=",".join(str(_log_int(rng, 16, 160)) for _ in range(rng.choice((2, 3)))),
                 R=_log_int(rng, 64, 270), Z=_log_int(rng, 16, 100))
        c["nA"] = min(c["nA"], 180)
    if kind in ("gradient", "dual", "mlem"):  # an iterated step: at most the listed work
        c["Nz"] = min(c["Nz"], 64)
    return c


# --------------------------------------------------------------------------------------------------- inputs
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _gen(seed):
    return torch.Generator(device="cpu").manual_seed(int(seed) & 0x7FFFFFFF)


def _uniform(g, lo, hi):
    return float(torch.rand((), generator=g, dtype=torch.float64)) * (hi - lo) + lo


def _tables(kvp, kind):
    """(attenuation [6][NE] cm^2/g FP32, pdf [NE] FP32) on 1 keV bins from 10 keV: photoelectric + Compton
    ("two_term"), or with element-dependent slopes and a coherent term ("measured", of full rank)."""
    e = np.arange(10, kvp + 1, dtype=np.float64) + 0.5
    z = np.array([1, 6, 7, 8, 15, 20], np.float64)
    a = np.array([1.008, 12.011, 14.007, 15.999, 30.974, 40.078])
    k = e / 510.99895
    l1 = np.log1p(2 * k)
    kn = 2 * np.pi * 2.8179403262e-13 ** 2 * ((1 + k) / k ** 2 * (2 * (1 + k) / (1 + 2 * k) - l1 / k) + l1 / (2 * k)
                                             - (1 + 3 * k) / (1 + 2 * k) ** 2)
    comp = (z / a)[:, None] * 6.02214076e23 * kn[None, :]
    if kind == "two_term":
        mu = z[:, None] ** 4 / e[None, :] ** 3 + comp
    else:
        slope = np.array([3.25, 3.16, 3.13, 3.10, 3.01, 2.93])
        mu = (20.0 * z[:, None] ** 3.1 / 8.0 * e[None, :] ** -slope[:, None]
              + comp * (1.0 - np.exp(-e[None, :] / (0.9 * z[:, None] ** 0.667)))
              + 0.9 * z[:, None] ** 1.6 / e[None, :] ** (1.75 + 0.006 * z[:, None]))
    f = np.maximum(0.0, (kvp - e) / e) + 0.3 * (np.exp(-0.5 * (e - 59.0) ** 2) + np.exp(-0.5 * (e - 67.0) ** 2)) * (kvp > 70)
    return mu.astype(np.float32), (f / f.sum()).astype(np.float32)


def _angles(n):
    return np.deg2rad(-180.0 + 360.0 / n * np.arange(n) + 1e-4)


def _trig(c):
    """cos, sin and the panel's centre columns / rows per angle (both centres go by the panel's height)."""
    ang = _angles(c["nA"])
    pix = PITCH * (PIXNUM / c["H"])
    n = len(ang)
    xc = np.full(n, -c["H"] / 2.0 - c.get("shift", 0.0) * 10.0 / pix)
    xc = xc + (c["H"] - c["W"]) / 2.0  # panels that are not square stay centred on the axis
    return np.cos(ang), np.sin(ang), xc, np.full(n, -c["H"] / 2.0)


def _labels(c, seed, Nz=None):
    """Tissue labels [z][y][x]: a body ellipse in air and seeded ellipsoids of other tissues."""
    g, dev = _gen(seed), _device()
    N, Nz = c["N"], Nz or c["Nz"]
    fx, fz = min(N * c["s"], 30.0) / 2, Nz * c["t"] / 2
    x = ((torch.arange(N, device=dev) - N / 2 + 0.5) * c["s"])
    z = ((torch.arange(Nz, device=dev) - Nz / 2 + 0.5) * c["t"])
    X, Y, Zg = x[None, None, :], x[None, :, None], z[:, None, None]
    ax, ay = fx * _uniform(g, 0.75, 0.9), fx * _uniform(g, 0.6, 0.8)
    lab = torch.where((X / ax) ** 2 + (Y / ay) ** 2 + 0 * Zg <= 1.0, 1, 0).to(torch.uint8)
    for i in range(14):
        cx, cy, cz = _uniform(g, -0.6, 0.6) * ax, _uniform(g, -0.6, 0.6) * ay, _uniform(g, -1.0, 1.0) * fz
        rx, ry, rz = (_uniform(g, 0.05, 0.3) * fx for _ in range(3))
        inside = ((X - cx) / rx) ** 2 + ((Y - cy) / ry) ** 2 + ((Zg - cz) / rz) ** 2 <= 1.0
        lab[inside & (lab > 0)] = 2 + (i + int(seed)) % (len(TISSUES) - 2)
    return lab


def _u16_volume(c, seed, Nz=None):
    """uint16 densities x 1000, [z][mat][y][x] (as an int16 tensor)."""
    lab = _labels(c, seed, Nz).long()
    lut = (torch.tensor(TISSUES, dtype=torch.float64, device=lab.device) * 1000.0).to(torch.int16)
    return torch.stack([lut[:, m][lab] for m in range(NMAT)], 1).contiguous()


def _maps(c, seed):
    """FP32 maps [mat][z][y][x] of a fit in progress: tissue densities with 5 % of texture."""
    lab = _labels(c, seed).long()
    lut = torch.tensor(TISSUES, dtype=torch.float32, device=lab.device)
    tex = torch.rand(lab.shape, generator=torch.Generator(device=lab.device).manual_seed(int(seed) + 1), device=lab.device)
    return torch.stack([lut[:, m][lab] * (0.95 + 0.1 * tex) for m in range(NMAT)]).contiguous()


def _line_lengths(n, H, W, ang, shift_px, seed, flip):
    """Path lengths [cm] [n][H][W] through a seeded set of spheres seen from a circular orbit."""
    g, dev = _gen(seed), _device()
    u = ((torch.arange(W, device=dev) - W / 2 + 0.5 - shift_px) * (PITCH_ISO * PIXNUM / W)).view(1, 1, W)
    v = ((torch.arange(H, device=dev) - H / 2 + 0.5) * (PITCH_ISO * PIXNUM / (W if flip else H))).view(1, H, 1)
    a = torch.tensor(ang, dtype=torch.float32, device=dev).view(-1, 1, 1)
    ca, sa = torch.cos(a), torch.sin(a)
    sx, sy = -SAD * sa, SAD * ca
    dx, dy, dz = u * ca - sx, u * sa - sy, v
    d2 = dx * dx + dy * dy + dz * dz
    total = torch.zeros((n, H, W), device=dev)
    for i in range(6):
        r = _uniform(g, 7.0, 9.0) if i == 0 else _uniform(g, 0.8, 3.0)
        cx, cy, cz = (0.0, 0.0, 0.0) if i == 0 else (_uniform(g, -4, 4), _uniform(g, -4, 4), _uniform(g, -3, 3))
        weight = 1.0 if i == 0 else _uniform(g, -0.4, 0.8)
        ox, oy, oz = sx - cx, sy - cy, -cz
        b = ox * dx + oy * dy + oz * dz
        disc = b * b - d2 * (ox * ox + oy * oy + oz * oz - r * r)
        total += weight * 2.0 * torch.sqrt(disc.clamp_(min=0.0) / d2)
    return total.clamp_(min=0.0)


def _transmissions(n, H, W, ang, shift_px, seed):
    """Noisy transmissions in (0, 1] as a detector gives them."""
    q = 0.2 * _line_lengths(n, H, W, ang, shift_px, seed, True)
    noise = torch.randn(q.shape, generator=torch.Generator(device=q.device).manual_seed(int(seed) + 2), device=q.device)
    return (torch.exp(-q) * (1.0 + 0.004 * noise)).clamp_(min=1e-4).contiguous()


def _projector(c, Nz=None):
    from virtualcbct_amd.projector import Projector
    return Projector(c["N"], c["s"], Nz or c["Nz"], c["t"], c["H"], c["W"], c["nA"], *_trig(c))


def _targets(c, seed, spectra):
    """Measured log projections of another object: path lengths times each spectrum's effective attenuation."""
    q = _line_lengths(c["nA"], c["H"], c["W"], _angles(c["nA"]), 0.0, seed + 5, False)
    mus = []
    for mu, pdf in spectra:
        w = np.array(TISSUES[1]) @ mu.astype(np.float64)
        mus.append(-math.log(float((pdf * np.exp(-10.0 * w)).sum() / pdf.sum())) / 10.0)
    return torch.stack([m * q for m in mus]).contiguous()


def _fdk_angles(c):
    n = c["nA"]
    return _angles(n)[::-1].copy(), np.full(n, float(c.get("shift", 0.0))), np.zeros(n)


def _zstart(c):
    return -int(c["Z"] * c.get("step", 0.1) / 2)


def _plan(c, **kw):
    from virtualcbct_amd.fdk import FdkPlan
    a, xs, ys = _fdk_angles(c)
    return FdkPlan(c["H"], c["W"], c["nA"], c["R"], c["Z"], _zstart(c), c.get("step", 0.1), c.get("scale", 0.1), 1000,
                   a, xs, ys, **kw)


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "forward":
        P = _projector(c)
        P.set_spectrum(*_tables(100, c["table"]))
        vol = _u16_volume(c, seed)
        if not c["upload"]:
            P.set_volume(vol)
            vol = None
        out = torch.empty(P.shape_proj, dtype=torch.float32, device="cuda")
        return dict(kind=kind, P=P, vol=vol, out=out)
    if kind == "gradient":
        P = _projector(c)
        spec = _tables(100, c["table"])
        P.set_spectrum(*spec)
        maps = _maps(c, seed)
        target = _targets(c, seed, [spec])[0].contiguous()
        if c["form"] == "autograd":
            maps.requires_grad_(True)
        return dict(kind=kind, form=c["form"], P=P, maps=maps, target=target)
    if kind == "dual":
        P = _projector(c)
        spectra = [_tables(kv, "two_term") for kv in (80, 120)]
        P.set_spectra(spectra)
        return dict(kind=kind, P=P, maps=_maps(c, seed), targets=_targets(c, seed, spectra),
                    grad=torch.empty(P.shape_maps, dtype=torch.float32, device="cuda"),
                    loss=torch.zeros(1, dtype=torch.float64, device="cuda"))
    if kind == "mlem":
        from virtualcbct_amd.iterative import MlemTV
        P = _projector(c)
        b = (0.2 * _line_lengths(c["nA"], c["H"], c["W"], _angles(c["nA"]), 0.0, seed, False)).contiguous()
        solver = MlemTV(P, np.full(NMAT, 0.2), b, weight_tv=1e-5)
        lab = _labels(c, seed)
        tex = torch.randint(0, 60, lab.shape, generator=torch.Generator(device=lab.device).manual_seed(int(seed) + 3),
                            device=lab.device)
        x = torch.where(lab > 0, 870 + 25 * lab.int() + tex, 2 + 0 * tex).to(torch.int16).contiguous()
        return dict(kind=kind, solver=solver, x=x)
    if kind in ("fdk", "fdk_once"):
        a, xs, ys = _fdk_angles(c)
        shift_px = xs[0] / (0.05 * 800 / c["W"])
        proj = _transmissions(c["nA"], c["H"], c["W"], a, shift_px, seed)
        if kind == "fdk_once":
            return dict(kind=kind, proj=proj, a=a, xs=xs, ys=ys, c=dict(c))
        plan = _plan(c, half_fan=c["half_fan"], window_alpha=c["alpha"])
        filtered = torch.empty(plan.shape_filtered, dtype=torch.float32, device="cuda")
        return dict(kind=kind, plan=plan, proj=proj, filtered=filtered)
    if kind == "batch":
        from virtualcbct_amd.batch import Batch
        B = Batch()
        spec = _tables(100, "two_term")
        outs, recons, keep = [], [], []
        for i, Nz in enumerate(int(v) for v in c["slices"].split(",")):
            P = _projector(c, Nz)
            P.set_spectrum(*spec)
            P.set_volume(_u16_volume(c, seed + 31 * i, Nz))
            out = torch.empty(P.shape_proj, dtype=torch.float32, device="cuda")
            plan = _plan(c)
            filt = torch.empty(plan.shape_filtered, dtype=torch.float32, device="cuda")
            rec = torch.empty(plan.shape_recon, dtype=torch.float32, device="cuda")
            B.add_forward(P, out, 1000.0)
            B.add_fdk(plan, out, filt, rec)
            outs.append(out)
            recons.append(rec)
            keep += [P, plan, filt]
        return dict(kind=kind, B=B, outs=outs, recons=recons, keep=keep)
    raise ValueError(kind)


def run(state):
    st, kind = state, state["kind"]
    if kind == "forward":
        if st["vol"] is not None:
            st["P"].set_volume(st["vol"])
        return st["P"].forward(1000.0, out=st["out"])
    if kind == "gradient":
        if st["form"] == "loss":
            st["P"].set_volume(st["maps"])
            grad, loss = st["P"].adjoint(st["target"], 1.0)
            return dict(grad=grad, loss=loss)
        from virtualcbct_amd.autograd import poly_logproj
        st["maps"].grad = None
        p = poly_logproj(st["maps"], st["P"], 1.0)
        ((p - st["target"]) ** 2).sum().backward()
        return dict(p=p.detach(), grad=st["maps"].grad)
    if kind == "dual":
        st["P"].set_volume(st["maps"])
        grad, loss = st["P"].multi_loss_grad(st["targets"], 1.0, grad=st["grad"], loss=st["loss"])
        return dict(grad=grad, loss=loss)
    if kind == "mlem":
        return st["solver"].step(st["x"])
    if kind == "fdk":
        rec = st["plan"].execute(st["proj"], filtered=st["filtered"])
        return dict(filtered=st["filtered"], recon=rec)
    if kind == "fdk_once":
        from virtualcbct_amd.fdk import fdk_device
        c = st["c"]
        return fdk_device(st["proj"], _zstart(c), c["step"], c["scale"], c["R"], c["Z"], 1000, st["a"], st["xs"], st["ys"])
    st["B"].run()
    return dict(proj=list(st["outs"]), recon=list(st["recons"]))


# --------------------------------------------------------------------------------------------------- work
def _segments(c, Nz):
    """Voxels crossed by all rays, roughly: for each ray its share of the volume's height times its path."""
    fov = c["N"] * c["s"]
    pix = PITCH_ISO * PIXNUM / c["H"]
    rows = min(c["H"], Nz * c["t"] / pix)
    cols = min(c["W"], fov / pix)
    return c["nA"] * rows * cols * c["N"] * 0.78 * 1.25


def work(case):
    """Bytes: inputs read once and outputs written once.  Operations: a multiply-add per channel and crossed voxel (two
    channels where the table has a two-term form), the spectral sums, a filter's transforms, and 8 per sampled pixel
    of a backprojection."""
    c, kind = case, case["kind"]
    if kind in ("fdk", "fdk_once"):
        px = c["nA"] * c["H"] * c["W"]
        vox = c["R"] ** 2 * c["Z"]
        bytes_ = 4.0 * px + 4.0 * vox + (4.0 * px if kind == "fdk" else 0.0)
        return dict(bytes=bytes_, flops=px * 2 * 5 * 2 * math.log2(2 * c["W"]) + 0.785 * vox * c["nA"] * 8.0)
    rays = c["nA"] * c["H"] * c["W"]
    if kind == "batch":
        b = f = 0.0
        for Nz in (int(v) for v in c["slices"].split(",")):
            b += 12.0 * c["N"] ** 2 * Nz + 8.0 * rays + 4.0 * c["R"] ** 2 * c["Z"]
            f += 4.0 * _segments(c, Nz) + rays * 91 * 6.0 + 0.785 * c["R"] ** 2 * c["Z"] * c["nA"] * 8.0
        return dict(bytes=b, flops=f)
    vox, seg = c["N"] ** 2 * c["Nz"], _segments(c, c["Nz"])
    ch = 2 if c.get("table", "two_term") == "two_term" else 6
    if kind == "forward":
        return dict(bytes=12.0 * vox + 4.0 * rays, flops=2.0 * ch * seg + rays * 91 * (2.0 * ch + 2))
    if kind == "gradient":
        return dict(bytes=48.0 * vox + 8.0 * rays, flops=4.0 * ch * seg + rays * 91 * (4.0 * ch + 4))
    if kind == "dual":
        return dict(bytes=48.0 * vox + 8.0 * rays, flops=8.0 * seg + rays * 182 * 12.0)
    return dict(bytes=8.0 * vox + 4.0 * rays, flops=4.0 * seg)  # mlem: one channel, there and back


# --------------------------------------------------------------------------------------------------- 64 bits
def _trace(c, Nz, a0, a1, visit):
    """Walks every ray of the angles [a0, a1) over the planes of its major axis, as the projector defines its
    segments, in 64 bits; visit(rays, cells, lengths) is called with the charged segments (cells index [z][y][x]).
    Returns the cos^3 factor of each ray."""
    dev, f8 = _device(), torch.float64
    N, s, t, H, W = c["N"], c["s"], c["t"], c["H"], c["W"]
    cs, sn, xc, yc = (torch.tensor(v[a0:a1], dtype=f8, device=dev).view(-1, 1, 1) for v in _trig(c))
    j = torch.arange(H, device=dev, dtype=f8).view(1, H, 1)
    jj = torch.arange(W, device=dev, dtype=f8).view(1, 1, W)
    shape = (a1 - a0, H, W)
    pz = (-(yc + j) * PITCH_ISO * (PIXNUM / H)).expand(shape).reshape(-1)
    pr = (PITCH_ISO * (xc + jj) * (PIXNUM / H)).expand(shape)
    px, py = (pr * cs).reshape(-1), (pr * sn).reshape(-1)
    sx, sy = (-SAD * sn).expand(shape).reshape(-1), (SAD * cs).expand(shape).reshape(-1)
    leng = SAD * SAD / (SAD * SAD + (pr.reshape(-1) ** 2 + pz * pz))
    leng = leng * torch.sqrt(leng)
    nxm, nzm = int(N * 0.5), int(Nz * 0.5)
    lim, rmax = nxm * s, N * 0.5 * s
    # the first two hits with the box, in the order y = +lim, y = -lim, x = +lim, x = -lim
    hits = []
    for axis, at in ((1, lim), (1, -lim), (0, lim), (0, -lim)):
        if axis:
            f = (at - sy) / (py - sy)
            x, y = f * (px - sx) + sx, torch.full_like(sy, at)
            ok = x.abs() < lim
        else:
            f = (at - sx) / (px - sx)
            x, y = torch.full_like(sx, at), f * (py - sy) + sy
            ok = y.abs() < lim
        hits.append((ok, x, y, f * pz))
    seen = torch.zeros_like(sx, dtype=torch.int64)
    first = [torch.zeros_like(sx) for _ in range(3)]
    second = [torch.zeros_like(sx) for _ in range(3)]
    for ok, *h in hits:
        for q in range(3):
            first[q] = torch.where(ok & (seen == 0), h[q], first[q])
            second[q] = torch.where(ok & (seen == 1), h[q], second[q])
        seen += ok
    d0 = sum((p - o) ** 2 for p, o in zip(first, (sx, sy, 0.0)))
    d1 = sum((p - o) ** 2 for p, o in zip(second, (sx, sy, 0.0)))
    near = d0 < d1
    (xi, yi, zi), (xf, yf, zf) = ([torch.where(near, p, q) for p, q in zip(a, b)]
                                  for a, b in ((first, second), (second, first)))
    # rays that can reach the volume's height (the others charge nothing)
    reach = (seen >= 2) & (torch.minimum(zi, zf) < (nzm + 2) * t + 1.0) & (torch.maximum(zi, zf) > (nzm - Nz - 1) * t - 1.0)
    ray = reach.nonzero().squeeze(1)
    if not len(ray):
        return leng
    pick = lambda *v: [x[ray] for x in v]  # noqa: E731
    sx, sy, px, py, pz, xi, yi, zi, xf, yf, zf = pick(sx, sy, px, py, pz, xi, yi, zi, xf, yf, zf)
    xm = (xi - xf).abs() > (yi - yf).abs()
    w = lambda a, b: torch.where(xm, a, b)  # noqa: E731
    su, sv, pu, pv, ui, vi, uf, vf = w(sx, sy), w(sy, sx), w(px, py), w(py, px), w(xi, yi), w(yi, xi), w(xf, yf), w(yf, xf)
    pha, dirv, dirz = torch.sign(uf - ui), torch.sign(vf - vi), torch.sign(zf - zi)
    uin = torch.trunc(ui) + torch.where(ui * (uf - ui) > 0, pha, torch.zeros_like(pha))

    def index(a, b, flipped, scale, n):
        q = torch.where(flipped, -(a + b), a + b) * 0.5 / scale + n
        return torch.trunc(q).long()

    def charge(a, b, on):
        (ua, va, za), (ub, vb, zb) = a, b
        iu = index(ua, ub, ~xm, s, nxm)
        iv = index(va, vb, xm, s, nxm)
        iz = index(za, zb, torch.ones_like(xm), t, nzm)
        on = on & (iu >= 0) & (iu < N) & (iv >= 0) & (iv < N) & (iz >= 0) & (iz < Nz)
        on = on & (torch.sqrt((ua + ub) ** 2 + (va + vb) ** 2) * 0.5 < rmax)
        k = on.nonzero().squeeze(1)
        if len(k):
            x, y = torch.where(xm, iu, iv)[k], torch.where(xm, iv, iu)[k]
            length = torch.sqrt((ua - ub) ** 2 + (va - vb) ** 2 + (za - zb) ** 2)[k]
            visit(ray[k], (iz[k] * N + y) * N + x, length)

    def at_u(u):
        f = (u - su) / (pu - su)
        return u, f * (pv - sv) + sv, f * pz

    u, v, z = at_u(uin)
    last = (ui, vi, zi)
    alive = (u.abs() <= lim) & (v.abs() <= lim)
    vma = zma = None
    for k in range(8 * N):
        here = at_u(uin + pha * k * s)
        u, v0, z0 = here[0], v, z
        v, z = here[1], here[2]
        vmb, zmb = vma, zma
        vma, zma = torch.trunc(v / s), torch.trunc(z / t)
        if k:
            hv = alive & ((vma != vmb) | (torch.sign(v) != torch.sign(v0)))
            hz = alive & (zma != zmb)
            vb = vma * s - torch.where(((v <= 0) & (dirv < 0)) | ((v >= 0) & (dirv > 0)), torch.zeros_like(v), dirv * s)
            f = (vb - sv) / (pv - sv)
            cv = (f * (pu - su) + su, vb, f * pz)
            zb = zma * t - torch.where(((z < 0) & (dirz < 0)) | ((z > 0) & (dirz > 0)), torch.zeros_like(z), dirz * t)
            f = zb / pz
            cz = (f * (pu - su) + su, f * (pv - sv) + sv, zb)
            dist = lambda q: sum((p - o) ** 2 for p, o in zip(here, q))  # noqa: E731
            zero = torch.zeros_like(z)
            chv, chz = torch.where(hv, dist(cv), zero), torch.where(hz, dist(cz), zero)
            both = hv & hz
            zfirst, vfirst = both & (chz > chv), both & (chz < chv)
            onlyz, onlyv = hz & ~hv & (chz != 0), hv & ~hz & (chv != 0)
            m1z, m1v = zfirst | onlyz, vfirst | onlyv
            e1 = tuple(torch.where(m1z, p, torch.where(m1v, q, o)) for p, q, o in zip(cz, cv, here))
            e2 = tuple(torch.where(zfirst, q, torch.where(vfirst, p, o)) for p, q, o in zip(cz, cv, here))
            charge(last, e1, alive)
            charge(e1, e2, alive & (m1z | m1v))
            charge(e2, here, alive & (zfirst | vfirst))
        else:
            charge(last, here, alive)
        last = here
        alive = alive & (u.abs() <= lim) & (v.abs() <= lim)
        if k % 16 == 15 and not bool(alive.any()):
            break
    return leng


LIMIT = 4.5e9  # ray-steps that the 64-bit walk is worth


def _chunks(c, Nz):
    per = max(1, int(3.0e6 // (c["H"] * c["W"])))
    return [(a, min(a + per, c["nA"])) for a in range(0, c["nA"], per)]


def _line_integrals(c, Nz, cells):
    """[nA*H*W][6] from cells [z*y*x][6], and the cos^3 factors."""
    L = torch.zeros((c["nA"] * c["H"] * c["W"], NMAT), dtype=torch.float64, device=cells.device)
    leng = []
    for a0, a1 in _chunks(c, Nz):
        part = L[a0 * c["H"] * c["W"]: a1 * c["H"] * c["W"]]

        def visit(ray, cell, length):
            part.index_add_(0, ray, cells[cell].double() * length[:, None])

        leng.append(_trace(c, Nz, a0, a1, visit))
    return L, torch.cat(leng)


def _flip(c, v):
    """[rays] in kernel row order -> [nA][H][W] with the rows reversed."""
    return v.view(c["nA"], c["H"], c["W"]).flip(1)


def _intensity(c, seed, Nz, table):
    vol = _u16_volume(c, seed, Nz)
    cells = vol.permute(0, 2, 3, 1).reshape(-1, NMAT).to(torch.int32).bitwise_and(0xFFFF).float()
    L, leng = _line_integrals(c, Nz, cells)
    mu, pdf = (torch.tensor(v.astype(np.float64), device=L.device) for v in table)
    out = torch.zeros(len(L), dtype=torch.float64, device=L.device)
    for e in range(len(pdf)):
        out += pdf[e] * torch.exp(-(L @ mu[:, e]) / 1000.0) * leng
    return _flip(c, out)


def _gradient(c, seed, table):
    maps = _maps(c, seed)
    cells = maps.permute(1, 2, 3, 0).reshape(-1, NMAT).contiguous()
    L, _ = _line_integrals(c, c["Nz"], cells)
    mu, pdf = (torch.tensor(v.astype(np.float64), device=L.device) for v in table)
    x = L @ mu
    low = x.min(1, keepdim=True).values
    we = pdf * torch.exp(-(x - low))
    p = low[:, 0] - torch.log(we.sum(1) / pdf.sum())
    mubar = (we @ mu.T) / we.sum(1, keepdim=True)
    target = _flip(c, _targets(c, seed, [table])[0].double().reshape(-1)).reshape(-1)
    res = p - target
    coef = 2.0 * res[:, None] * mubar
    grad = torch.zeros_like(cells, dtype=torch.float64)
    for a0, a1 in _chunks(c, c["Nz"]):
        part = coef[a0 * c["H"] * c["W"]: a1 * c["H"] * c["W"]]
        _trace(c, c["Nz"], a0, a1, lambda ray, cell, length: grad.index_add_(0, cell, part[ray] * length[:, None]))
    grad = grad.view(c["Nz"], c["N"], c["N"], NMAT).permute(3, 0, 1, 2).contiguous()
    return _flip(c, p), grad, (res * res).sum().view(1)


def _ramp(W, pitch, alpha):
    """The filter's taps h(d), d = -(W-1) .. W-1, in 64 bits."""
    cut, const = 1.60, 1.0 / (8.0 * math.pi ** 2 * pitch * 800 / W)
    d = np.arange(-(W - 1), W, dtype=np.float64)
    d[W - 1] = 1.0
    theta, delta = math.pi * cut * d, cut * d
    eta, xi = 1.0 / (1.0 - 1.0 / delta), 1.0 / (1.0 + 1.0 / delta)
    ct, st, b = np.cos(theta), np.sin(theta), 1.0 - alpha
    co, so = math.cos(math.pi), math.sin(math.pi)
    h = const / d / d * (2 * alpha * theta * st + 2 * alpha * (ct - 1) + xi * b * theta * (st * co + ct * so)
                         + eta * b * theta * (st * co - ct * so) + xi * xi * b * (ct * co - st * so - 1)
                         + eta * eta * b * (ct * co + st * so - 1))
    h[W - 1] = cut * cut / 4.0 / (pitch * 800 / W) * (alpha * 0.5 + b * (so / math.pi + (co - 1.0) / math.pi ** 2))
    return h


def _fdk(proj, c, a, xs, ys, alpha=0.5, half_fan=False):
    """(filtered, recon) in 64 bits."""
    dev, f8 = proj.device, torch.float64
    n, H, W = proj.shape
    q = -torch.log(proj.double())
    pitch = PITCH_ISO
    if half_fan:
        pix = 0.05 * 800 / W
        sh = xs / pix
        pad = int(round(2.0 * abs(sh).max()))
        off = 0 if sh.max() > 0 else pad
        Wo = W + pad
        col = torch.arange(W, dtype=f8, device=dev)[None, :]
        centre = torch.tensor(W / 2.0 + sh - 0.5, device=dev)[:, None]
        side = torch.tensor(np.where(sh > 0, -1.0, 1.0), device=dev)[:, None]
        tau = torch.tensor(W / 2.0 - abs(sh), device=dev)[:, None]
        r = ((col - centre) * side / tau).clamp(-1.0, 1.0)
        w2 = 2.0 * torch.sin(math.pi / 4 * (1.0 + r)) ** 2
        q = torch.nn.functional.pad(q * w2[:, None, :], (off, Wo - W - off))
        xs, ys = (sh + off - pad / 2.0) * (0.05 * 800 / Wo), (ys / pix - pad / 2.0) * (0.05 * 800 / Wo)
        pitch, W = PITCH_ISO * Wo / W, Wo
    pw = pitch * 800 / W
    length = 1 << (3 * W).bit_length()
    h = torch.fft.rfft(torch.tensor(_ramp(W, pitch, alpha), device=dev), n=length)
    filt = torch.empty((n, H, W), dtype=f8, device=dev)
    m, row = torch.arange(W, dtype=f8, device=dev), torch.arange(H, dtype=f8, device=dev)
    for k in range(n):
        y = torch.fft.irfft(torch.fft.rfft(q[k], n=length) * h, n=length)[:, W - 1: 2 * W - 1]
        p1 = (-W / 2.0 - xs[k] / (0.05 * 800 / W) - 1 + m).abs() * pw
        p2 = (-W / 2.0 - ys[k] / (0.05 * 800 / W) - 1 + row).abs() * pw
        filt[k] = y * (100.0 / torch.sqrt(10000.0 + p1[None, :] ** 2 + p2[:, None] ** 2))
    R, Z = c["R"], c["Z"]
    rad, centre = (R - 1) / 2.0, R / 2.0 - 0.5
    i = torch.arange(R, dtype=f8, device=dev)
    xx, yy = ((i - centre) * c.get("scale", 0.1))[None, :], (-(i - centre) * c.get("scale", 0.1))[:, None]
    inside = (i[:, None] - rad) ** 2 + (i[None, :] - rad) ** 2 <= rad * rad
    zz = (_zstart(c) + torch.arange(Z, dtype=f8, device=dev) * c.get("step", 0.1))[:, None, None]
    rec = torch.zeros((Z, R, R), dtype=f8, device=dev)
    for k in range(n):
        if k in (0, n - 1):
            dbeta = abs(a[1] - a[0]) / 2 if k == 0 else abs(a[-1] - a[-2]) / 2
        else:
            dbeta = abs(a[k + 1] - a[k - 1]) / 2
            if dbeta > math.pi / 2:
                dbeta = abs(a[k + 1] + (2 if a[k + 1] < 0 else -2) * math.pi - a[k - 1]) / 2
        co, si = math.cos(a[k]), math.sin(a[k])
        X, Y = xx * co + yy * si, -xx * si + yy * co
        L2 = 1.0 - Y / 100.0
        U = X / L2 / pw
        w = U - torch.floor(U)
        col = torch.floor(W // 2 + U + xs[k] / (0.05 * 800 / W) - 0.5).long()
        zeta = H // 2 + zz / L2 / pw
        line = torch.floor(zeta).long()
        wz = zeta - torch.floor(zeta)
        ok = inside & (col >= 0) & (col <= W - 1) & (line >= 0) & (line <= H - 1)
        w = torch.where(col == W - 1, torch.zeros_like(w), w)
        wz = torch.where(line == H - 1, torch.zeros_like(wz), wz)
        c0, c1 = col.clamp(0, W - 1), (col + 1).clamp(0, W - 1)
        l0, l1 = line.clamp(0, H - 1), (line + 1).clamp(0, H - 1)
        P = filt[k]
        top = P[l0, c0.expand_as(l0)] * (1 - w) + P[l0, c1.expand_as(l0)] * w
        low = P[l1, c0.expand_as(l0)] * (1 - w) + P[l1, c1.expand_as(l0)] * w
        rec += torch.where(ok, (top * (1 - wz) + low * wz) / L2 / L2 * (dbeta * 1000), torch.zeros_like(rec))
    return filt, rec


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind in ("fdk", "fdk_once"):
        a, xs, ys = _fdk_angles(c)
        proj = _transmissions(c["nA"], c["H"], c["W"], a, xs[0] / (0.05 * 800 / c["W"]), seed)
        filt, rec = _fdk(proj, c, a, xs, ys, c.get("alpha", 0.5), c.get("half_fan", False))
        return rec if kind == "fdk_once" else dict(filtered=filt, recon=rec)
    steps = c["nA"] * c["H"] * c["W"] * (c["N"] + 20.0)
    if kind == "forward":
        return None if steps > LIMIT else _intensity(c, seed, c["Nz"], _tables(100, c["table"]))
    if kind == "gradient":
        if steps > LIMIT:
            return None
        p, grad, loss = _gradient(c, seed, _tables(100, c["table"]))
        return dict(p=p, grad=grad) if c["form"] == "autograd" else dict(grad=grad, loss=loss)
    if kind == "batch":
        slices = [int(v) for v in c["slices"].split(",")]
        if steps * len(slices) > LIMIT:
            return None
        table = _tables(100, "two_term")
        proj = [_intensity(c, seed + 31 * i, Nz, table) for i, Nz in enumerate(slices)]
        return dict(proj=proj, recon=[None] * len(proj))
    return None
