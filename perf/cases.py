"""What users of this library have it do, as cases that can be timed.

Each case is one pass through public entry points (phasecon_amd.mbir,
.pcmbir, .warmstart, or the C-ABIs they bind) on seeded synthetic data:

  equits       equits of the MBIR ICD from a saved object (the solver's loop)
  setup        what every multi-resolution stage begins with: the system
               matrix, the error sinogram and the FP64 cost
  fbp          filtered back-projection of a scan (the learned start's input)
  reconstruct  the drop-in reconstruct(), all stages, host arrays in and out
  tomo         the PCMBIR tomographic ICD between two cost evaluations
  sd           steepest-descent phase retrieval of every view
  estimate     the per-view ADMM (simplex search and steepest descent)
  paganin      single-material Paganin retrieval of every view
  unet_forward inference of the warm-start network
  unet_train   one Adam step of it; unet_grad its loss and gradients

listed() holds named cases over the range of use, draw() more of the same
ranges.  exact() restates each path in 64 bits with torch alone.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64
I0 = 5e3          # photons per detector sample
SIG = dict(sig_s=0.01, sig_t=0.001, c_s=0.01, c_t=0.01, p_s=1.2, p_t=1.1)
KEV = 17.0        # photon energy of the phase-contrast cases
DIST = 1e5        # propagation distance, um
DOB = 1000.0      # delta over beta
KW = 2.0 * math.pi * 1e-6 / (1.23984e-9 / KEV)  # wavenumber per 1 um voxel
LAM = 4.135668e-19 * 299792458e6 / KEV           # wavelength, um
NU = 0.5


def listed():
    return [
        # the smallest scan of the repository: launches and host latency
        dict(name="equits-32x32x4", kind="equits", cols=32, rows=4, frames=1, vpf=24, mxy=1, mz=1,
             tile=8, pair=False, afp16=False, equits=10),
        # the plain 4D workload at full resolution, the solver's main loop
        dict(name="equits-256x256x8x16", kind="equits", cols=256, rows=8, frames=16, vpf=16,
             mxy=1, mz=1, tile=8, pair=True, afp16=False, equits=8),
        # a coarse stage of an odd-sized scan, rows not a power of two,
        # FP16 system matrix
        dict(name="equits-75x75x12x5-coarse", kind="equits", cols=150, rows=24, frames=5, vpf=29,
             mxy=2, mz=2, tile=8, pair=False, afp16=True, equits=8),
        # the set-up of the plain 4D workload's last stage
        dict(name="setup-256x256x8x16", kind="setup", cols=256, rows=8, frames=16, vpf=16, mxy=1,
             mz=1),
        # the network input of the learned start on the same scan
        dict(name="fbp-256x256x8x16", kind="fbp", cols=256, rows=8, frames=16, vpf=16, mxy=1, mz=1),
        # a whole drop-in call on a small 4D scan (three stages)
        dict(name="reconstruct-64x64x8x4", kind="reconstruct", cols=64, rows=8, frames=4, vpf=16,
             equits=12),
        # the PCMBIR object size: the tomographic part of a head iteration
        dict(name="tomo-256x256x256x360", kind="tomo", cols=256, rows=256, views=360, tile=8,
             equits=2),
        # the padded 512^2 detector of the PCMBIR workload, windowed as the
        # drop-in does
        dict(name="sd-24x512x512", kind="sd", views=24, rows=512, cols=512, iters=40, window=True),
        # the ADMM of a few views: the simplex search dominates
        dict(name="estimate-16x256x256", kind="estimate", views=16, rows=256, cols=256, pret=3,
             iters=10, tomo=False),
        # the initial estimate of a short scan: a small call
        dict(name="paganin-4x256x128", kind="paganin", views=4, rows=256, cols=128),
        # inference on every frame of the plain 4D workload
        dict(name="unet-16x8x256x256", kind="unet_forward", n=16, d=8, h=256, w=256, channels=16,
             cin=2),
        # a training step at the size the warm start is trained with
        dict(name="unet-train-8x8x64x64", kind="unet_train", n=8, d=8, h=64, w=64, channels=16,
             cin=2),
    ]


def draw(rng):
    def log(lo, hi, step=1):
        return max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step)

    kind = rng.choice(["equits"] * 3 + ["sd"] * 2 + ["unet_forward"] * 2 +
                      ["setup", "fbp", "reconstruct", "tomo", "estimate", "paganin", "unet_train",
                       "unet_grad"])
    if kind in ("equits", "setup", "fbp"):
        mxy = rng.choice([1, 1, 1, 2, 4])
        mz = rng.choice([1, 1, 2])
        c = dict(kind=kind, cols=log(32, 256, 2 * mxy), rows=log(4, 32, 2 * mz), frames=log(1, 16),
                 vpf=log(8, 40), mxy=mxy, mz=mz)
        while c["cols"] ** 2 * c["rows"] * c["frames"] * c["vpf"] > 256 ** 2 * 8 * 16 * 16:
            c["frames"] = max(1, c["frames"] // 2)
            c["vpf"] = max(8, c["vpf"] - 3)
            c["rows"] = max(2 * mz, c["rows"] - 2 * mz)
        if kind == "equits":
            c.update(tile=rng.choice([8, 10, 12]), pair=rng.random() < 0.5,
                     afp16=rng.random() < 0.25, equits=rng.randint(3, 8))
        return c
    if kind == "reconstruct":
        return dict(kind=kind, cols=log(32, 80, 8), rows=rng.choice([4, 8, 12]),
                    frames=rng.randint(1, 4), vpf=rng.randint(12, 24), equits=rng.randint(6, 12))
    if kind == "tomo":
        return dict(kind=kind, cols=log(48, 160, 2), rows=log(16, 200, 2), views=log(40, 200),
                    tile=8, equits=rng.randint(1, 2))
    if kind == "sd":
        r, k = rng.choice([32, 64, 128, 256, 512, 1024]), rng.choice([32, 64, 128, 256, 512, 1024])
        return dict(kind=kind, views=max(1, min(log(1, 60), 24 * 512 * 512 // (r * k))), rows=r,
                    cols=k, iters=rng.randint(5, 50), window=rng.random() < 0.5)
    if kind == "estimate":
        r, k = rng.choice([32, 64, 128, 256]), rng.choice([32, 64, 128, 256])
        return dict(kind=kind, views=log(1, 16), rows=r, cols=k, pret=rng.randint(1, 3),
                    iters=rng.randint(3, 10), tomo=rng.random() < 0.4)
    if kind == "paganin":
        return dict(kind=kind, views=log(1, 40), rows=rng.choice([64, 128, 256, 512]),
                    cols=rng.choice([32, 64, 128, 256, 512]))
    n, d, h, w = log(1, 16), rng.choice([4, 8, 12, 16]), log(16, 256, 4), rng.choice([64, 128, 256])
    most = 16 * 8 * 256 * 256 if kind == "unet_forward" else 16 * 8 * 64 * 64
    while n * d * h * w > most:
        n, h = max(1, n // 2), max(16, h // 8 * 4)
        w = w if n > 1 or h > 16 else 64
    return dict(kind=kind, n=n, d=d, h=h, w=w, channels=rng.choice([8, 16, 16, 24, 32]),
                cin=rng.choice([1, 2, 2, 3]))


# ------------------------------------------------------------- inputs
def _rng(case, seed):
    key = sum((i + 1) * ord(ch) for i, ch in enumerate(case["kind"]))
    return np.random.default_rng([seed, key])


class _Phantom:
    """A disc of value lo with seeded ellipsoids of added value hi - lo that
    drift from frame to frame, in units of the half-width (x, y) and of the
    height (z); its line integrals are closed-form."""

    def __init__(self, rng, frames, lo=0.005, hi=0.02, count=20):
        self.lo, self.add, self.count = lo, hi - lo, count
        self.c = rng.uniform(-0.5, 0.5, (count, 2))
        self.v = rng.normal(0.0, 0.01, (count, 2))
        self.r = rng.uniform(0.05, 0.2, (count, 2))
        self.phi = rng.uniform(0, math.pi, count)
        self.zc = rng.uniform(0, 1, count)
        self.rz = rng.uniform(0.15, 0.6, count)
        self.frames = frames

    def parts(self, frame):
        yield self.lo, 0.0, 0.0, 0.85, 0.85, 0.0, 0.0, math.inf
        for e in range(self.count):
            cx, cy = self.c[e] + self.v[e] * frame
            yield (self.add, cx, cy, self.r[e, 0], self.r[e, 1], self.phi[e], self.zc[e],
                   self.rz[e])

    def lines(self, theta, frame, cols, rows, half):
        """[len(theta)][rows][cols]: line integrals in voxels of half-width
        `half` at the detector samples, view angle theta."""
        t = torch.as_tensor(theta, dtype=F64, device=DEV)[:, None, None]
        u = ((torch.arange(cols, dtype=F64, device=DEV) + 0.5) / cols * 2 - 1)[None, None, :]
        z = ((torch.arange(rows, dtype=F64, device=DEV) + 0.5) / rows)[None, :, None]
        out = torch.zeros((len(theta), rows, cols), dtype=F64, device=DEV)
        for val, cx, cy, a, b, phi, zc, rz in self.parts(frame):
            q = (1 - ((z - zc) / rz) ** 2).clamp(min=0)  # squared scale of the section
            n1 = torch.cos(t) * math.cos(phi) - torch.sin(t) * math.sin(phi)
            n2 = -torch.cos(t) * math.sin(phi) - torch.sin(t) * math.cos(phi)
            A2 = (a * n1) ** 2 + (b * n2) ** 2
            s2 = (u - (cx * torch.cos(t) - cy * torch.sin(t))) ** 2
            out += (2 * val * a * b * half) * torch.sqrt((q * A2 - s2).clamp(min=0)) / A2
        return out

    def voxels(self, frame, n, nz):
        """[nz][n][n] values at the voxel centres."""
        u = (torch.arange(n, dtype=F64, device=DEV) + 0.5) / n * 2 - 1
        y, x = u[None, :, None], u[None, None, :]
        z = ((torch.arange(nz, dtype=F64, device=DEV) + 0.5) / nz)[:, None, None]
        out = torch.zeros((nz, n, n), dtype=F64, device=DEV)
        for val, cx, cy, a, b, phi, zc, rz in self.parts(frame):
            e1 = (x - cx) * math.cos(phi) + (y - cy) * math.sin(phi)
            e2 = -(x - cx) * math.sin(phi) + (y - cy) * math.cos(phi)
            out += val * (((e1 / a) ** 2 + (e2 / b) ** 2 + ((z - zc) / rz) ** 2) <= 1)
        return out


def _angles(case):
    """Interlaced views: vpf per frame over 180 degrees, each frame's set
    rotated by a quarter of the spacing against the one before."""
    f, v = case["frames"], case["vpf"]
    a = (np.arange(v)[None, :] + (np.arange(f)[:, None] % 4) / 4.0) * (math.pi / v)
    return a.reshape(-1).astype(np.float32)


def _scan(case, seed):
    rng = _rng(case, seed)
    rows, cols, frames, vpf = case["rows"], case["cols"], case["frames"], case["vpf"]
    ph = _Phantom(rng, frames)
    ang = _angles(case)
    line = torch.cat([ph.lines(ang[f * vpf:(f + 1) * vpf].astype(np.float64), f, cols, rows,
                               cols / 2) for f in range(frames)])
    g = torch.Generator(device=DEV).manual_seed(seed)
    counts = torch.poisson(I0 * torch.exp(-line).float(), generator=g).clamp(min=1)
    scan = dict(
        name="perf", projections=torch.log(I0 / counts).float().cpu().numpy(),
        weights=counts.cpu().numpy(), angles=ang,
        proj_times=np.arange(frames * vpf, dtype=np.float32),
        recon_times=(np.arange(frames + 1) * vpf).astype(np.float32), proj_rows=rows,
        proj_cols=cols, proj_num=frames * vpf, recon_num=frames, vox_wid=1.0,
        rot_center=cols / 2.0, seed=seed, **SIG)
    x = None
    if case["kind"] in ("equits", "setup"):
        n, nz = cols // case["mxy"], rows // case["mz"]
        x = torch.stack([ph.voxels(f, n, nz) for f in range(frames)])
        x = x * (1 + 0.05 * torch.randn(x.shape, generator=g, device=DEV, dtype=F64))
        x = x.float().cpu().numpy()
    return scan, x


def _fields(case, seed):
    """(zr, zi, D, y): the log-transmittance z of every view (weak absorption,
    phase of about half a radian), the illumination factor and the measured
    amplitudes |H D exp(-z)|."""
    rng = _rng(case, seed)
    n, r, k = case["views"], case["rows"], case["cols"]
    ph = _Phantom(rng, 1, lo=0.1, hi=0.5)
    theta = np.arange(n) * (math.pi / n) + rng.uniform(0, 0.1)
    zi = 0.1 + ph.lines(theta, 0, r, k, 0.6).transpose(1, 2)
    g = torch.Generator(device=DEV).manual_seed(seed)
    zr = 0.02 + 0.1 * zi + 0.002 * torch.rand(zi.shape, generator=g, device=DEV, dtype=F64)
    beam = torch.exp(-sum((torch.linspace(-1, 1, q, dtype=F64, device=DEV) ** 2).reshape(s)
                          for q, s in ((r, (r, 1)), (k, (1, k)))))
    D = 0.6 + 0.4 * beam + 0.02 * torch.rand(zi.shape, generator=g, device=DEV, dtype=F64)
    D = torch.complex(D, torch.zeros_like(D))
    y = _fresnel(D * torch.exp(-torch.complex(zr, zi)), _window(case), False).abs()
    y = (y * (1 + 0.01 * torch.randn(y.shape, generator=g, device=DEV, dtype=F64))).clamp(min=1e-3)
    return zr, zi, D, torch.complex(y, torch.zeros_like(y))


def _c64(t):
    return t.to(torch.complex64).cpu().numpy()


def _window(case):
    if not case.get("window", case["kind"] == "estimate"):
        return None
    u, v = _freqs(case["rows"], case["cols"])
    s = 2.0 / math.sqrt(LAM * DIST)
    return torch.exp(-(u * u + v * v) / (2 * s * s)).float()


def _ptr(a):
    return a.ctypes.data_as(C.c_void_p)


def _unet_params(case, rng):
    c, out = case["channels"], []
    for i, (ci, co) in enumerate(_unet_layers(c, case["cin"])):
        s = math.sqrt(2.0 / (27 * ci)) * (0.3 if i == 10 else 1.0)
        out += [rng.standard_normal(co * 27 * ci) * s, rng.standard_normal(co) * 0.02]
    return np.concatenate(out).astype(np.float32)


def _unet_data(case, seed):
    """Scaled attenuation volumes: a piecewise constant image with noise as
    the network's input channels, the image itself as the target."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    n, d, h, w, cin = (case[k] for k in ("n", "d", "h", "w", "cin"))
    t = torch.nn.functional.interpolate(
        torch.rand((n, 1, 2, 4, 4), generator=g, device=DEV), size=(d, h, w), mode="trilinear",
        align_corners=True)[:, 0]
    t = 0.25 + 0.75 * (t > 0.5).float()
    x = t[..., None] + 0.3 * torch.randn((n, d, h, w, cin), generator=g, device=DEV)
    return x.cpu().numpy(), t.cpu().numpy()


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind in ("equits", "setup", "fbp"):
        from phasecon_amd.mbir import Stage
        scan, x = _scan(case, seed)
        st = s["st"] = Stage(scan, mult_xy=case["mxy"], mult_z=case["mz"], tile=case.get("tile", 8),
                             afp16=case.get("afp16", False))
        st.build_amatrix()
        if x is not None:
            st.set_object(x)
        if kind == "equits":
            st.option("pair_parities", int(case["pair"]))
            st.snapshot()
    elif kind == "reconstruct":
        from phasecon_amd.mbir import default_options
        s["scan"], _ = _scan(case, seed)
        o = s["options"] = default_options()
        o.write_files, o.max_equits, o.p_t = 0, case["equits"], SIG["p_t"]
    elif kind == "tomo":
        from phasecon_amd.mbir import TomoStage, tomo_prior
        from phasecon_amd.synth import geometry_scan
        td, tb = _tomo_targets(case, seed)
        prior = tomo_prior((2e-7, 1e-3, 0.01, 0.01), (2e-10, 1e-3, 0.01, 0.01), 1,
                           float(case["views"]), KW, delta_over_beta=DOB, mu=0.5, alpha=1.5)
        st = s["st"] = TomoStage(geometry_scan(case["rows"], case["cols"], case["views"]), prior,
                                 tile=case["tile"])
        zero = np.zeros(st.shape_x, np.float32)
        st.set_objects(zero, zero)
        st.init_errors(td, tb)
    elif kind in ("sd", "estimate", "paganin"):
        from phasecon_amd.pcmbir import PhaseRetrieval
        win = _window(case)
        n, r, k = case["views"], case["rows"], case["cols"]
        pr = s["pr"] = PhaseRetrieval(n, r, k, 1.0, 1.0, LAM, DIST,
                                      None if win is None else win.cpu().numpy())
        zr, zi, D, y = _fields(case, seed)
        if kind == "paganin":
            s["y"], s["D"] = (np.ascontiguousarray(_c64(a)) for a in (y, D))
            s["zr"], s["zi"] = np.empty((n, r, k)), np.empty((n, r, k))
        else:
            zr, zi = 0.9 * zr, 0.9 * zi
            w = _c64(torch.exp(-torch.complex(zr, zi)))
            pr.set_problem(_c64(y), _c64(D), np.float32(1), w, w, None, NU)
        if kind == "sd":
            s["w"], s["om"] = (np.empty((n, r, k, 2), np.float32) for _ in range(2))
        if kind == "estimate":
            pr.set_nms_prior(2e-2, 1e-2, 2e-2, 1e-2, 50.0, True, 1.2, NU)
            if case["tomo"]:
                pr.set_tomo_target(0.5, (1.05 * torch.complex(zr, zi)).cpu().numpy())
            s["zr"], s["zi"] = zr.cpu().numpy(), zi.cpu().numpy()
    else:
        from phasecon_amd.warmstart import UNet
        net = s["net"] = UNet(channels=case["channels"], in_channels=case["cin"])
        net.set_params(_unet_params(case, _rng(case, seed)))
        s["x"], s["t"] = _unet_data(case, seed)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "equits":
        st = s["st"]
        st.snapshot(restore=True)
        st.init_error()
        for it in range(1, case["equits"] + 1):
            st.icd_graph(1, it)
        cost = st.cost(estimate=True)
        return dict(x=st.get_object(), cost=cost)
    if kind == "setup":
        st = s["st"]
        st.build_amatrix()
        st.init_error()
        return dict(cost=st.cost(fresh=True), e=st.get_error())
    if kind == "fbp":
        return s["st"].fbp()
    if kind == "reconstruct":
        from phasecon_amd.mbir import reconstruct
        x, _, cost = reconstruct(s["scan"], convg_thresh=1e-3, options=s["options"])
        return dict(x=x, cost=cost)
    if kind == "tomo":
        st = s["st"]
        c0 = st.tomo_cost()
        for i in range(case["equits"]):
            st.equits(1, i + 1, 761521 + i)
        c1 = st.tomo_cost()
        xd, xb = st.get_objects()
        return dict(c0=c0, c1=c1, xd=xd, xb=xb)
    if kind == "sd":
        pr = s["pr"]
        it, _ = pr.sd_run(case["iters"], 0.0)
        if pr.L.pcmbir_hip_get_phase_state(pr.h, _ptr(s["w"]), _ptr(s["om"])):
            raise RuntimeError("pcmbir_hip_get_phase_state failed")
        return dict(iters=it, w=s["w"], om=s["om"])
    if kind == "estimate":
        return s["pr"].estimate(s["zr"], s["zi"], case["pret"], 0.0, case["iters"], 0.0)
    if kind == "paganin":
        pr = s["pr"]
        if pr.L.pcmbir_hip_paganin(pr.h, _ptr(s["y"]), _ptr(s["D"]), DOB, 2 * math.pi / LAM,
                                   _ptr(s["zr"]), _ptr(s["zi"])):
            raise RuntimeError("pcmbir_hip_paganin failed")
        return dict(zr=s["zr"], zi=s["zi"])
    net = s["net"]
    if kind == "unet_forward":
        return net.forward(s["x"])
    if kind == "unet_grad":
        loss, g = net.gradients(s["x"], s["t"])
        return dict(loss=loss, g=g)
    loss = net.train_step(s["x"], s["t"], 1e-3)
    return dict(loss=loss, params=net.params())


# --------------------------------------------- what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind in ("equits", "setup", "fbp"):
        nx, nz = case["cols"] // case["mxy"], case["rows"] // case["mz"]
        f, v, W = case["frames"], case["vpf"], 2 * case["mxy"] + 1
        vox, sino = nx * nx * nz * f, case["cols"] * case["rows"] * f * v
        hits = nx * nx * f * v * W * case["rows"]      # (column, view, bin, row) entries
        a = nx * nx * f * v * (4 * W + 4)
        if kind == "equits":  # A, x, e, w of each equit, the object out
            n = case["equits"]
            aw = nx * nx * f * v * ((2 if case["afp16"] else 4) * W + 4)
            return dict(bytes=n * (aw + 8.0 * vox + 12.0 * sino) + 4.0 * vox,
                        flops=n * (6.0 * hits + 28 * 14.0 * vox))
        if kind == "setup":  # A out; x, y, w in, e out
            return dict(bytes=a + 8.0 * vox + 16.0 * sino, flops=4.0 * hits + 14 * 10.0 * vox)
        return dict(bytes=a + 4.0 * vox + 4.0 * sino,
                    flops=4.0 * hits + 5.0 * sino * math.log2(case["cols"]))
    if kind == "reconstruct":
        vox = case["cols"] ** 2 * case["rows"] * case["frames"]
        sino = case["cols"] * case["rows"] * case["frames"] * case["vpf"]
        hits = 3.0 * case["cols"] * sino
        return dict(bytes=case["equits"] * (16.0 * case["cols"] * sino / case["rows"] + 8.0 * vox +
                                            12.0 * sino) + 4.0 * vox + 8.0 * sino,
                    flops=case["equits"] * (6.0 * hits + 28 * 14.0 * vox))
    if kind == "tomo":
        nx, nz, v, n = case["cols"], case["rows"], case["views"], case["equits"]
        vox, sino = nx * nx * nz, nx * nz * v
        return dict(bytes=n * (16.0 * nx * nx * v + 16.0 * vox + 16.0 * sino) + 16.0 * vox +
                    16.0 * sino,
                    flops=n * (8.0 * 3 * nx * nx * v * nz + 28 * 40.0 * vox))
    if kind in ("sd", "estimate", "paganin"):
        px = float(case["views"] * case["rows"] * case["cols"])
        fft = 10.0 * px * math.log2(case["rows"] * case["cols"])  # one H: two FFTs
        if kind == "paganin":
            return dict(bytes=px * (16 + 16), flops=fft)
        if kind == "sd":  # y, D, v, lambda in; w, Omega in and out each iteration
            return dict(bytes=case["iters"] * px * (28 + 32.0), flops=case["iters"] * 4 * fft)
        return dict(bytes=case["pret"] * px * (48.0 + case["iters"] * 60.0),
                    flops=case["pret"] * (px * (30 * 2 * 18 * 12.0) + case["iters"] * 4 * fft))
    px = float(case["n"] * case["d"] * case["h"] * case["w"])
    flops = sum(2.0 * 27 * ci * co * px / (1, 1, 8, 8, 64, 64, 8, 8, 1, 1, 1)[i]
                for i, (ci, co) in enumerate(_unet_layers(case["channels"], case["cin"])))
    if kind == "unet_forward":
        return dict(bytes=px * 4 * (case["cin"] + 1), flops=flops)
    acts = 2.0 * px * (case["channels"] * (4 + 6 / 8.0 * 2 + 4 / 64.0 * 4))  # stored, read back
    return dict(bytes=px * 4 * (case["cin"] + 1) + 2 * acts, flops=3 * flops)


def tolerance(case):
    """About four times what two correct runs were seen to differ by."""
    kind = case["kind"]
    if kind in ("equits", "reconstruct"):
        # several tiles update one error sinogram at once, so a column may
        # read it before or after a neighbour's update: runs of the same code
        # differ by that (up to 0.009 seen), and so do sweeps of another speed
        return dict(rel=0.02, max=0.9)
    if kind == "tomo":
        return dict(rel=0.01, max=0.99)  # the same (0.0022, single voxels 0.5)
    if kind == "setup":
        return dict(rel=2e-7)   # FP64 sums, e rounded to 32 bits once (2.5e-8)
    if kind == "fbp":
        return dict(rel=6e-7)   # 32-bit sums over the views (1.5e-7)
    if kind == "sd":
        return dict(rel=1e-6)   # 32-bit transforms (1.8e-7 between two FFTs)
    if kind == "estimate":
        # a last-bit difference turns some comparisons of the search (6e-5
        # between two FFTs, single pixels 0.0013)
        return dict(rel=2.5e-4, max=0.01)
    if kind == "paganin":
        return dict(rel=4e-6)   # the logarithm of a 32-bit transform (9.4e-7)
    return dict(rel=0.01, max=0.5)  # bf16 activations (0.001 to 0.004)


# ------------------------------------------------- the same in 64 bits
def _freqs(rows, cols):
    i, j = torch.arange(rows, dtype=F64, device=DEV), torch.arange(cols, dtype=F64, device=DEV)
    u = torch.where(i >= rows // 2, i - rows, i) / rows
    v = torch.where(j >= cols // 2, j - cols, j) / cols
    return u[:, None], v[None, :]


def _fresnel(x, win, herm):
    u, v = _freqs(*x.shape[-2:])
    phi = -(u * u + v * v) * (math.pi * LAM * DIST)
    if herm:
        f = torch.complex(torch.cos(phi), -torch.sin(phi))
    else:
        f = torch.complex(torch.cos(phi), torch.sin(phi)) * (1 if win is None else win.double())
    return torch.fft.ifft2(torch.fft.fft2(x) * f)


class _System:
    """Geometry and system matrix of a stage (pitch 1, centred rotation
    axis): windows of W detector channels per (column, view), the response of
    a square voxel under a Hamming beam tabulated at 64 offsets."""

    def __init__(self, cols, mxy, angles):
        self.Nr, self.W, self.d = cols, 2 * mxy + 1, float(mxy)
        self.n = cols // mxy
        self.R0 = -cols / 2.0
        self.off = (self.d / math.sqrt(2.0) + 0.5) / 64
        self.ang = torch.as_tensor(np.asarray(angles, np.float64), dtype=F64, device=DEV)
        self.H = self._response()
        i = torch.arange(self.n, dtype=F64, device=DEV)
        self.x = (self.R0 + (i + 0.5) * self.d)[None, :].expand(self.n, -1).reshape(-1)
        self.y = (-cols / 2.0 + (i + 0.5) * self.d)[:, None].expand(-1, self.n).reshape(-1)
        self.mask = self.x ** 2 + self.y ** 2 < (cols / 2.0) ** 2

    def _response(self):
        k = torch.arange(512, dtype=F64, device=DEV)
        beam = 0.54 - 0.46 * torch.cos(2 * math.pi / 512 * k)
        beam = beam / beam.sum()
        a = torch.remainder(self.ang, math.pi / 2)[:, None]
        top = torch.where(a <= math.pi / 4, self.d / torch.cos(a), self.d / torch.cos(math.pi / 2 - a))
        h = math.cos(math.pi / 4)
        outer, inner = h * torch.cos(math.pi / 4 - a), h * torch.cos(math.pi / 4 + a).abs()
        t = (2.0 * torch.arange(1536, dtype=F64, device=DEV) / 1536)[None, :]
        rise = (outer - inner).clamp(min=1e-300)
        trap = torch.minimum((t - (1 - outer)) / rise, (1 + outer - t) / rise).clamp(0, 1) * top
        trap = trap.float().double()
        lo = torch.arange(64, dtype=F64, device=DEV)[:, None] * self.off - self.d
        b = torch.floor((-0.5 + k / 512 - lo) * (1536 / (2 * self.d))).long()
        ok = (b >= 0) & (b < 1536)
        H = torch.stack([(trap[:, b[i].clamp(0, 1535)] * (beam * ok[i])).sum(-1)
                         for i in range(64)], 1)
        return torch.cat([H.float().double(), torch.zeros((len(self.ang), 1), dtype=F64,
                                                          device=DEV)], 1)

    def window(self, p):
        """(channels, values) [columns][W] of view p, 0 where there is none."""
        r = self.x * torch.cos(self.ang[p]) - self.y * torch.sin(self.ang[p])
        lo, hi = torch.floor(r - self.d - self.R0), torch.floor(r + self.d - self.R0)
        j = lo.clamp(min=0)[:, None] + torch.arange(self.W, dtype=F64, device=DEV)[None, :]
        dist = (r[:, None] - (self.R0 + j + 0.5)).abs()
        k = torch.floor(dist / self.off)
        ok = (j <= hi.clamp(max=self.Nr - 1)[:, None]) & (k < 64)
        ok &= ((r + self.d >= self.R0) & (r - self.d <= self.Nr + self.R0))[:, None]
        wh = dist - k * self.off
        kk = k.clamp(0, 63).long()
        f = ((self.off - wh) * self.H[p][kk] + wh * self.H[p][kk + 1]) / self.off
        return j.clamp(0, self.Nr - 1).long(), torch.where(ok & (f > 0), f, torch.zeros_like(f))

    def forward(self, p, x):
        """[Nr][nz] of x [columns][nz]."""
        out = torch.zeros((self.Nr, x.shape[1]), dtype=F64, device=DEV)
        j, a = self.window(p)
        for k in range(self.W):
            out.index_add_(0, j[:, k], a[:, k:k + 1] * x)
        return out

    def back(self, p, q):
        """[columns][nz] of q [Nr][nz]."""
        j, a = self.window(p)
        return sum(a[:, k:k + 1] * q[j[:, k]] for k in range(self.W))


def _prior_cost(x, per_frame, mxy):
    """qGGMRF cost of x [t][z][y][x], each neighbour pair once."""
    dist = {(a, b, c): math.sqrt(a * a + b * b + c * c) for a in (-1, 0, 1) for b in (-1, 0, 1)
            for c in (-1, 0, 1) if (a, b, c) != (0, 0, 0)}
    norm = 2.0 + sum(1 / v for v in dist.values())
    scale = mxy ** 3 * per_frame

    def rho(d, sig, p, c):
        a = d.abs()
        return (a * a / sig ** 2) / (c + a ** (2 - p) / sig ** (2 - p))

    total = 0.0
    for (a, b, c), v in dist.items():
        if (a, b, c) < (0, 0, 0):
            continue
        cut = [(slice(max(0, -o), n - max(0, o)), slice(max(0, o), n - max(0, -o)))
               for o, n in zip((a, b, c), x.shape[1:])]
        d = x[:, cut[0][0], cut[1][0], cut[2][0]] - x[:, cut[0][1], cut[1][1], cut[2][1]]
        total += scale / v / norm * float(rho(d, SIG["sig_s"] * mxy, SIG["p_s"], SIG["c_s"]).sum())
    if x.shape[0] > 1:
        total += scale / norm * float(rho(x[1:] - x[:-1], SIG["sig_t"] * per_frame, SIG["p_t"],
                                          SIG["c_t"]).sum())
    return total


def _exact_setup(case, seed):
    scan, x0 = _scan(case, seed)
    S = _System(case["cols"], case["mxy"], scan["angles"])
    x = torch.as_tensor(x0, device=DEV).double()
    y, w = (torch.as_tensor(scan[k], device=DEV).double() for k in ("projections", "weights"))
    e = torch.zeros((y.shape[0], y.shape[2], y.shape[1]), dtype=F64, device=DEV)
    for p in range(y.shape[0]):
        xc = x[p // case["vpf"]].reshape(x.shape[1], -1).t()
        e[p] = y[p].t() - S.forward(p, xc).repeat_interleave(case["mz"], 1)
    data = float((e * e * w.transpose(1, 2)).sum()) / 2
    prior = _prior_cost(x, case["vpf"], case["mxy"])
    return dict(cost=np.array([data + prior, data, prior]), e=e)


def _exact_fbp(case, seed):
    scan, _ = _scan(case, seed)
    S = _System(case["cols"], case["mxy"], scan["angles"])
    y = torch.as_tensor(scan["projections"], device=DEV).double()
    nz, zo, f, v = case["rows"] // case["mz"], case["mz"], case["frames"], case["vpf"]
    k = torch.arange(S.Nr, dtype=F64, device=DEV)
    k = k[:, None] - k[None, :]
    ramp = torch.where(torch.remainder(k, 2) == 1, -1 / (math.pi * k.clamp(min=-1e9)) ** 2,
                       torch.where(k == 0, 0.25, 0.0))
    out = torch.zeros((f, S.n * S.n, nz), dtype=F64, device=DEV)
    one = torch.zeros((f, S.n * S.n, 1), dtype=F64, device=DEV)
    for p in range(f * v):
        q = ramp @ y[p].t()
        out[p // v] += S.back(p, q.reshape(S.Nr, nz, zo).sum(2))
        one[p // v] += S.back(p, ramp @ S.forward(p, S.mask.double()[:, None])) * zo
    K = one[:, S.mask].mean()
    return (out / K).transpose(1, 2).reshape(f, nz, S.n, S.n)


def _tomo_targets(case, seed):
    ph = _Phantom(_rng(case, seed), 1, lo=2e-7, hi=1e-6)
    theta = np.arange(case["views"], dtype=np.float32) * np.float32(math.pi / case["views"])
    td = KW * ph.lines(theta.astype(np.float64), 0, case["cols"], case["rows"], case["cols"] / 2)
    td = td.transpose(1, 2).float().contiguous()
    return td.cpu().numpy(), (td / DOB).cpu().numpy()


def _exact_sd(case, seed):
    zr, zi, D, y = _fields(case, seed)
    win = _window(case)
    r32 = lambda a: a.to(torch.complex64).to(torch.complex128)  # noqa: E731
    w = r32(torch.exp(-0.9 * torch.complex(zr, zi)))
    D, y, v = r32(D), r32(y), w
    tiny = np.finfo(np.float64).tiny

    def omega(w):
        h = _fresnel(D * w, win, False)
        q = y * h.conj() / (h.abs() ** 2 + tiny)
        return q / (q.abs() + tiny)

    def dot(a, b):
        return (a * b.conj()).real.sum((1, 2), keepdim=True)

    om = omega(w)
    for _ in range(case["iters"]):
        b = _fresnel(om.conj() * (_fresnel(D * w, win, False) * om - y), win, True) * D.conj()
        g = b + NU * (w - v)
        b = _fresnel(om.conj() * (_fresnel(D * g, win, False) * om), win, True) * D.conj()
        alpha = dot(g, g) / (dot(g, b) + NU * dot(g, g))
        w = w - alpha * g
        om = omega(w)
    return dict(iters=None, w=torch.view_as_real(w), om=torch.view_as_real(om))


def _exact_paganin(case, seed):
    _, _, D, y = _fields(case, seed)
    D, y = (a.to(torch.complex64).to(torch.complex128) for a in (D, y))
    u, v = _freqs(case["rows"], case["cols"])
    tran = DIST * DOB / (4 * math.pi / LAM) * (u * u + v * v) * 4 * math.pi ** 2 + 1
    f = torch.fft.ifft2(torch.fft.fft2(y.real ** 2 / (D.abs() ** 2)) / tran).real
    t = -torch.log(f.abs())
    return dict(zr=t / 2, zi=t * DOB / 2)


def _unet_layers(c, cin):
    return [(cin, c), (c, c), (c, 2 * c), (2 * c, 2 * c), (2 * c, 4 * c), (4 * c, 4 * c),
            (6 * c, 2 * c), (2 * c, 2 * c), (3 * c, c), (c, c), (c, 1)]


def _unet_net(case, flat, x):
    """The network on one batch [N][D][H][W][cin], FP64."""
    P, i = [], 0
    for ci, co in _unet_layers(case["channels"], case["cin"]):
        P.append((flat[i:i + co * 27 * ci].reshape(co, 27, ci), flat[i + co * 27 * ci:][:co]))
        i += co * 27 * ci + co

    def conv(a, l, relu=True):
        w, b = P[l]
        d, h, wd = a.shape[1:4]
        ap = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1, 1, 1))
        o = b
        for t in range(27):
            z, y, q = t // 9, t // 3 % 3, t % 3
            o = o + ap[:, z:z + d, y:y + h, q:q + wd] @ w[:, t].t()
        return torch.relu(o) if relu else o

    def pool(a):
        n, d, h, w, c = a.shape
        return a.reshape(n, d // 2, 2, h // 2, 2, w // 2, 2, c).mean((2, 4, 6))

    def up(a):
        for k in (1, 2, 3):
            a = a.repeat_interleave(2, k)
        return a

    s1 = conv(conv(x, 0), 1)
    s2 = conv(conv(pool(s1), 2), 3)
    b = conv(conv(pool(s2), 4), 5)
    b = conv(conv(torch.cat([up(b), s2], -1), 6), 7)
    b = conv(conv(torch.cat([up(b), s1], -1), 8), 9)
    return x[..., 0] + conv(b, 10, False)[..., 0]


def _exact_unet(case, seed):
    x, t = (torch.as_tensor(a, device=DEV).double() for a in _unet_data(case, seed))
    flat = torch.as_tensor(_unet_params(case, _rng(case, seed)), device=DEV).double()
    if case["kind"] == "unet_forward":
        with torch.no_grad():
            return torch.cat([_unet_net(case, flat, x[i:i + 1]) for i in range(len(x))])
    flat.requires_grad_(True)
    loss = 0.0
    for i in range(len(x)):  # one volume at a time: the graphs are large
        part = ((_unet_net(case, flat, x[i:i + 1]) - t[i:i + 1]) ** 2).sum() / t.numel()
        part.backward()
        loss += float(part.detach())
    g = flat.grad
    if case["kind"] == "unet_grad":
        return dict(loss=loss, g=g)
    return dict(loss=loss, params=(flat - 1e-3 * g / (g.abs() + 1e-8)).detach())


def exact(case, seed):
    kind = case["kind"]
    if kind == "setup":
        return _exact_setup(case, seed)
    if kind == "fbp":
        return _exact_fbp(case, seed)
    if kind == "tomo":  # from zero objects the first cost is the targets'
        td, tb = (torch.as_tensor(a, device=DEV).double() for a in _tomo_targets(case, seed))
        c = float((td * td).sum() + (tb * tb).sum()) * 0.5 / 2
        return dict(c0=np.array([c, c, 0.0]), c1=None, xd=None, xb=None)
    if kind == "sd":
        return _exact_sd(case, seed)
    if kind == "paganin":
        return _exact_paganin(case, seed)
    if kind.startswith("unet"):
        return _exact_unet(case, seed)
    return None  # the ICD's and the simplex search's paths have no one value
