"""Timed cases of the engine's public entry points.

Each case is one call (or the few calls that belong together) that a user's
program makes: plain and frozen-phonon HRTEM, STEM scans, uneven job sets,
potentials, transmission functions, partial coherence and the surrogate
network.  `prepare` makes what such a program holds before the call (inputs in
HBM, tables, weights), `run` makes one pass, `work` states what a pass cannot do without,
and `exact` gives the pass's results in 64 bits from plain torch.

The transmission stacks are synthetic specimens: SrTiO3-like layers of
thermally displaced atoms whose screened-Coulomb phases are summed in Fourier
space, exp(i phase), band limited to 2/3, so that the waves scatter as they do
in the real ones.
"""
import math

import numpy as np
import torch

import multislice_amd as msx

PIX = 0.1          # Angstrom per pixel, about the sampling of the configurations in use
A0 = 3.905         # SrTiO3 lattice constant
BW = 2.0 / 3.0

# Kirkland's fparams (a1 b1 a2 b2 a3 b3 c1 d1 c2 d2 c3 d3) and Doyle-Turner's
# (a1 b1 .. a4 b4) for O, Si, Ti, Sr: the 64-bit potentials are summed from them
FPARAMS = {
    8: (3.68590229e-1, 3.67542561e-1, 1.32896450e-1, 1.93954830e+1, 2.77101233e-1, 3.67539567e-1,
        8.39309305e-2, 7.58355003e-1, 1.81631127e-1, 2.04360334e+0, 1.05289871e-3, 3.12500946e-2),
    14: (1.20120147e-1, 7.06310153e+1, 1.06498026e+0, 1.04600373e+0, 1.82256296e-1, 8.68866872e-2,
         3.06076088e-2, 2.14762808e-1, 1.10867696e+0, 3.69205948e+0, 1.58258089e+0, 9.93119843e+0),
    22: (7.37291729e-1, 8.32612403e+0, 9.96300042e-1, 4.96982599e-1, 3.55417565e-1, 7.26595855e-2,
         1.63350335e-2, 7.31735660e-2, 3.60199179e-1, 9.57232308e-1, 1.42171303e+0, 1.58512114e+1),
    38: (1.59192012e+0, 2.23207098e-1, 1.68248494e-2, 1.86484813e-2, 1.97760024e+0, 6.41852247e+0,
         4.59884866e+0, 2.52850287e+1, 1.56342068e-3, 1.60766776e-2, 1.74105846e-1, 2.01554275e-1),
}
DOYLE_TURNER = {
    8: (0.4548, 23.7803, 0.9173, 7.6220, 0.4719, 2.1440, 0.1384, 0.2959),
    14: (2.1293, 57.7748, 2.5333, 16.4756, 0.8349, 2.8796, 0.3216, 0.3860),
    22: (3.5653, 81.9821, 2.8181, 19.0486, 1.8930, 3.5904, 0.4825, 0.3855),
    38: (5.8478, 104.9721, 4.0026, 19.3666, 2.3420, 3.7368, 0.8795, 0.4142),
}
U_RMS = {8: 0.095, 14: 0.076, 22: 0.075, 38: 0.088}


def listed():
    return [
        # the smallest HRTEM run: one plane wave through an 80-slice Si slab on
        # 256^2 (the tutorial-sized call; latency and launches count)
        dict(name="hrtem_256_one_wave", kind="hrtem", nx=256, ny=256, nslice=80, nwave=1, kev=200.0, prec="f32"),
        # a few tilted-cell waves in the FP64 engine on a rectangular grid, as
        # run to check an FP32 result
        dict(name="hrtem_384x512_f64", kind="hrtem", nx=384, ny=512, nslice=30, nwave=3, kev=300.0, prec="f64",
             tilt=0.004),
        # large frozen-phonon HRTEM: 8 configurations of 2048^2 through one
        # batched loop, then the objective-lens images
        dict(name="frozen_phonon_2048", kind="frozen", n=2048, nslice=12, nconf=8, kev=300.0),
        # a queue of uneven HRTEM jobs (grids 256 to 1024, mixed beam energies
        # and thicknesses) submitted at once
        dict(name="uneven_jobs", kind="jobs", njobs=24, nmin=256, nmax=1024, smin=10, smax=48),
        # the batched STEM scan with its saved tuning and graphs on
        dict(name="stem_512", kind="stem", nx=512, ny=512, nslice=100, nprobe=320, ncheck=1, ndet=2, kev=300.0,
             tuned=True),
        # a STEM thickness series on a small grid with nothing tuned: ragged
        # probe count, four annuli, three thicknesses
        dict(name="stem_256_thickness", kind="stem", nx=256, ny=256, nslice=40, nprobe=777, ncheck=3, ndet=4,
             kev=300.0, tuned=False),
        # the potential of one displaced configuration of the large frozen-
        # phonon specimen, atoms resident in HBM
        dict(name="potential_2048", kind="potential", n=2048, cells=52, nslice=24, where="device", radius=3.0),
        # transmission functions of a slab of layers
        dict(name="transmission_1024", kind="transmission", nx=1024, ny=1024, nlayer=40, kev=300.0),
        # reciprocal-space (Doyle-Turner) potential of a supercell
        dict(name="potential_rec_512", kind="rec", nx=512, ny=512, cells=12, nslice=20),
        # a partial-coherence image: illumination cone and defocus spread
        dict(name="partial_coherence_256", kind="partial", n=256, nslice=80, cone=2.5e-3, dfdelt=10.0),
        # the surrogate on one 128^2 image of 4 configurations
        dict(name="surrogate_forward_128", kind="unet", levels=4, base=32, cin=4, n=1, h=128, w=128),
        # four training steps of the surrogate on minibatches of 16 32^2 images
        dict(name="surrogate_train_32", kind="train", levels=4, base=32, cin=4, n=16, h=32, w=32, steps=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("hrtem", "hrtem", "frozen", "jobs", "stem", "stem", "potential", "potential", "transmission",
                       "rec", "partial", "unet", "train"))
    grids = (128, 256, 384, 512, 768, 1024)
    kev = rng.choice((100.0, 200.0, 300.0))
    if kind == "hrtem":
        nx, ny = rng.choice(grids), rng.choice(grids)
        prec = rng.choice(("f32", "f32", "f64"))
        px = nx * ny * (2 if prec == "f64" else 1)
        nwave = _log_int(rng, 1, max(1, min(16, (1 << 22) // px)))
        return dict(kind=kind, nx=nx, ny=ny, nslice=_log_int(rng, 5, 100), nwave=nwave, kev=kev, prec=prec,
                    tilt=rng.choice((0.0, 0.006)))
    if kind == "frozen":
        return dict(kind=kind, n=rng.choice((768, 1024, 2048)), nslice=_log_int(rng, 3, 12),
                    nconf=_log_int(rng, 1, 8), kev=kev)
    if kind == "jobs":
        return dict(kind=kind, njobs=_log_int(rng, 2, 24), nmin=256, nmax=rng.choice((384, 768, 1024)), smin=5,
                    smax=_log_int(rng, 8, 48))
    if kind == "stem":
        nx, ny = rng.choice((128, 256, 384, 512)), rng.choice((128, 256, 384, 512))
        cap = max(1, min(900, (80 << 20) // (nx * ny)))
        return dict(kind=kind, nx=nx, ny=ny, nslice=_log_int(rng, 8, 100), nprobe=_log_int(rng, 5, cap),
                    ncheck=rng.choice((1, 1, 2, 4)), ndet=rng.choice((1, 2, 3, 5)), kev=kev, tuned=False)
    if kind == "potential":
        n = rng.choice((256, 512, 1024, 2048))
        return dict(kind=kind, n=n, cells=max(2, int(n * PIX / A0) + rng.choice((-1, 0, 1))),
                    nslice=_log_int(rng, 2, max(4, min(100, (24 * 2048 * 2048) // (n * n)))),
                    where=rng.choice(("device", "host")), radius=rng.choice((2.0, 3.0, 4.0)))
    if kind == "transmission":
        nx, ny = rng.choice(grids + (2048,)), rng.choice(grids)
        return dict(kind=kind, nx=nx, ny=ny, nlayer=_log_int(rng, 1, max(2, min(100, (40 << 20) // (nx * ny)))), kev=kev)
    if kind == "rec":
        nx, ny = rng.choice((128, 256, 512)), rng.choice((128, 256, 512))
        return dict(kind=kind, nx=nx, ny=ny, cells=rng.randint(2, 12), nslice=_log_int(rng, 1, 20))
    if kind == "partial":
        return dict(kind=kind, n=rng.choice((128, 256)), nslice=_log_int(rng, 8, 80),
                    cone=rng.uniform(1e-3, 2.5e-3), dfdelt=rng.choice((10.0, 20.0, 40.0)))
    if kind == "unet":
        h, w = 8 * rng.randint(4, 20), 8 * rng.randint(4, 20)
        return dict(kind=kind, levels=rng.choice((3, 4)), base=rng.choice((16, 32)), cin=rng.choice((1, 4)),
                    n=_log_int(rng, 1, max(1, (1 << 18) // (h * w))), h=h, w=w)
    return dict(kind="train", levels=rng.choice((3, 4)), base=rng.choice((16, 32)), cin=rng.choice((1, 4)),
                n=_log_int(rng, 2, 16), h=8 * rng.randint(3, 6), w=8 * rng.randint(3, 6), steps=rng.randint(1, 4))


# ------------------------------------------------------------------ inputs
_ctx = {}


def _context(tuned=False):
    """One long-lived context, as a program keeps, and a second one that holds
    the saved tuning of the 512^2 scan and replays its loops from graphs."""
    if not tuned:
        return msx.context()
    if "tuned" not in _ctx:
        c = msx.Context(0)
        c.set_tuning(512, 512, msx.F32, dict(row_wpb=8, col_wpb=-1, batch=160, col_tile=8, row_plan=0, col_plan=0))
        c.set_graphs(True)
        _ctx["tuned"] = c
    return _ctx["tuned"]


def _gen(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + salt)


def _freq2(n, a):
    """freqn's k^2 in float arithmetic."""
    i = np.arange(n)
    i = np.where(i > int(n / 2.0 + 0.5), i - n, i)
    k = i.astype(np.float32) / np.float32(a)
    return k * k


def _freq(n, a):
    i = np.arange(n)
    return np.where(i > int(n / 2.0 + 0.5), i - n, i) / float(a)


def _k2max(nx, ny, ax, by, bw):
    k = min(np.float32(nx) / np.float32(np.float32(2) * np.float32(ax)),
            np.float32(ny) / np.float32(np.float32(2) * np.float32(by)))
    k = np.float32(np.float32(bw) * k)
    return np.float32(k * k)


def _mask(nx, ny, ax, by, bw=BW):
    k2 = _freq2(nx, ax)[:, None] + _freq2(ny, by)[None, :]
    return torch.from_numpy(k2 < _k2max(nx, ny, ax, by, bw)).cuda()


def _k2grid(nx, ny, ax, by):
    return torch.from_numpy(_freq2(nx, ax)[:, None] + _freq2(ny, by)[None, :]).cuda()


def _phases(nlayer, nx, ny, seed, salt=0):
    """(nlayer, nx, ny) float32 phases sigma V of displaced SrTiO3-like layers."""
    ax, by = nx * PIX, ny * PIX
    g = _gen(seed, salt)
    mx, my = max(1, round(ax / A0)), max(1, round(by / A0))
    basis = ((38, 0.0, 0.0, 0), (8, 0.5, 0.5, 0), (22, 0.5, 0.5, 1), (8, 0.5, 0.0, 1), (8, 0.0, 0.5, 1))
    ii, jj = torch.meshgrid(torch.arange(mx, device="cuda"), torch.arange(my, device="cuda"), indexing="ij")
    out = torch.empty((nlayer, nx, ny), dtype=torch.float32, device="cuda")
    kx = torch.from_numpy(_freq(nx, ax)).cuda()[:, None]
    ky = torch.from_numpy(_freq(ny, by)).cuda()[None, :]
    k2 = kx * kx + ky * ky
    shape = (torch.exp(-0.35 * k2) / (k2 + 0.15)).to(torch.float32)
    shape *= 0.6 / 38 / float(shape.mean())
    for l in range(nlayer):
        rho = torch.zeros(nx * ny, dtype=torch.int32, device="cuda")
        for Z, fx, fy, par in basis:
            if par != l % 2:
                continue
            d = torch.randn((2, mx, my), generator=g, device="cuda") * U_RMS[Z]
            px = torch.round(((ii + fx) * (ax / mx) + d[0]) / PIX).long() % nx
            py = torch.round(((jj + fy) * (by / my) + d[1]) / PIX).long() % ny
            rho.index_add_(0, (px * ny + py).reshape(-1), torch.full((mx * my,), Z, dtype=torch.int32, device="cuda"))
        out[l] = torch.fft.ifft2(torch.fft.fft2(rho.reshape(nx, ny).to(torch.float32)) * shape).real
    return out


def _trans(nlayer, nx, ny, seed, salt=0, f64=False):
    ph = _phases(nlayer, nx, ny, seed, salt)
    m = _mask(nx, ny, nx * PIX, ny * PIX)
    out = torch.empty((nlayer, nx, ny), dtype=torch.complex128 if f64 else torch.complex64, device="cuda")
    for l in range(nlayer):
        p = ph[l].to(torch.float64) if f64 else ph[l]
        out[l] = torch.fft.ifft2(torch.fft.fft2(torch.polar(torch.ones_like(p), p)) * m)
    return out


def _crystal(cells, a, b, c, nslice, seed):
    """Displaced SrTiO3 layers filling a x b x c, `nslice` atomic planes."""
    rng = np.random.default_rng(seed)
    dz = c / nslice
    ii, jj = np.meshgrid(np.arange(cells), np.arange(cells), indexing="ij")
    rec = []
    for l in range(nslice):
        for Z, fx, fy, par in ((38, 0, 0, 0), (8, .5, .5, 0), (22, .5, .5, 1), (8, .5, 0, 1), (8, 0, .5, 1)):
            if par != l % 2:
                continue
            n = ii.size
            d = rng.standard_normal((3, n)) * U_RMS[Z]
            at = np.zeros(n, msx.ATOM_DTYPE)
            at["Z"], at["occ"] = Z, 1.0
            at["x"] = (ii.ravel() + fx) * (a / cells) + d[0]
            at["y"] = (jj.ravel() + fy) * (b / cells) + d[1]
            at["z"] = (l + 0.5) * dz + np.clip(d[2], -0.4 * dz, 0.4 * dz)
            rec.append(at)
    return np.concatenate(rec)


def _conv_specs(case):
    C = [case["base"] << l for l in range(case["levels"])]
    s = []
    for l in range(case["levels"]):
        s += [(case["cin"] if l == 0 else C[l - 1], C[l], 3, l), (C[l], C[l], 3, l)]
    for l in range(case["levels"] - 2, -1, -1):
        s += [(C[l + 1] + C[l], C[l], 3, l), (C[l], C[l], 3, l)]
    return s + [(C[0], 1, 1, 0)]


def _params(case, seed):
    rng = np.random.default_rng(seed)
    out, specs = [], _conv_specs(case)
    for i, (ci, co, k, _) in enumerate(specs):
        sd = math.sqrt(2.0 / (ci * k * k)) * (0.1 if i == len(specs) - 1 else 1.0)
        out += [rng.standard_normal(co * ci * k * k) * sd, rng.standard_normal(co) * 0.02]
    return np.concatenate(out).astype(np.float32)


def _images(n, c, h, w, seed, salt):
    """ADF-like images around a mean of 1: a smooth column pattern plus the
    scatter between configurations."""
    g = _gen(seed, salt)
    y = torch.arange(h, device="cuda")[:, None] / h
    x = torch.arange(w, device="cuda")[None, :] / w
    ph = torch.rand((n, 4), generator=g, device="cuda") * 6.2831853
    f = 4 * math.pi
    base = 1 + 0.5 * (torch.cos(f * y + ph[:, 0, None, None]) * torch.cos(f * x + ph[:, 1, None, None]))
    base = base + 0.2 * torch.cos(2 * f * (x + y) + ph[:, 2, None, None])
    im = base[:, None] + 0.08 * torch.randn((n, c, h, w), generator=g, device="cuda")
    return im.contiguous(), base.contiguous()


def _hk(case):
    return np.arange(case["nslice"], dtype=np.int32)


def _jobs(case, seed):
    rng = np.random.default_rng(case["njobs"] * 977 + case["smax"])  # the job list is the case's, the specimens the seed's
    sizes = [n for n in (256, 384, 512, 768, 1024) if case["nmin"] <= n <= case["nmax"]]
    jobs = []
    for j in range(case["njobs"]):
        n = int(rng.choice(sizes))
        ns = int(rng.integers(case["smin"], case["smax"] + 1))
        jobs.append((n, ns, float(rng.choice((200.0, 300.0))), j))
    return jobs


_LENS = dict(cs=1.3e7, df=700.0, aobj=0.024, dfa2=30.0, dfa2phi=0.5)
_SPREAD = 40.0


def prepare(case, seed):
    k = case["kind"]
    s = dict(case=case, ctx=_context(bool(case.get("tuned"))))
    if k == "hrtem":
        nx, ny, f64 = case["nx"], case["ny"], case["prec"] == "f64"
        cdt = torch.complex128 if f64 else torch.complex64
        s["trans"] = _trans(case["nslice"], nx, ny, seed, f64=f64)
        s["cz"], s["layer"] = np.full(case["nslice"], 1.9525), _hk(case)
        s["psi0"] = torch.ones((nx, ny), dtype=cdt, device="cuda")
        s["psi"] = torch.empty((case["nwave"], nx, ny), dtype=cdt, device="cuda")
    elif k == "frozen":
        n = case["n"]
        cz, layer = np.full(case["nslice"], 1.9525), _hk(case)
        s["psi0"] = torch.ones((n, n), dtype=torch.complex64, device="cuda")
        s["jobs"] = [dict(trans=_trans(case["nslice"], n, n, seed, c),
                          psi=torch.empty((n, n), dtype=torch.complex64, device="cuda"), psi0=s["psi0"], ax=n * PIX,
                          by=n * PIX, kev=case["kev"], cz=cz, layer=layer) for c in range(case["nconf"])]
    elif k == "jobs":
        s["jobs"], one = [], {}
        for n, ns, kev, j in _jobs(case, seed):
            if n not in one:
                one[n] = torch.ones((n, n), dtype=torch.complex64, device="cuda")
            s["jobs"].append(dict(trans=_trans(ns, n, n, seed, j), psi=torch.empty_like(one[n]), psi0=one[n],
                                  ax=n * PIX, by=n * PIX, kev=kev, cz=np.full(ns, 2.0), layer=np.arange(ns)))
    elif k == "stem":
        nx, ny = case["nx"], case["ny"]
        s["trans"] = _trans(case["nslice"], nx, ny, seed)
        s["cz"], s["layer"] = np.full(case["nslice"], 1.9525), _hk(case)
        s.update(_stem_set(case, seed))
    elif k == "potential":
        at = _crystal(case["cells"], case["n"] * PIX, case["n"] * PIX, 1.9525 * case["nslice"], case["nslice"], seed)
        s["atoms"] = at
        if case["where"] == "device":
            s["atoms"] = torch.from_numpy(at.view(np.uint8).copy()).cuda()
        s["V"] = torch.empty((case["nslice"], case["n"], case["n"]), dtype=torch.float32, device="cuda")
    elif k == "transmission":
        nx, ny = case["nx"], case["ny"]
        s["V"] = _phases(case["nlayer"], nx, ny, seed) * (1000.0 / _sigma(case["kev"]))
        s["t"] = torch.empty((case["nlayer"], nx, ny), dtype=torch.complex64, device="cuda")
    elif k == "rec":
        c = 1.9525 * case["nslice"]
        s["cell"] = (case["cells"] * A0, case["cells"] * A0, c)
        s["atoms"] = _crystal(case["cells"], *s["cell"], case["nslice"], seed)
        s["V"] = torch.empty((case["nslice"], case["nx"], case["ny"]), dtype=torch.float32, device="cuda")
    elif k == "partial":
        s["trans"] = _trans(case["nslice"], case["n"], case["n"], seed)
        s["cz"], s["layer"] = np.full(case["nslice"], 1.35775), _hk(case)
    elif k == "unet":
        s["net"] = msx.UNet(s["ctx"], case["levels"], case["base"], in_channels=case["cin"])
        s["net"].set_params(_params(case, seed))
        x = _images(case["n"], case["cin"], case["h"], case["w"], seed, 1)[0]
        s["x"] = x[:, 0].contiguous() if case["cin"] == 1 else x
        s["out"] = torch.empty((case["n"], case["h"], case["w"]), dtype=torch.float32, device="cuda")
    elif k == "train":
        s["net"] = msx.UNet(s["ctx"], case["levels"], case["base"], in_channels=case["cin"])
        s["net"].set_params(_params(case, seed))
        s["batches"] = []
        for i in range(case["steps"]):
            x, t = _images(case["n"], case["cin"], case["h"], case["w"], seed, 10 + i)
            s["batches"].append((x[:, 0].contiguous() if case["cin"] == 1 else x, t))
    return s


def _stem_set(case, seed):
    """Probe (21 mrad, Cs 1 um), ragged scan of the central cells, annuli up to
    the band limit, evenly spaced thicknesses."""
    nx, ny, kev = case["nx"], case["ny"], case["kev"]
    lam = _wavelength(kev)
    rng = np.random.default_rng(seed)
    pos = np.stack([nx * PIX * (0.4 + 0.2 * rng.random(case["nprobe"])),
                    ny * PIX * (0.4 + 0.2 * rng.random(case["nprobe"]))], 1)
    kb = BW * 0.5 / PIX
    edges = [0.0, 0.010 / lam] + [kb * f for f in (0.3, 0.5, 0.7, 0.9, 1.01)]
    det = [(edges[0], edges[1])] + [(edges[1 + d], edges[2 + d]) for d in range(1, case["ndet"])]
    if case["ndet"] == 2:
        det[1] = (0.8 * kb, 1.5 * kb)
    ck = [max(1, round(case["nslice"] * (i + 1) / case["ncheck"])) for i in range(case["ncheck"])]
    return dict(probe=dict(alpha_max=0.021, cs=1.0e4, df=0.0), pos=pos, det=det, ck=ck)


def run(s):
    case, ctx = s["case"], s["ctx"]
    k = case["kind"]
    if k == "hrtem":
        tl = case.get("tilt", 0.0)
        ctx.multislice(s["trans"], s["cz"], s["layer"], s["psi"], case["nx"] * PIX, case["ny"] * PIX, case["kev"],
                       tilt=(tl, -0.5 * tl), psi0=s["psi0"])
        return s["psi"]
    if k == "frozen":
        ctx.multislice_batch(s["jobs"])
        im = [ctx.ctf_image(j["psi"], j["ax"], j["by"], j["kev"], 1.2e7, -600.0, 0.020) for j in s["jobs"]]
        return [[j["psi"] for j in s["jobs"]], im]
    if k == "jobs":
        ctx.multislice_batch(s["jobs"])
        return [j["psi"] for j in s["jobs"]]
    if k == "stem":
        out = ctx.stem(s["trans"], s["cz"], s["layer"], case["nx"] * PIX, case["ny"] * PIX, case["kev"], s["probe"],
                       s["pos"], s["det"], s["ck"])
        return out.astype(np.float32)  # scans are stored and trained on as float images
    if k == "potential":
        L = case["n"] * PIX
        return ctx.potential(s["atoms"], (L, L, 1.9525 * case["nslice"]), case["n"], case["n"], case["nslice"],
                             case["radius"], out=s["V"])
    if k == "transmission":
        return ctx.transmission(s["V"], case["nx"] * PIX, case["ny"] * PIX, case["kev"], out=s["t"])
    if k == "rec":
        return ctx.potential_rec(s["atoms"], s["cell"], case["nx"], case["ny"], case["nslice"], dw=0.5, out=s["V"])
    if k == "partial":
        L = case["n"] * PIX
        img, _, _ = ctx.partial_coherence(s["trans"], s["cz"], s["layer"], L, L, 200.0, _LENS, 0.0, case["cone"],
                                          _SPREAD, case["dfdelt"])
        return img.float()  # the float image that is written out
    if k == "unet":
        return s["net"].forward(s["x"], out=s["out"])
    loss = [s["net"].train_step(x, t, 1e-3) for x, t in s["batches"]]
    return dict(loss=np.array(loss, np.float32), params=s["net"].params())


# ------------------------------------------------------------------ work
def _fft_flops(nx, ny):
    return 5.0 * nx * ny * math.log2(nx * ny)


def _slice_work(nx, ny, nslice, nwave, cbytes, own_trans=False):
    px = nx * ny
    return (px * cbytes * (nslice * (nwave if own_trans else 1) + 2 * nwave),
            nwave * nslice * (2 * _fft_flops(nx, ny) + 18.0 * px))


def work(case):
    k = case["kind"]
    if k == "hrtem":
        by, fl = _slice_work(case["nx"], case["ny"], case["nslice"], case["nwave"], 16 if case["prec"] == "f64" else 8)
    elif k == "frozen":
        n = case["n"]
        by, fl = _slice_work(n, n, case["nslice"], case["nconf"], 8, True)
        by += case["nconf"] * n * n * 4
        fl += case["nconf"] * 2 * _fft_flops(n, n)
    elif k == "jobs":
        by = fl = 0.0
        for n, ns, _, _ in _jobs(case, 0):
            b, f = _slice_work(n, n, ns, 1, 8)
            by, fl = by + b, fl + f
    elif k == "stem":
        nx, ny = case["nx"], case["ny"]
        by = nx * ny * 8.0 * case["nslice"] + case["nprobe"] * (16 + 8 * case["ndet"] * case["ncheck"])
        fl = case["nprobe"] * case["nslice"] * (2 * _fft_flops(nx, ny) + 18.0 * nx * ny)
    elif k == "potential":
        n, px = case["n"], case["n"] ** 2
        nat = case["cells"] ** 2 * (2 * ((case["nslice"] + 1) // 2) + 3 * (case["nslice"] // 2))
        pairs = nat * math.pi * case["radius"] ** 2 / PIX ** 2
        by, fl = px * case["nslice"] * 4.0 + nat * 32.0, pairs * 12.0
    elif k == "transmission":
        px = case["nx"] * case["ny"] * case["nlayer"]
        by, fl = px * 12.0, case["nlayer"] * 2 * _fft_flops(case["nx"], case["ny"])
    elif k == "rec":
        px = case["nx"] * case["ny"]
        nat = case["cells"] ** 2 * (2 * ((case["nslice"] + 1) // 2) + 3 * (case["nslice"] // 2))
        by, fl = px * case["nslice"] * 4.0 + nat * 32.0, px * (8.0 * nat) + case["nslice"] * _fft_flops(*(case["nx"], case["ny"]))
    elif k == "partial":
        n = case["n"]
        nang = len(_angles(case))
        nd = 2 * int(2.5 * _SPREAD / case["dfdelt"]) + 1
        by, fl = _slice_work(n, n, case["nslice"], nang, 8)
        by = n * n * 8.0 * (case["nslice"] + 1)
        fl += nang * (1 + nd) * _fft_flops(n, n)
    else:
        conv = sum(2.0 * ci * co * kk * kk * (case["h"] >> l) * (case["w"] >> l) for ci, co, kk, l in _conv_specs(case))
        npar = sum(ci * co * kk * kk + co for ci, co, kk, _ in _conv_specs(case))
        px = case["n"] * case["h"] * case["w"]
        if k == "unet":
            by, fl = 4.0 * (npar + px * (case["cin"] + 1)), conv * case["n"]
        else:  # weights and both moments read and written each step, the weights handed out at the end
            by = case["steps"] * (4.0 * px * (case["cin"] + 1) + 24.0 * npar) + 4.0 * npar
            fl = 3.0 * conv * case["n"] * case["steps"]
    return {"bytes": float(by), "flops": float(fl)}


# ------------------------------------------------------------------ 64 bits
def _wavelength(kev):
    return 12.3984244 / math.sqrt(kev * (2 * 510.99906 + kev))


def _sigma(kev):
    x = (510.99906 + kev) / (2.0 * 510.99906 + kev)
    return 2.0 * math.pi * x / (_wavelength(kev) * kev)


def _propagator(nx, ny, kev, cz, tilt=(0.0, 0.0)):
    lam = _wavelength(kev)
    ax, by = nx * PIX, ny * PIX
    kx = torch.from_numpy(_freq(nx, ax)).cuda()[:, None]
    ky = torch.from_numpy(_freq(ny, by)).cuda()[None, :]
    ph = math.pi * cz * (kx * kx * lam - kx * 2 * math.tan(tilt[0]) + ky * ky * lam - ky * 2 * math.tan(tilt[1]))
    return torch.polar(torch.ones_like(ph), -ph) * _mask(nx, ny, ax, by)


def _propagate(psi, trans, nslice, P, checks=None):
    """Kirkland's loop with +i forward transforms; `checks` {slice: fn(spectrum)}."""
    for s in range(nslice):
        f = torch.fft.ifft2(psi * trans[s].to(torch.complex128), norm="forward") * P
        if checks and s + 1 in checks:
            checks[s + 1](f)
            if s + 1 == max(checks):
                return None
        psi = torch.fft.fft2(f, norm="forward")
    return psi


def _lens_image(psi, n, kev, cs, df, aobj):
    lam = _wavelength(kev)
    k2f = _k2grid(n, n, n * PIX, n * PIX)
    kx = torch.from_numpy(_freq(n, n * PIX)).cuda()
    k2 = kx[:, None] ** 2 + kx[None, :] ** 2
    chi = math.pi * lam * k2 * (0.5 * cs * lam * lam * k2 - df)
    H = torch.polar(torch.ones_like(chi), -chi) * (k2f <= float(np.float32((aobj / lam) ** 2)))
    return torch.fft.fft2(torch.fft.ifft2(psi, norm="forward") * H, norm="forward").abs() ** 2


def _angles(case):
    lam, r = np.float32(_wavelength(200.0)), np.float32(1.0) / np.float32(case["n"] * PIX)
    q2 = np.float32(np.float32(case["cone"]) / lam) ** 2
    m = int(np.float32(case["cone"]) / (lam * r) + np.float32(1.5))
    return [(ix, iy) for iy in range(-m, m + 1) for ix in range(-m, m + 1)
            if np.float32((ix * r) ** 2) + np.float32((iy * r) ** 2) <= q2]


def _exact_stem(case, seed):
    nx, ny, kev = case["nx"], case["ny"], case["kev"]
    tr, st = _trans(case["nslice"], nx, ny, seed), _stem_set(case, seed)
    lam = _wavelength(kev)
    P = _propagator(nx, ny, kev, 1.9525)
    k2f = _k2grid(nx, ny, nx * PIX, ny * PIX)
    kx = torch.from_numpy(_freq(nx, nx * PIX)).cuda()[:, None]
    ky = torch.from_numpy(_freq(ny, ny * PIX)).cuda()[None, :]
    k2 = kx * kx + ky * ky
    ap = k2f <= float(np.float32((st["probe"]["alpha_max"] / lam) ** 2))
    amp = math.sqrt(nx * ny / int(ap.sum()))
    chi = math.pi * lam * k2 * (0.5 * st["probe"]["cs"] * lam * lam * k2 - st["probe"]["df"])
    out = np.zeros((case["ncheck"], case["ndet"], case["nprobe"]))
    masks = [((k2f >= float(np.float32(lo * lo))) & (k2f <= float(np.float32(hi * hi)))) for lo, hi in st["det"]]
    step = max(1, (1 << 25) // (nx * ny))
    for p0 in range(0, case["nprobe"], step):
        pos = torch.from_numpy(st["pos"][p0:p0 + step]).cuda()
        ph = -chi + 2 * math.pi * (kx * pos[:, 0, None, None] + ky * pos[:, 1, None, None])
        psi = torch.fft.fft2(torch.polar(torch.full_like(ph, amp), ph) * ap, norm="forward")

        def record(i):
            def fn(f):
                for d, m in enumerate(masks):
                    out[i, d, p0:p0 + step] = ((f.abs() ** 2 * m).sum((-2, -1)) / (nx * ny)).cpu().numpy()
            return fn
        _propagate(psi, tr, case["nslice"], P, {c: record(i) for i, c in enumerate(st["ck"])})
    return out


def _vz(Z, r2):
    p = FPARAMS[Z]
    r = torch.sqrt(r2).clamp_min(1e-10)
    v = torch.zeros_like(r)
    for i in (0, 2, 4):
        v += 300.8242834 * p[i] * torch.special.modified_bessel_k0(2 * 3.141592654 * math.sqrt(p[i + 1]) * r)
    for i in (6, 8, 10):
        v += 150.4121417 * p[i] / p[i + 1] * torch.exp(-(3.141592654 * r) ** 2 / p[i + 1])
    return v


def _exact_potential(case, seed):
    n, L, ns = case["n"], case["n"] * PIX, case["nslice"]
    at = _crystal(case["cells"], L, L, 1.9525 * ns, ns, seed)
    dx, rad = L / n, case["radius"]
    h = int(math.ceil(rad / dx)) + 1
    off = torch.arange(-h, h + 1, device="cuda")
    V = torch.zeros((ns, n * n), dtype=torch.float64, device="cuda")
    kz = np.floor(at["z"] / 1.9525).astype(int)
    for s in range(ns):
        for Z in np.unique(at["Z"]):
            sel = at[(kz == s) & (at["Z"] == Z)]
            for c in range(0, len(sel), 2048):
                x = torch.from_numpy(sel["x"][c:c + 2048].copy()).cuda()
                y = torch.from_numpy(sel["y"][c:c + 2048].copy()).cuda()
                ix, iy = torch.round(x / dx).long()[:, None] + off, torch.round(y / dx).long()[:, None] + off
                r2 = (((ix.double() * dx - x[:, None]) ** 2)[:, :, None] +
                      ((iy.double() * dx - y[:, None]) ** 2)[:, None, :])
                keep = r2 < rad * rad
                at_px = ((ix % n) * n)[:, :, None] + (iy % n)[:, None, :]
                V[s].index_add_(0, at_px[keep], _vz(int(Z), r2[keep]))
    return V.reshape(ns, n, n)


def _exact_rec(case, seed):
    nx, ny, ns = case["nx"], case["ny"], case["nslice"]
    a = case["cells"] * A0
    at = _crystal(case["cells"], a, a, 1.9525 * ns, ns, seed)
    kz = np.floor(at["z"] / 1.9525).astype(int)
    hx, hy = torch.from_numpy(_freq(nx, 1.0)).cuda(), torch.from_numpy(_freq(ny, 1.0)).cuda()
    s2 = 0.25 * ((hx / a)[:, None] ** 2 + (hy / a)[None, :] ** 2)
    live = (hx.abs() < nx // 2)[:, None] & (hy.abs() < ny // 2)[None, :]
    out = torch.empty((ns, nx, ny), dtype=torch.float64, device="cuda")
    for s in range(ns):
        F = torch.zeros((nx, ny), dtype=torch.complex128, device="cuda")
        for Z in np.unique(at["Z"]):
            sel = at[(kz == s) & (at["Z"] == Z)]
            if not len(sel):
                continue
            x, y = torch.from_numpy(sel["x"] / a).cuda(), torch.from_numpy(sel["y"] / a).cuda()
            px, py = -2 * math.pi * hx[:, None] * x[None, :], -2 * math.pi * hy[:, None] * y[None, :]
            S = torch.polar(torch.ones_like(px), px) @ torch.polar(torch.ones_like(py), py).T.contiguous()
            d = DOYLE_TURNER[int(Z)]
            f = sum(d[2 * j] * torch.exp(-(d[2 * j + 1] + 0.5) * s2) for j in range(4))
            F += S * (f / (a * a))
        out[s] = torch.fft.ifft2(F * live, norm="forward").real * (300.8242834 / (2 * math.pi))
    return out


def _exact_partial(case, seed):
    n, L = case["n"], case["n"] * PIX
    tr = _trans(case["nslice"], n, n, seed)
    q = _angles(case)
    x = torch.arange(n, device="cuda", dtype=torch.float64) / (n - 1)
    psi = torch.stack([torch.polar(torch.ones((n, n), dtype=torch.float64, device="cuda"),
                                   2 * math.pi * (ix * x[:, None] + iy * x[None, :])) for ix, iy in q])
    psi = _propagate(psi, tr, case["nslice"], _propagator(n, n, 200.0, 1.35775))
    spec = torch.fft.ifft2(psi, norm="forward")
    lam = _wavelength(200.0)
    kx = torch.from_numpy(_freq(n, L)).cuda()
    k2 = kx[:, None] ** 2 + kx[None, :] ** 2
    phi = torch.atan2(kx[None, :].expand(n, n), kx[:, None].expand(n, n))
    ap = _k2grid(n, n, L, L) <= float(np.float32((_LENS["aobj"] / lam) ** 2))
    img, wsum = torch.zeros((n, n), dtype=torch.float64, device="cuda"), 0.0
    nd = int(2.5 * _SPREAD / case["dfdelt"])
    for i in range(-nd, nd + 1):
        w = math.exp(-0.5 * (i * case["dfdelt"] / _SPREAD) ** 2)
        chi = math.pi * lam * k2 * (0.5 * _LENS["cs"] * lam * lam * k2 - (_LENS["df"] + i * case["dfdelt"]) +
                                    _LENS["dfa2"] * torch.sin(2 * (phi - _LENS["dfa2phi"])))
        H = torch.polar(torch.ones_like(chi), -chi) * ap
        img += w * (torch.fft.fft2(spec * H, norm="forward").abs() ** 2).sum(0)
        wsum += w
    return img / (len(q) * wsum)


def _unet64(case, p, x):
    """The network in FP64 on the packed weights p; x (n, cin, h, w)."""
    L, specs = case["levels"], _conv_specs(case)
    offs = np.cumsum([0] + [ci * co * k * k + co for ci, co, k, _ in specs])

    def conv(i, v):
        ci, co, k, _ = specs[i]
        w = p[int(offs[i]):int(offs[i]) + ci * co * k * k].reshape(co, ci * k * k)
        b = p[int(offs[i]) + ci * co * k * k:int(offs[i + 1])]
        n, _, h, wd = v.shape
        u = torch.nn.functional.unfold(v, k, padding=k // 2)
        y = torch.stack([w @ u[j] for j in range(n)]) + b[:, None]
        return y.reshape(n, co, h, wd)

    enc, v = [], x
    for l in range(L):
        v = torch.relu(conv(2 * l + 1, torch.relu(conv(2 * l, v))))
        enc.append(v)
        if l < L - 1:
            v = torch.nn.functional.avg_pool2d(v, 2)
    i = 2 * L
    for l in range(L - 2, -1, -1):
        v = torch.cat([v.repeat_interleave(2, 2).repeat_interleave(2, 3), enc[l]], 1)
        v = torch.relu(conv(i + 1, torch.relu(conv(i, v))))
        i += 2
    return x.mean(1) + conv(i, v)[:, 0]


def _exact_train(case, seed):
    p = torch.from_numpy(_params(case, seed)).cuda().double().requires_grad_()
    m, v, loss = torch.zeros_like(p), torch.zeros_like(p), []
    for i in range(case["steps"]):
        x, t = _images(case["n"], case["cin"], case["h"], case["w"], seed, 10 + i)
        e = ((_unet64(case, p, x.double()) - t.double()) ** 2).mean()
        g, = torch.autograd.grad(e, p)
        loss.append(float(e))
        with torch.no_grad():
            m = 0.9 * m + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            p -= 1e-3 * (m / (1 - 0.9 ** (i + 1))) / (torch.sqrt(v / (1 - 0.999 ** (i + 1))) + 1e-8)
    return dict(loss=np.array(loss), params=p.detach())


def exact(case, seed):
    k = case["kind"]
    if k == "hrtem":
        f64 = case["prec"] == "f64"
        tl = case.get("tilt", 0.0)
        tr = _trans(case["nslice"], case["nx"], case["ny"], seed, f64=f64)
        psi = torch.ones((case["nx"], case["ny"]), dtype=torch.complex128, device="cuda")
        psi = _propagate(psi, tr, case["nslice"],
                         _propagator(case["nx"], case["ny"], case["kev"], 1.9525, (tl, -0.5 * tl)))
        return psi[None].expand(case["nwave"], -1, -1)
    if k == "frozen":
        n, out = case["n"], []
        P = _propagator(n, n, case["kev"], 1.9525)
        for c in range(case["nconf"]):
            psi = torch.ones((n, n), dtype=torch.complex128, device="cuda")
            out.append(_propagate(psi, _trans(case["nslice"], n, n, seed, c), case["nslice"], P))
        return [out, [_lens_image(p, n, case["kev"], 1.2e7, -600.0, 0.020) for p in out]]
    if k == "jobs":
        return [_propagate(torch.ones((n, n), dtype=torch.complex128, device="cuda"), _trans(ns, n, n, seed, j), ns,
                           _propagator(n, n, kev, 2.0)) for n, ns, kev, j in _jobs(case, seed)]
    if k == "stem":
        return _exact_stem(case, seed)
    if k == "potential":
        return _exact_potential(case, seed)
    if k == "transmission":
        V = _phases(case["nlayer"], case["nx"], case["ny"], seed) * (1000.0 / _sigma(case["kev"]))
        m = _mask(case["nx"], case["ny"], case["nx"] * PIX, case["ny"] * PIX)
        out = torch.empty(V.shape, dtype=torch.complex128, device="cuda")
        for l in range(case["nlayer"]):
            p = V[l].double() * (_sigma(case["kev"]) / 1000.0)
            out[l] = torch.fft.ifft2(torch.fft.fft2(torch.polar(torch.ones_like(p), p)) * m)
        return out
    if k == "rec":
        return _exact_rec(case, seed)
    if k == "partial":
        return _exact_partial(case, seed)
    if k == "unet":
        x = _images(case["n"], case["cin"], case["h"], case["w"], seed, 1)[0].double()
        p = torch.from_numpy(_params(case, seed)).cuda().double()
        return torch.cat([_unet64(case, p, x[i:i + 1]) for i in range(case["n"])])
    return _exact_train(case, seed)
