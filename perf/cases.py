"""Timing cases: the work a user has this package do, through its public calls.

``listed`` holds the calls of a run from the initial conditions to the 21-cm
power spectrum at the sizes of the package's configurations; ``draw`` gives
more of the same kinds over their ranges.  A case is a dict of plain values;
``prepare`` makes its inputs on the GPU from a seed, ``run`` is one pass,
``work`` its unavoidable bytes and operations and ``exact`` the same outputs
in 64 bits, in plain torch.

Kinds:
  bubbles     conv_bubbles on one density box
  batch       BatchedBubbles on boxes of mixed size, barrier and efficiency
  initialize  initial conditions: random field, smoothed box, displacements
  perturb     Zel'dovich mass move to z, and the velocity boxes at z
  power       brightness temperature and its binned power spectrum
  infer       U-Net surrogate, inference
  train       U-Net surrogate, one training step
"""
import importlib
import math
import random

import numpy as np
import torch

DEV = "cuda"
# defaults of the radius schedule (Parameter_files/INIT_PARAMS.py)
R_MAX, R_MIN, R_FACTOR, L_FACTOR = 30.0, 0.5, 1.1, float(np.float32(0.620350491))
D_INIT = 0.12 * 9.0 / 301.0  # linear growth at z = 300
GROUPS = 3                   # box sides in a batch


def _mod(name):
    return importlib.import_module("21cmpy_amd." + name)


def _growth(z):
    return 0.12 * 9.0 / (1.0 + z)


# ------------------------------------------------------------------ cases

def listed():
    return [
        # the smallest box (64^3, linear density): a quick look, latency counts
        dict(name="bubbles_64_linear", kind="bubbles", D=64, box_len=100.0, linear=True, filter=1, update=0,
             zeta=30.0, z=8.0, mean=0.5),
        # the default HII_DIM, nonlinear density
        dict(name="bubbles_128_nonlinear", kind="bubbles", D=128, box_len=128.0, linear=False, filter=1, update=0,
             zeta=40.0, z=8.0, mean=0.4),
        # the benchmark's box, half way through reionization
        dict(name="bubbles_256_nonlinear", kind="bubbles", D=256, box_len=300.0, linear=False, filter=1, update=0,
             zeta=30.0, z=8.0, mean=0.5),
        # the largest box of the configurations
        dict(name="bubbles_512_linear", kind="bubbles", D=512, box_len=500.0, linear=True, filter=1, update=0,
             zeta=25.0, z=8.0, mean=0.5),
        # a side that is no power of two and has no tuned transform
        dict(name="bubbles_200_ragged", kind="bubbles", D=200, box_len=300.0, linear=False, filter=1, update=0,
             zeta=30.0, z=9.0, mean=0.3),
        # the sphere-painting algorithm
        dict(name="bubbles_128_spheres", kind="bubbles", D=128, box_len=200.0, linear=False, filter=1, update=1,
             zeta=30.0, z=8.0, mean=0.3),
        # many boxes at once: a parameter study
        dict(name="batch_64_mixed", kind="batch", nbox=64, d0=96, d1=128, d2=160, cell=1.5625, linear=True, filter=1,
             pick=0),
        # initial conditions of the benchmark's box
        dict(name="initialize_512_256", kind="initialize", DIM=512, HII_DIM=256, box_len=300.0, pspec="powerlaw"),
        # its density and velocities at z
        dict(name="perturb_512_256", kind="perturb", DIM=512, HII_DIM=256, box_len=300.0, scheme="cic",
             velocities=True, z=8.0),
        # its 21-cm signal
        dict(name="power_256", kind="power", D=256, box_len=300.0, nbins=40, z=8.0, x_HI=0.5, dimensional=False),
        # the surrogate, serving and training
        dict(name="infer_128", kind="infer", D=128, batch=8),
        dict(name="train_128", kind="train", D=128, batch=4, lr=1e-4),
    ]


def _log_even(rng, lo, hi):
    return 2 * int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / 2))


def draw(rng):
    kind = rng.choice(["bubbles", "bubbles", "bubbles", "batch", "initialize", "perturb", "power", "infer", "train"])
    if kind == "bubbles":
        # half of them on the sides with tuned transforms, half on any even side
        D = rng.choice([64, 96, 128, 160, 256]) if rng.random() < 0.5 else _log_even(rng, 48, 300)
        return dict(kind=kind, D=D, box_len=round(D * rng.uniform(0.9, 2.0), 1), linear=rng.random() < 0.5,
                    filter=rng.choice([0, 1, 1, 1, 2]), update=1 if D <= 160 and rng.random() < 0.25 else 0,
                    zeta=round(rng.uniform(10.0, 60.0), 2), z=round(rng.uniform(6.5, 11.0), 2),
                    mean=round(rng.uniform(0.1, 0.85), 3))
    if kind == "batch":
        sides = [rng.choice([64, 96, 128, 160]) for _ in range(GROUPS)]
        return dict(kind=kind, nbox=rng.randint(3, 40), d0=sides[0], d1=sides[1], d2=sides[2],
                    cell=round(rng.uniform(1.0, 2.0), 3), linear=rng.random() < 0.5, filter=1,
                    pick=rng.randrange(1 << 20))
    if kind == "initialize":
        hii = _log_even(rng, 32, 256)
        ratio = rng.choice([r for r in (1, 2, 2, 3, 4) if r * hii <= 512])
        return dict(kind=kind, DIM=ratio * hii, HII_DIM=hii, box_len=round(hii * rng.uniform(0.9, 2.0), 1),
                    pspec=rng.choice(["powerlaw", "powerlaw", "planck"]))
    if kind == "perturb":
        ratio = rng.choice([1, 2, 2, 4])
        dim = 16 * ratio * max(1, int(round(math.exp(rng.uniform(math.log(64), math.log(480))) / (16 * ratio))))
        return dict(kind=kind, DIM=dim, HII_DIM=dim // ratio, box_len=round(dim / ratio * rng.uniform(0.9, 2.0), 1),
                    scheme=rng.choice(["cic", "ngp"]), velocities=rng.random() < 0.5, z=round(rng.uniform(6.5, 16.0), 2))
    if kind == "power":
        D = _log_even(rng, 48, 300)
        return dict(kind=kind, D=D, box_len=round(D * rng.uniform(0.9, 2.0), 1), nbins=rng.randint(12, 100),
                    z=round(rng.uniform(6.5, 11.0), 2), x_HI=round(rng.uniform(0.1, 0.95), 3),
                    dimensional=rng.random() < 0.3)
    # the sides the network takes whole: its third level works on D/4, a multiple of 16
    D = rng.choice([64, 64, 128, 128, 192])
    batch = rng.randint(1, {64: 32, 128: 8, 192: 2}[D] // (1 if kind == "infer" else 2))
    if kind == "infer":
        return dict(kind=kind, D=D, batch=batch)
    return dict(kind=kind, D=D, batch=batch, lr=round(10.0 ** rng.uniform(-4.0, -2.7), 6))


# ------------------------------------------------------------------ inputs

def _modes(D, box_len, device=DEV):
    """|k| of the r2c half spectrum of a D^3 box, in 64 bits."""
    n = torch.fft.fftfreq(D, 1.0 / D, dtype=torch.float64, device=device)
    c = torch.arange(D // 2 + 1, dtype=torch.float64, device=device)
    m2 = (n * n)[:, None, None] + (n * n)[None, :, None] + (c * c)[None, None, :]
    return (2.0 * math.pi / box_len) * torch.sqrt(m2)


def _shape(k, D, box_len):
    """k^-2.5 exp(-(k/k_nyq)^2), 0 at k = 0: the benchmark's spectrum up to its amplitude."""
    return torch.where(k > 0, k.clamp_min(1e-30) ** -2.5 * torch.exp(-(k * box_len / (math.pi * D)) ** 2), 0.0)


def _field(D, box_len, gen, sigma=0.6):
    """A Gaussian random density box of the benchmark's spectrum and per-cell sigma."""
    x = torch.randn((D, D, D), generator=gen, device=DEV)
    f = torch.fft.rfftn(x)
    del x
    f *= torch.sqrt(_shape(_modes(D, box_len), D, box_len)).float()
    d = torch.fft.irfftn(f, s=(D, D, D))
    return (d * (sigma / d.double().std().float())).contiguous()


def _nonlinear(d, growth):
    """A mass-moved density at growth D(z) stands in as the lognormal map of the linear one."""
    g = d * growth
    return (torch.exp(g - 0.5 * g.double().var().float()) - 1.0).contiguous()


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _barrier(zeta, z, mean):
    """deltac = 1.686/D(z), and sigma_min^2 with zeta erfc(deltac/sqrt(2 sigma_min^2)) = mean: the
    mean collapsed fraction times the efficiency, near the ionized fraction."""
    deltac = 1.686 / _growth(z)
    y = torch.tensor(1.0 - mean / zeta, dtype=torch.float64)
    return deltac, 0.5 * (deltac / float(torch.erfinv(y))) ** 2


def _batch_specs(case):
    """Parameters of the boxes of a batch: like the package's manifest, partly ionized."""
    rng = random.Random(int(case["pick"]))
    out = []
    for i in range(case["nbox"]):
        D = (case["d0"], case["d1"], case["d2"])[i % GROUPS if i < GROUPS else rng.randrange(GROUPS)]
        zeta, z, mean = rng.uniform(10.0, 60.0), rng.choice([7.0, 8.0, 9.0, 10.0]), rng.uniform(0.2, 0.8)
        deltac, smin2 = _barrier(zeta, z, mean)
        out.append({"D": D, "box_len": case["cell"] * D, "zeta": zeta, "deltac": deltac, "sigma_min2": smin2, "z": z})
    return out


def _displacements(d, box_len, ratio):
    """The three displacement boxes of a density box, on every ratio-th cell."""
    D = d.shape[0]
    f = torch.fft.rfftn(d)
    n = torch.fft.fftfreq(D, 1.0 / D, device=DEV)
    c = torch.arange(D // 2 + 1, dtype=torch.float32, device=DEV)
    ax = (n[:, None, None], n[None, :, None], c[None, None, :])
    # only modes the coarse grid resolves, and no Nyquist modes
    k2 = ax[0] ** 2 + ax[1] ** 2 + ax[2] ** 2
    f *= torch.where((k2 > 0) & (k2 < (0.5 * D / ratio) ** 2), 1.0 / k2.clamp_min(1.0), 0.0)
    out = []
    for a in ax:
        v = torch.fft.irfftn(f * (1j * a), s=(D, D, D)) * (box_len / (2.0 * math.pi))
        out.append(v[::ratio, ::ratio, ::ratio].contiguous())
    return tuple(out)


_PARAMS = {}


def _params():
    """The trained surrogate weights that ship with the package."""
    if not _PARAMS:
        s = _mod("surrogate")
        _PARAMS.update(s.UNet3D.load_file(s.WEIGHTS)[0])
    return _PARAMS


def _surrogate_inputs(case, seed):
    D, B = case["D"], case["batch"]
    g = _gen(seed)
    delta = torch.stack([_field(D, D * 1.5625, g) for _ in range(B)])
    cond = torch.rand((B, 2), generator=g, device=DEV) * 2.0 - 1.0
    return delta, cond


def _target(delta):
    """An ionized field: 1 where the smoothed density is high, else a partial value."""
    B, D = delta.shape[:2]
    out = []
    for b in range(B):
        f = torch.fft.rfftn(delta[b])
        k = _modes(D, float(D)).float()
        s = torch.fft.irfftn(f * torch.exp(-0.5 * (2.0 * k) ** 2), s=(D, D, D))
        s = s / s.std()
        out.append(torch.where(s > 0.2, 1.0, 0.3 * torch.sigmoid(2.0 * s)))
    return torch.stack(out).contiguous()


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "bubbles":
        s["fb"] = _mod("Programs.find_HII_bubbles")
        d = _field(case["D"], case["box_len"], _gen(seed))
        s["delta"] = d if case["linear"] else _nonlinear(d, _growth(case["z"]))
        s["deltac"], s["smin2"] = _barrier(case["zeta"], case["z"], case["mean"])
    elif kind == "batch":
        specs = _batch_specs(case)
        g = _gen(seed)
        s["deltas"] = []
        for b in specs:
            d = _field(b["D"], b["box_len"], g)
            s["deltas"].append(d if case["linear"] else _nonlinear(d, _growth(b["z"])))
        # buffers, tables and the captured graph are kept by such a program
        s["bb"] = _mod("Programs.find_HII_bubbles_batched").BatchedBubbles(
            specs, fil=case["filter"], LE=case["linear"], stream=torch.cuda.Stream())
    elif kind == "initialize":
        s["init"] = _mod("Programs.initialize")
        s["seed"] = int(seed) & 0x7FFFFFFF
    elif kind == "perturb":
        s["pf"] = _mod("Programs.perturb_field")
        s["delta"] = _field(case["DIM"], case["box_len"], _gen(seed))
        s["v"] = _displacements(s["delta"], case["box_len"], case["DIM"] // case["HII_DIM"])
    elif kind == "power":
        s["dt"] = _mod("Programs.delta_T")
        d = _field(case["D"], case["box_len"], _gen(seed))
        s["delta"] = _nonlinear(d, _growth(case["z"]))
        # neutral outside the densest cells, a few per cent ionized there
        cut = float(torch.quantile(d.flatten()[:: max(1, d.numel() // 1000003)], case["x_HI"]))
        s["xH"] = torch.where(d > cut, 0.0, 1.0 - 0.1 * torch.sigmoid(d)).contiguous()
        s["edges"] = s["dt"].log_edges(case["box_len"], case["D"], case["nbins"])
    elif kind in ("infer", "train"):
        U = _mod("surrogate").UNet3D
        s["delta"], s["cond"] = _surrogate_inputs(case, seed)
        s["model"] = U(D=case["D"], batch=case["batch"], params=_params())
        if kind == "train":
            s["target"] = _target(s["delta"])
            # a run under way: the moments of earlier steps
            m = s["model"]
            g = _gen(int(seed) + 1)
            m.m.copy_(1e-4 * torch.randn(m.nparams, generator=g, device=DEV))
            m.v.copy_(1e-6 * (0.5 + torch.rand(m.nparams, generator=g, device=DEV)))
            m.step_count = 200
    else:
        raise ValueError(f"unknown kind {kind!r}")
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "bubbles":
        return s["fb"].conv_bubbles(s["delta"], {"BoxSize": c["box_len"], "HIIdim": c["D"]}, fil=c["filter"],
                                    update=c["update"], LE=c["linear"], quiet=True, deltac=s["deltac"],
                                    sigma_min2=s["smin2"], zeta=c["zeta"])
    if kind == "batch":
        s["bb"].set_deltas(s["deltas"])
        s["bb"].run()
        return [s["bb"].ionized(i) for i in range(c["nbox"])]
    if kind == "initialize":
        return s["init"].init(DIM=c["DIM"], HII_DIM=c["HII_DIM"], BOX_LEN=c["box_len"], seed=s["seed"],
                              pspec=c["pspec"], save=False)
    if kind == "perturb":
        out = {"density": s["pf"].evolve_zeldovich(c["z"], s["delta"], v=s["v"], growth=_growth(c["z"]),
                                                   growth_init=D_INIT, box_len=c["box_len"], scheme=c["scheme"],
                                                   save=False)}
        if c["velocities"]:
            out["v"] = s["pf"].velocities_at(c["z"], s["delta"], HII_DIM=c["HII_DIM"], box_len=c["box_len"],
                                             ddt_over_d=1.0)
        return out
    if kind == "power":
        dT, total = s["dt"].brightness_temperature(s["xH"], s["delta"], c["z"])
        K, k_ave, ps, n = s["dt"].power_spectrum(dT, c["box_len"], s["edges"], field_sum=total,
                                                 dimensional=c["dimensional"])
        return {"dT": dT, "sum": total, "k": k_ave, "ps": ps, "counts": n}
    m = s["model"]
    if kind == "infer":
        return m.forward(s["delta"], s["cond"], keep=False)
    prob = m.forward(s["delta"], s["cond"])
    loss = m.backward(s["target"])
    m.step(c["lr"])
    return {"prob": prob, "loss": loss, "grad": m.grad, "weights": m.flat}


# ------------------------------------------------------------------ bytes and operations

def _radii(D, box_len):
    cell, R, out = box_len / D, R_MAX, []
    while True:
        final = R / R_FACTOR <= L_FACTOR * cell or R / R_FACTOR <= R_MIN
        R32 = float(np.float32(R))
        out.append(R32)
        if final:
            return out
        R = R32 / R_FACTOR


def _fft_flops(D):
    return 2.5 * D ** 3 * math.log2(D ** 3)  # one real transform


def _layers(D):
    h, q = D // 2, D // 4
    return [(D, 1, 16), (D, 16, 16), (h, 16, 32), (h, 32, 32), (q, 32, 64), (q, 64, 64), (h, 64, 32), (h, 32, 32),
            (D, 32, 16), (D, 16, 16)]


def work(case):
    kind = case["kind"]
    if kind in ("bubbles", "batch"):
        boxes = [(case["D"], case["box_len"])] if kind == "bubbles" else \
            [(b["D"], b["box_len"]) for b in _batch_specs(case)]
        nbytes = flops = 0
        for D, L in boxes:
            nbytes += 8 * D ** 3
            flops += _fft_flops(D) + len(_radii(D, L)) * (_fft_flops(D) + (12 if case["linear"] else 40) * D ** 3)
        return {"bytes": nbytes, "flops": flops}
    if kind == "initialize":
        D, d = case["DIM"], case["HII_DIM"]
        return {"bytes": 8 * D * D * (D // 2 + 1) + 4 * D ** 3 + 16 * d ** 3,
                "flops": _fft_flops(D) + 4 * _fft_flops(d) + 60 * D ** 3}
    if kind == "perturb":
        D, d = case["DIM"], case["HII_DIM"]
        w = {"bytes": 4 * D ** 3 + 16 * d ** 3, "flops": (60 if case["scheme"] == "cic" else 20) * D ** 3}
        if case["velocities"]:
            w["bytes"] += 4 * D ** 3 + 12 * d ** 3
            w["flops"] += _fft_flops(D) + 3 * _fft_flops(d) + 30 * d ** 3
        return w
    if kind == "power":
        D = case["D"]
        return {"bytes": 16 * D ** 3, "flops": _fft_flops(D) + 15 * D ** 3}
    D, B = case["D"], case["batch"]
    macs = sum(27 * ci * co * s ** 3 for s, ci, co in _layers(D)) + 64 * 32 * (D // 2) ** 3 + 33 * 16 * D ** 3
    nbytes = 8 * B * D ** 3
    if kind == "infer":
        return {"bytes": nbytes, "flops": 2 * B * macs}
    return {"bytes": nbytes + 4 * B * D ** 3 + 28 * 336000, "flops": 6 * B * macs}


# ------------------------------------------------------------------ the same in 64 bits

def _erfc(x):
    return torch.special.erfc(x)


def _sigma2(R, k, weight, shape_sum_inv):
    y = k * R
    w = torch.where(y < 1e-2, 1.0 - y * y / 10.0, 3.0 * (torch.sin(y) - y * torch.cos(y)) / y.clamp_min(1e-9) ** 3)
    return float((weight * w * w).sum() * shape_sum_inv)


def _ball(seeds, R2):
    """Cells closer than sqrt(R2) to a seed, inside the box."""
    o = int(math.isqrt(int(R2)))
    if float(o * o) >= R2:
        o -= 1
    far = 1 << 28
    d = torch.where(seeds, 0, far).to(torch.int32)
    n = d.shape[0]
    for axis in range(3):
        best = d.clone()
        for s in range(1, min(o, n - 1) + 1):
            a, b = d.narrow(axis, 0, n - s), d.narrow(axis, s, n - s)
            lo, hi = best.narrow(axis, 0, n - s), best.narrow(axis, s, n - s)
            torch.minimum(lo, b + s * s, out=lo)
            torch.minimum(hi, a + s * s, out=hi)
        d = best
    return d.double() < R2


def _exact_bubbles(delta, D, L, linear, fil, update, zeta, deltac, smin2):
    N = D ** 3
    k = _modes(D, L)
    wgt = torch.full((D // 2 + 1,), 2.0, dtype=torch.float64, device=DEV)
    wgt[0] = wgt[-1] = 1.0
    weight = _shape(k, D, L) * wgt
    inv = 0.36 / float(weight.sum())
    deltac = float(np.float32(deltac))
    growth_inv = 1.0 if linear else float(np.float32(deltac / 1.686))
    f = torch.fft.rfftn(delta.double()) * growth_inv
    fc_mean = float(np.float32(math.erfc(deltac / math.sqrt(2.0 * smin2))))
    ion = torch.zeros((D, D, D), dtype=torch.float64, device=DEV)
    radii = _radii(D, L)
    for i, R in enumerate(radii):
        denom = math.sqrt(2.0 * (smin2 - _sigma2(R, k, weight, inv)))
        kR = k * R
        w = torch.ones_like(k)
        if fil == 0:
            x = kR.clamp_min(1e-4)
            w = torch.where(kR > 1e-4, 3.0 * (torch.sin(x) / x ** 3 - torch.cos(x) / x ** 2), w)
        if fil <= 1:
            kR = kR * 0.413566994
            w = torch.where(kR > 1.0, 0.0, w)
        w = w * torch.exp(-0.5 * (kR * 0.643) ** 2)
        s = torch.fft.irfftn(f * w, s=(D, D, D))
        fc = _erfc((deltac - s) / denom)
        if not linear:
            fc = fc * (fc_mean / (fc.sum() / N))
        hit = fc * zeta >= 1.0
        if i == len(radii) - 1:
            return torch.where((ion == 1.0) | hit, 1.0, fc * zeta)
        ion[_ball(hit, float(np.float32(R) * np.float32(R))) if update else hit] = 1.0


def _philox(ctr_lo, ctr_hi, key):
    """Philox4x32-10 (Salmon et al., SC'11) on int64 tensors of 32-bit words; two of the four results."""
    M = 0xFFFFFFFF

    def mul(a, x):  # high and low words of a 32 x 32 product, in pieces that fit 63 bits
        p = (a & 0xFFFF) * x
        q = (a >> 16) * x + (p >> 16)
        return (q >> 16) & M, ((q & 0xFFFF) << 16 | (p & 0xFFFF)) & M

    x0, x1, x2, x3 = ctr_lo, ctr_hi, torch.zeros_like(ctr_lo), torch.zeros_like(ctr_lo)
    k0, k1 = key, 0
    for r in range(10):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & M, (k1 + 0xBB67AE85) & M
        h0, l0 = mul(0xD2511F53, x0)
        h1, l1 = mul(0xCD9E8D57, x2)
        x0, x1, x2, x3 = h1 ^ x1 ^ k0, l1, h0 ^ x3 ^ k1, l0
    return x0, x1


def _exact_spectrum(D, L, seed):
    """The c2r-ready Hermitian half spectrum of the power-law random field."""
    H, V = D // 2 + 1, L ** 3
    wgt = torch.full((H,), 2.0, dtype=torch.float64, device=DEV)
    wgt[0] = wgt[-1] = 1.0
    amp = 0.36 * V / float((_shape(_modes(D, L), D, L) * wgt).sum())
    out = torch.empty((D, D, H), dtype=torch.complex128, device=DEV)
    b = torch.arange(D, device=DEV)[:, None]
    c = torch.arange(H, device=DEV)[None, :]
    n = lambda i: torch.where(i > D // 2, i - D, i).double()  # noqa: E731
    edge = (c == 0) | (c == D // 2)
    for a in range(D):
        ma, mb = (D - a) % D, (D - b) % D
        mirror = edge & ((ma * D + mb) < (a * D + b))
        selfconj = edge & (mb == b) & (ma == a)
        rep = torch.where(mirror, ma * D + mb, a * D + b) * H + c
        u0, u1 = _philox(rep & 0xFFFFFFFF, rep >> 32, int(seed))
        ua, ub = ((u0 >> 8).double() + 0.5) * 2.0 ** -24, ((u1 >> 8).double() + 0.5) * 2.0 ** -24
        r = torch.sqrt(-2.0 * torch.log(ua))
        na = float(a - D if a > D // 2 else a)
        k = (2.0 * math.pi / L) * torch.sqrt(na * na + n(b) ** 2 + c.double() ** 2)
        A = torch.sqrt(amp / V * _shape(k, D, L))
        re, im = r * torch.cos(2.0 * math.pi * ub), r * torch.sin(2.0 * math.pi * ub)
        h = A * math.sqrt(0.5)
        out[a] = torch.complex(torch.where(selfconj, A * re, h * re),
                               torch.where(selfconj, 0.0, torch.where(mirror, -h * im, h * im)))
    return out


def _exact_fields(spec, D, d, L, smoothed):
    """Smoothed box (where asked for) and displacement boxes of a c2r-ready half spectrum, every D/d-th cell."""
    R = float(np.float32(float(np.float32(L_FACTOR) * np.float32(L)) / d))
    kR = _modes(D, L) * R
    x = kR.clamp_min(1e-4)
    w = torch.where(kR > 1e-4, 3.0 * (torch.sin(x) / x ** 3 - torch.cos(x) / x ** 2), 1.0)
    del x
    kR *= 0.413566994
    w = torch.where(kR > 1.0, 0.0, w * torch.exp(-0.5 * (kR * 0.643) ** 2))
    del kR
    f = spec * w
    del w
    q = D // d
    inv = lambda g: (torch.fft.irfftn(g, s=(D, D, D), norm="forward")[::q, ::q, ::q]).contiguous()  # noqa: E731
    sm = inv(f) if smoothed else None
    dk = 2.0 * math.pi / L
    n = torch.fft.fftfreq(D, 1.0 / D, dtype=torch.float64, device=DEV)
    n[D // 2] = D // 2
    c = torch.arange(D // 2 + 1, dtype=torch.float64, device=DEV)
    ax = (n[:, None, None], n[None, :, None], c[None, None, :])
    k2 = (ax[0] ** 2 + ax[1] ** 2 + ax[2] ** 2) * dk
    k2[0, 0, 0] = 1.0
    vs = [inv(f * (1j * torch.where(a == D // 2, 0.0, a) / k2)) for a in ax]
    return sm, vs


def _exact_move(delta, v, D, d, L, growth, scheme):
    ratio = D // d
    s = float(np.float32(np.float32(np.float32(growth) - np.float32(D_INIT)) / np.float32(L)))
    gi = float(np.float32(D_INIT))
    acc = torch.zeros(d ** 3, dtype=torch.float64, device=DEV)
    grid = (torch.arange(D, dtype=torch.float64, device=DEV) + 0.5) / D
    cell = torch.arange(D, device=DEV) // ratio
    for i0 in range(0, D, 32):
        i1 = min(D, i0 + 32)
        ii = cell[i0:i1]
        pos = []
        for a, x in enumerate(v):
            g = (grid[i0:i1][:, None, None], grid[None, :, None], grid[None, None, :])[a]
            pos.append((g + x.double()[ii][:, cell][:, :, cell] * s) * d)
        m = 1.0 + gi * delta[i0:i1].double()
        if scheme == "ngp":
            p = [torch.floor(x).long() % d for x in pos]
            acc.index_add_(0, ((p[0] * d + p[1]) * d + p[2]).flatten(), m.flatten())
            continue
        lo = [torch.floor(x - 0.5) for x in pos]
        t = [x - 0.5 - y for x, y in zip(pos, lo)]
        for corner in range(8):
            idx, w = 0, m
            for a in range(3):
                o = corner >> a & 1
                idx = idx * d + (lo[a].long() + o) % d
                w = w * (t[a] if o else 1.0 - t[a])
            acc.index_add_(0, idx.flatten(), w.flatten())
    return (acc / ratio ** 3 - 1.0).reshape(d, d, d)


def _exact_power(s, c):
    D, L, z = c["D"], c["box_len"], c["z"]
    h, ob, om = 0.673, 0.0487, 0.315
    tb = 27 * (ob * h * h / 0.023) * math.sqrt((0.15 / om / h / h) * (1 + z) / 10.0)
    dT = tb * s["xH"].double() * (1.0 + s["delta"].double())
    total = dT.sum()
    V, N = L ** 3, D ** 3
    x = (dT / (total / N) - 1.0) * (V / N)
    if c["dimensional"]:
        x = x * (total / N)
    p = torch.fft.rfftn(x).abs() ** 2
    k = _modes(D, L)
    wgt = torch.full((D // 2 + 1,), 2.0, dtype=torch.float64, device=DEV)
    wgt[0] = wgt[-1] = 1.0
    wgt = wgt.expand_as(k).flatten()
    edges = torch.as_tensor(np.asarray(s["edges"], dtype=np.float64), device=DEV)
    # the bin of a mode from its integer |n|^2, as k differs by rounding alone between modes of one shell
    m2 = torch.round((k * L / (2.0 * math.pi)) ** 2).long().flatten()
    shell = (2.0 * math.pi / L) * torch.sqrt(torch.arange(3 * (D // 2) ** 2 + 1, dtype=torch.float64, device=DEV))
    bins = torch.searchsorted(edges, shell)
    bins[0] = len(edges)
    b = bins[m2]
    nb = len(edges) + 1
    add = lambda w: torch.zeros(nb, dtype=torch.float64, device=DEV).index_add_(0, b, w)[:-1]  # noqa: E731
    n = add(wgt)
    kk = k.flatten()
    ps = add(wgt * kk ** 3 * p.flatten() / (2.0 * math.pi ** 2 * V)) / n.clamp_min(1)
    return {"dT": dT, "sum": total.reshape(1), "k": add(wgt * kk) / n.clamp_min(1), "ps": ps, "counts": None}


def _rows(x, w):
    """x @ w over the last axis of a tall x, some rows at a time."""
    flat = x.reshape(-1, x.shape[-1])
    return torch.cat([r @ w for r in flat.split(1 << 19)]).reshape(*x.shape[:-1], w.shape[1])


class _Conv(torch.autograd.Function):
    """Periodic 3^3 convolution, channels last: x (B,D,D,D,ci), w (co,27,ci)."""

    @staticmethod
    def forward(ctx, x, w):
        ctx.save_for_backward(x, w)
        y = 0
        for t in range(27):
            y = y + _rows(torch.roll(x, (1 - t // 9, 1 - t // 3 % 3, 1 - t % 3), (1, 2, 3)), w[:, t].T)
        return y

    @staticmethod
    def backward(ctx, g):
        x, w = ctx.saved_tensors
        gx, gw = torch.zeros_like(x), torch.zeros_like(w)
        rows = x.reshape(-1, x.shape[-1]).split(1 << 19)
        for t in range(27):
            back = torch.roll(g, (t // 9 - 1, t // 3 % 3 - 1, t % 3 - 1), (1, 2, 3))
            gx += _rows(back, w[:, t])
            for u, v in zip(back.reshape(-1, w.shape[0]).split(1 << 19), rows):
                gw[:, t] += u.T @ v
        return gx, gw


def _exact_net(p, delta, cond):
    """Logits of the surrogate, channels last."""
    B, D = delta.shape[:2]
    x = torch.cat([(delta / 0.6).unsqueeze(-1), cond[:, None, None, None, :].expand(B, D, D, D, 2)], -1)

    def conv(x, n):
        return torch.relu(_Conv.apply(x, p[n + ".w"]) + p[n + ".b"])

    def pool(x):
        b, s, c = x.shape[0], x.shape[1] // 2, x.shape[-1]
        return x.reshape(b, s, 2, s, 2, s, 2, c).mean((2, 4, 6))

    def up(x, n):
        w = p[n + ".w"]  # (co, 8, ci)
        b, s, co = x.shape[0], x.shape[1], w.shape[0]
        y = _rows(x, w.reshape(-1, w.shape[-1]).T).reshape(b, s, s, s, co, 2, 2, 2)
        return y.permute(0, 1, 5, 2, 6, 3, 7, 4).reshape(b, 2 * s, 2 * s, 2 * s, co) + p[n + ".b"]

    e1 = conv(conv(x, "in"), "e1")
    e2 = conv(conv(pool(e1), "e2a"), "e2b")
    b2 = conv(conv(pool(e2), "b1"), "b2")
    d2 = conv(conv(torch.cat([e2, up(b2, "up2")], -1), "d2a"), "d2b")
    d1 = conv(conv(torch.cat([e1, up(d2, "up1")], -1), "d1a"), "d1b")
    return (d1 * p["head.w"]).sum(-1) + p["head.b"]


def exact(case, seed):
    kind = case["kind"]
    if kind == "initialize":
        if case["pspec"] != "powerlaw":
            return None  # a fitted table of the package's own
        D, d, L = case["DIM"], case["HII_DIM"], case["box_len"]
        spec = _exact_spectrum(D, L, int(seed) & 0x7FFFFFFF)
        sm, vs = _exact_fields(spec, D, d, L, True)
        return {"spec": spec, "deltax": torch.fft.irfftn(spec, s=(D, D, D), norm="forward"), "smoothed": sm,
                "v": tuple(vs)}
    if kind == "infer" or kind == "train":
        delta, cond = _surrogate_inputs(case, seed)
        names = [n for n, _ in _mod("surrogate").param_shapes()]
        p = {n: torch.as_tensor(np.asarray(_params()[n], np.float32), device=DEV).double() for n in names}
        if kind == "infer":
            return torch.cat([torch.sigmoid(_exact_net(p, delta[b:b + 1].double(), cond[b:b + 1].double()))
                              for b in range(case["batch"])])
        for v in p.values():
            v.requires_grad_(True)
        prob, loss, grad = [], 0.0, 0.0
        target = _target(delta).double()
        for b in range(case["batch"]):
            logit = _exact_net(p, delta[b:b + 1].double(), cond[b:b + 1].double())
            part = torch.nn.functional.binary_cross_entropy_with_logits(logit, target[b:b + 1]) / case["batch"]
            grad = grad + torch.cat([g.flatten() for g in torch.autograd.grad(part, list(p.values()))])
            loss = loss + part.detach()
            prob.append(torch.sigmoid(logit.detach()))
        # AdamW from the state that prepare() set up, step 201
        g = _gen(int(seed) + 1)
        m = (1e-4 * torch.randn(grad.numel(), generator=g, device=DEV)).double()
        v = (1e-6 * (0.5 + torch.rand(grad.numel(), generator=g, device=DEV))).double()
        m, v = 0.9 * m + 0.1 * grad, 0.999 * v + 0.001 * grad * grad
        mh, vh = m / (1.0 - 0.9 ** 201), v / (1.0 - 0.999 ** 201)
        w = torch.cat([x.detach().flatten() for x in p.values()])
        w = w - case["lr"] * (mh / (vh.sqrt() + 1e-8) + 1e-4 * w)
        return {"prob": torch.cat(prob), "loss": loss.reshape(1), "grad": grad, "weights": w}
    if kind == "batch":
        specs, g, out = _batch_specs(case), _gen(seed), []
        for b in specs:
            d = _field(b["D"], b["box_len"], g)
            d = d if case["linear"] else _nonlinear(d, _growth(b["z"]))
            out.append(_exact_bubbles(d, b["D"], b["box_len"], case["linear"], case["filter"], 0, b["zeta"],
                                      b["deltac"], b["sigma_min2"]))
        return out
    c = case
    if kind == "bubbles":
        d = _field(c["D"], c["box_len"], _gen(seed))
        d = d if c["linear"] else _nonlinear(d, _growth(c["z"]))
        deltac, smin2 = _barrier(c["zeta"], c["z"], c["mean"])
        return _exact_bubbles(d, c["D"], c["box_len"], c["linear"], c["filter"], c["update"], c["zeta"], deltac, smin2)
    if kind == "perturb":
        D, d, L = c["DIM"], c["HII_DIM"], c["box_len"]
        delta = _field(D, L, _gen(seed))
        v = _displacements(delta, L, D // d)
        out = {"density": _exact_move(delta, v, D, d, L, _growth(c["z"]), c["scheme"])}
        if c["velocities"]:
            out["v"] = tuple(_exact_fields(torch.fft.rfftn(delta.double(), norm="forward"), D, d, L, False)[1])
        return out
    return _exact_power(prepare(case, seed), c)
