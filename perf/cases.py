"""The work that is timed: reconstructions and their read-outs, as a user's program runs them.

Each case is one call sequence through the public Python API on device-resident float32 arrays: a reconstruction
(run! + reconstructed_positions), a batch of reconstructions, repeated read-outs of a finished reconstruction, the sky
conversions at both ends of a survey pipeline, or a training step of the warm-start network.  Catalogs are lognormal
tracers with power-law spectra, drawn on the GPU from the seed; `exact` restates each path in plain torch in 64 bits.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "baorec.jl_amd", "python"))

import baorec_hip as bh  # noqa: E402

NET = os.path.join(ROOT, "baorec.jl_amd", "weights", "unet_lc128.bin")
F64 = torch.float64
DEV = "cuda"


# ------------------------------------------------------------------------------------------------------- the cases

def listed():
    return [
        # a quick look at a small simulation box: one short call, where launches and latency count
        dict(name="box64", kind="box", nx=64, ny=64, nz=64, n=20011, recon="iterative", los="z", mas="cic", graph=False),
        # the ordinary periodic box of a mock: 128^3 cells, 1M tracers, plane-parallel
        dict(name="box128", kind="box", nx=128, ny=128, nz=128, n=1000000, recon="iterative", los="z", mas="cic", graph=False),
        # the same mock in a loop of many realisations that reuses its arrays, replayed as a HIP graph
        dict(name="box128_graph", kind="box", nx=128, ny=128, nz=128, n=1000000, recon="iterative", los="z", mas="cic", graph=True),
        # a thin survey sample: ragged catalog sizes, TSC assignment, radial line of sight
        dict(name="cone256_tsc", kind="cone", nx=256, ny=256, nz=256, n=300007, nr=3000017, recon="iterative", mas="tsc", warm="none"),
        # the survey-sized lightcone, iterative FFT reconstruction
        dict(name="cone512", kind="cone", nx=512, ny=512, nz=512, n=2000000, nr=20000000, recon="iterative", mas="cic", warm="none"),
        # a small box through the multigrid solver to a tolerance: many launches on small grids
        dict(name="mg_box128", kind="box", nx=128, ny=128, nz=128, n=200003, recon="rbgs", los="local", mas="cic", warm="none"),
        # the multigrid solver as the reference schedules it (full multigrid, damped Jacobi), at its default size
        dict(name="mg_box512_fmg", kind="box", nx=512, ny=512, nz=512, n=1000000, recon="fmg", los="local", mas="cic", warm="none"),
        # the survey-sized lightcone through the multigrid solver to a tolerance, from the learned start
        dict(name="mg_cone512_learned", kind="cone", nx=512, ny=512, nz=512, n=2000000, nr=20000000, recon="rbgs", mas="cic", warm="learned"),
        # a batch of mocks of uneven sizes
        dict(name="batch16", kind="batch", nx=256, ny=256, nz=256, ncat=16, nmin=200000, nmax=5000000),
        # the randoms of a finished survey reconstruction, read out twice (with and without the RSD term)
        dict(name="readout512", kind="readout", nx=512, ny=512, nz=512, n=2000000, nr=20000000),
        # both ends of a survey pipeline: sky to Cartesian and back
        dict(name="sky22m", kind="sky", n=22000001),
        # one optimiser step of a fresh warm-start network on a batch of four 128^3 pairs, as it is trained
        dict(name="train128", kind="train", nx=128, ny=128, nz=128, batch=4),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["box", "box", "box", "cone", "cone", "mg", "mg", "batch", "readout", "sky", "train"])
    if kind == "box":   # cubic or not (x longest); the box has the grid's proportions
        sides = [rng.choice([32, 64, 128, 256, 512]) for _ in range(3)] if rng.random() < 0.5 else [rng.choice([32, 64, 128, 256, 512])] * 3
        return dict(kind="box", nx=max(sides), ny=sides[1], nz=sides[2], n=_log_int(rng, 5000, 5000000) | 1, recon="iterative",
                    los=rng.choice(["z", "local"]), mas=rng.choice(["cic", "cic", "tsc"]), graph=rng.random() < 0.25)
    if kind == "cone":
        side = rng.choice([64, 128, 256, 512])
        n = _log_int(rng, 20000, 1900000) | 1
        return dict(kind="cone", nx=side, ny=side, nz=side, n=n, nr=n * rng.randint(4, 10) + 1, recon="iterative",
                    mas=rng.choice(["cic", "cic", "tsc"]), warm="none")
    if kind == "mg":
        side = rng.choice([64, 128, 256])
        n = _log_int(rng, 20000, 1900000) | 1
        recon = rng.choice(["fmg", "rbgs", "rbgs"])
        warm = rng.choice(["none", "spectral", "refined", "learned"]) if recon == "rbgs" else "none"
        if rng.random() < 0.5:
            return dict(kind="cone", nx=side, ny=side, nz=side, n=n, nr=n * rng.randint(4, 10) + 1, recon=recon, mas="cic", warm=warm)
        return dict(kind="box", nx=side, ny=side, nz=side, n=n, recon=recon, los=rng.choice(["z", "local"]), mas="cic", warm=warm)
    if kind == "batch":
        side = rng.choice([64, 128, 256])
        return dict(kind="batch", nx=side, ny=side, nz=side, ncat=rng.randint(2, 12), nmin=_log_int(rng, 10000, 200000), nmax=_log_int(rng, 300000, 4000000))
    if kind == "readout":
        side = rng.choice([128, 256])
        n = _log_int(rng, 50000, 1000000) | 1
        return dict(kind="readout", nx=side, ny=side, nz=side, n=n, nr=n * rng.randint(4, 10) + 1)
    if kind == "sky":
        return dict(kind="sky", n=_log_int(rng, 1000, 22000000) | 1)
    side = rng.choice([32, 64, 64, 128])
    return dict(kind="train", nx=side, ny=side, nz=side, batch=rng.randint(1, 3))


# ---------------------------------------------------------------------------------------------------------- inputs

BOX = dict(bias=2.0, f=0.8, smoothing_radius=15.0)     # periodic boxes
CONE = dict(bias=2.2, f=0.75, smoothing_radius=15.0)   # lightcones
PAD = 180.0                                            # about a tenth of the shell's extent
SHELL = (1000.0, 1800.0)
TRAIN_LR = 1e-3                                        # the first learning rate of the training schedule


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _box_side(case):
    """Mpc/h per axis: 1000 along the longest side, cubic cells."""
    top = max(case["nx"], case["ny"], case["nz"])
    return [1000.0 * case[a] / top for a in ("nx", "ny", "nz")]


def _overdensity(g, mesh, side, slope):
    """A lognormal density of unit mean on mesh^3 cells of a box of `side`, P(k) = 2e4 (k / 0.1)^slope for 0.005 < k < 0.5."""
    k = 2 * math.pi * torch.fft.fftfreq(mesh, side / mesh, device=DEV)
    kr = 2 * math.pi * torch.fft.rfftfreq(mesh, side / mesh, device=DEV)
    kk = torch.sqrt(k[:, None, None] ** 2 + k[None, :, None] ** 2 + kr[None, None, :] ** 2)
    pk = torch.where((kk >= 0.005) & (kk <= 0.5), 2e4 * (kk.clamp(min=1e-6) / 0.1) ** slope, torch.zeros_like(kk))
    white = torch.randn(mesh, mesh, mesh, generator=g, device=DEV)
    field = torch.fft.irfftn(torch.fft.rfftn(white) * torch.sqrt(pk / (side / mesh) ** 3), s=(mesh,) * 3)
    var = field.var()
    field = field / torch.sqrt(var.clamp(min=1.0))
    return torch.exp(field - 0.5 * var.clamp(max=1.0))


def _sample(g, density, n, sides):
    """n points of a density on mesh^3 cells over [0, sides): three float32 arrays."""
    mesh = density.shape[0]
    cdf = torch.cumsum(density.reshape(-1).to(F64), 0)
    cell = torch.searchsorted(cdf, torch.rand(n, generator=g, device=DEV, dtype=F64) * cdf[-1]).clamp(max=mesh ** 3 - 1)
    index = (cell % mesh, cell // mesh % mesh, cell // mesh ** 2)
    out = []
    for a, side in zip(index, sides):
        p = (a + torch.rand(n, generator=g, device=DEV, dtype=F64)) * (side / mesh)
        out.append(p.clamp(max=side * (1 - 1e-7)).to(torch.float32))
    return out


def _box_catalog(g, case, n, slope=-1.5):
    sides = _box_side(case)
    return _sample(g, _overdensity(g, 128, max(sides), slope), n, sides) + [torch.ones(n, device=DEV)]


def _cone_catalog(g, n):
    """Tracers of the octant shell with n(r) ~ r^-0.5."""
    mesh, side = 128, SHELL[1]
    c = (torch.arange(mesh, device=DEV) + 0.5) * (side / mesh)
    r = torch.sqrt(c[:, None, None] ** 2 + c[None, :, None] ** 2 + c[None, None, :] ** 2)
    sel = torch.where((r >= SHELL[0]) & (r <= SHELL[1]), r ** -0.5, torch.zeros_like(r))
    return _sample(g, _overdensity(g, mesh, side, -1.5) * sel, n, [side] * 3) + [torch.ones(n, device=DEV)]


def _cone_randoms(g, n):
    u, ra, sd = (torch.rand(n, generator=g, device=DEV, dtype=F64) for _ in range(3))
    r = (SHELL[0] ** 2.5 + u * (SHELL[1] ** 2.5 - SHELL[0] ** 2.5)) ** 0.4
    ra = ra * (math.pi / 2)
    cd = torch.sqrt(1 - sd * sd)
    return [(r * cd * torch.cos(ra)).to(torch.float32), (r * cd * torch.sin(ra)).to(torch.float32), (r * sd).to(torch.float32),
            torch.ones(n, device=DEV)]


def _batch_sizes(case):
    """Sizes spread over [nmin, nmax] in the logarithm, in no order, odd."""
    return [int(case["nmin"] * (case["nmax"] / case["nmin"]) ** ((0.5 + 0.618034 * c) % 1)) | 1 for c in range(case["ncat"])]


def _catalogs(case, seed):
    """(data, randoms or None) of a box, cone or readout case."""
    g = _gen(seed)
    if case["kind"] == "box":
        return _box_catalog(g, case, case["n"]), None
    return _cone_catalog(g, case["n"]), _cone_randoms(g, case["nr"])


def _batch_catalogs(case, seed):
    g = _gen(seed)
    sizes = _batch_sizes(case)
    cats = [_box_catalog(g, case, n, slope=-1.0 - ((0.5 + 0.618034 * c) % 1)) for c, n in enumerate(sizes)]
    return [torch.cat([c[k] for c in cats]) for k in range(4)], np.cumsum([0] + sizes)


def _sky_catalog(case, seed):
    g, n = _gen(seed), case["n"]
    ra = 100.0 + 160.0 * torch.rand(n, generator=g, device=DEV)
    dec = -10.0 + 70.0 * torch.rand(n, generator=g, device=DEV)
    red = 0.4 + 0.7 * torch.rand(n, generator=g, device=DEV)
    return ra, dec, red


def _train_geometry(case):
    """The lightcone's box."""
    return dict(grid=(case["nx"], case["ny"], case["nz"]), size=[SHELL[1] + PAD] * 3, min=[-PAD / 2] * 3)


def _train_pairs(case, seed):
    """Right-hand sides (smoothed overdensities of the shell) and their converged potentials, float32."""
    geo, g = _train_geometry(case), _gen(seed)
    x = _centres(geo)
    r = torch.sqrt(x[0] ** 2 + x[1] ** 2 + x[2] ** 2)
    shell = ((r >= SHELL[0]) & (r <= SHELL[1]) & (torch.minimum(torch.minimum(x[0], x[1]), x[2]) > 0)).to(F64)
    f, phi = [], []
    for _ in range(case["batch"]):
        d = _overdensity(g, geo["grid"][0], geo["size"][0], -1.5).to(F64)
        d = (_smooth((d - d.mean()) * shell, geo, 15.0) / CONE["bias"]).to(torch.float32)
        f.append(d)
        phi.append(_solve(d.to(F64), geo, CONE["f"] / CONE["bias"], None).to(torch.float32))
    return torch.stack(f), torch.stack(phi)


def _network_start(seed):
    """Parameters of a fresh network: He-normal kernels, zero biases, a small head."""
    g, parts = _gen(seed + 1), []
    for c1, c2, co, _, _, _ in LAYERS:
        parts += [torch.randn(27 * (c1 + c2) * co, generator=g, device=DEV) * math.sqrt(2 / (27 * (c1 + c2))), torch.zeros(co, device=DEV)]
    return torch.cat(parts + [0.01 * torch.randn(16, generator=g, device=DEV), torch.zeros(1, device=DEV)])


# ----------------------------------------------------------------------------------------------------- the library

def _recon(case, **more):
    if case["kind"] in ("cone", "readout"):
        more = dict(CONE, box_pad=PAD, los=None, mas=case.get("mas", "cic"), **more)
    else:
        more = dict(BOX, box_size=_box_side(case), box_min=[0.0] * 3, los=None if case.get("los", "z") == "local" else (0.0, 0.0, 1.0),
                    mas=case.get("mas", "cic"), **more)
    if case.get("recon", "iterative") == "iterative":
        return bh.IterativeRecon(**more)
    if case["recon"] == "fmg":
        return bh.MultigridRecon(schedule="reference", **more)
    if case["warm"] == "learned":
        bh.warmstart_load(NET)
    return bh.MultigridRecon(schedule="rbgs", tolerance=1e-6, warm_start=case["warm"], **more)


def prepare(case, seed):
    kind = case["kind"]
    state = dict(case=case)
    if kind in ("box", "cone"):
        data, randoms = _catalogs(case, seed)
        state.update(data=data, randoms=randoms or [], recon=_recon(case), grid=(case["nx"], case["ny"], case["nz"]))
        if case.get("graph"):
            state["out"] = [torch.empty_like(a) for a in data[:3]]
    elif kind == "batch":
        data, offsets = _batch_catalogs(case, seed)
        state.update(data=data, offsets=offsets, recon=_recon(case), grid=(case["nx"], case["ny"], case["nz"]))
    elif kind == "readout":
        data, randoms = _catalogs(case, seed)
        torch.cuda.synchronize()
        recon = _recon(case, ctx=bh.Context(0))   # keeps its own result
        bh.run_(recon, (case["nx"], case["ny"], case["nz"]), *data, *randoms, copy=False)
        state.update(randoms=randoms, recon=recon)
    elif kind == "sky":
        state.update(sky=_sky_catalog(case, seed), cosmology=bh.Cosmology.desi())
    else:
        f, phi = _train_pairs(case, seed)
        geo = _train_geometry(case)
        ctx = bh.Context(0)   # its own network
        bh.warmstart_init(h_train=geo["size"][0] / geo["grid"][0], ctx=ctx)
        bh.warmstart_set_params(_network_start(seed).cpu().numpy(), ctx=ctx)
        state.update(f=f, phi=phi, recon=bh.MultigridRecon(**CONE, box_size=geo["size"], box_min=geo["min"], los=None, schedule="rbgs", ctx=ctx))
    torch.cuda.synchronize()   # the library works on a stream of its own
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("box", "cone"):
        recon, data = state["recon"], state["data"]
        if case.get("graph"):
            return bh.run_positions_graph(recon, state["grid"], *data, out=state["out"])
        bh.run_(recon, state["grid"], *data, *state["randoms"], copy=False)
        return bh.reconstructed_positions(recon, *data[:3], field="sum")
    if kind == "batch":
        return bh.run_batch(state["recon"], state["grid"], *state["data"], state["offsets"])
    if kind == "readout":
        recon, xyz = state["recon"], state["randoms"][:3]
        return bh.reconstructed_positions(recon, *xyz, field="sum"), bh.reconstructed_positions(recon, *xyz, field="disp")
    if kind == "sky":
        xyz = bh.sky_to_cartesian(*state["sky"], state["cosmology"])
        return xyz, bh.cartesian_to_sky(*xyz, state["cosmology"])
    loss = bh.warmstart_step(state["recon"], state["f"], state["phi"], lr=TRAIN_LR)
    return {"loss": loss, "gradients": bh.warmstart_params("grads", ctx=state["recon"].ctx)}


def work(case):
    kind = case["kind"]
    if kind == "sky":
        return {"bytes": 48.0 * case["n"], "flops": 200.0 * case["n"]}
    cells = float(case["nx"] * case["ny"] * case["nz"])
    fft = 2.5 * cells * math.log2(cells)   # one real transform
    if kind == "train":
        # three products per convolution (forward, input and weight gradient), 27 taps
        macs = sum(27.0 * (c1 + c2) * co / 8 ** level for c1, c2, co, level, _, _ in LAYERS)
        return {"bytes": case["batch"] * cells * 8.0 + 4.0 * N_PARAMS, "flops": case["batch"] * cells * 6.0 * macs}
    if kind == "readout":
        return {"bytes": 12.0 * cells + 36.0 * case["nr"], "flops": 120.0 * case["nr"]}
    if kind == "batch":
        n = float(sum(_batch_sizes(case)))
        return {"bytes": 28.0 * n, "flops": case["ncat"] * fft * (2 + 3 * 2 + 3) + 200.0 * n}
    n, nr = case["n"], case.get("nr", 0)
    flops = fft * (4 if nr else 2) + 3 * fft + 150.0 * n + 50.0 * nr
    if case["recon"] == "iterative":
        flops += 3 * fft * (7 if case.get("los", "local") == "local" else 2)
    elif case["recon"] == "fmg":
        flops += cells * 8 / 7 * 6 * (10 * 55 + 60) * 8 / 7
    else:   # about four V-cycles of four sweeps and a residual
        flops += cells * 8 / 7 * 4 * (4 * 55 + 120)
    return {"bytes": 16.0 * (n + nr) + 12.0 * n, "flops": flops}


# ------------------------------------------------------------------------------------- the same in 64 bits, in torch

def _geometry(case, randoms=None):
    grid = (case["nx"], case["ny"], case["nz"])
    if randoms is None:
        return dict(grid=grid, size=_box_side(case), min=[0.0] * 3)
    lo = [float(a.min()) - PAD / 2 for a in randoms[:3]]
    side = max(float(a.max()) + PAD / 2 - b for a, b in zip(randoms[:3], lo))
    return dict(grid=grid, size=[side] * 3, min=lo)


def _axis(v, axis):
    """A vector along x (0), y (1) or z (2) of a (z, y, x) grid."""
    return v.reshape([-1 if 2 - k == axis else 1 for k in range(3)])


def _centres(geo):
    return [_axis(b + (torch.arange(n, device=DEV, dtype=F64) + 0.5) * (s / n), a)
            for a, (n, s, b) in enumerate(zip(geo["grid"], geo["size"], geo["min"]))]


def _waves(geo):
    out = []
    for a, (n, s) in enumerate(zip(geo["grid"], geo["size"])):
        i = torch.arange(n // 2 + 1 if a == 0 else n, device=DEV, dtype=F64)
        out.append(_axis((i if a == 0 else torch.where(i < (n + 1) // 2, i, i - n)) * (2 * math.pi / s), a))
    return out


def _inverse(spec, nx):
    """C2R whose self-conjugate x bins lose their imaginary parts."""
    s = torch.fft.ifftn(spec, dim=(0, 1))
    s[..., 0].imag.zero_()
    s[..., -1].imag.zero_()
    return torch.fft.irfft(s, n=nx, dim=2)


def _smooth(field, geo, radius):
    spec = torch.fft.rfftn(field)
    for k in _waves(geo):
        spec *= torch.exp(-0.5 * radius ** 2 * k * k)
    return _inverse(spec, geo["grid"][0])


def _deposit(cat, geo, mas):
    nx, ny, nz = geo["grid"]
    rho = torch.zeros(nx * ny * nz, device=DEV, dtype=F64)
    for part in zip(*(a.split(1 << 22) for a in cat)):
        idx, wts = [], []
        for p, n, s, b in zip(part[:3], geo["grid"], geo["size"], geo["min"]):
            u = (p.to(F64) - b) * (n / s)
            c = torch.floor(u + 0.5) if mas == "tsc" else torch.floor(u)
            d = u - c
            w = [0.5 * (0.5 - d) ** 2, 0.75 - d * d, 0.5 * (0.5 + d) ** 2] if mas == "tsc" else [1 - d, d]
            first = c.long() - (1 if mas == "tsc" else 0)
            idx.append([(first + k) % n for k in range(len(w))])
            wts.append(w)
        for k, wz in enumerate(wts[2]):
            for j, wy in enumerate(wts[1]):
                wzy = part[3].to(F64) * wz * wy
                row = nx * (idx[1][j] + ny * idx[2][k])
                for i, wx in enumerate(wts[0]):
                    rho.index_add_(0, row + idx[0][i], wzy * wx)
    return rho.reshape(nz, ny, nx)


def _delta(case, data, randoms, geo):
    """The smoothed overdensity over the bias."""
    par = CONE if randoms else BOX
    rho = _deposit(data, geo, case.get("mas", "cic"))
    total = rho.sum()
    rho = _smooth(rho, geo, par["smoothing_radius"])
    if not randoms:
        return (rho / (total / rho.numel()) - 1) / par["bias"]
    ran = _deposit(randoms, geo, case.get("mas", "cic"))
    total_r = ran.sum()
    ran = _smooth(ran, geo, par["smoothing_radius"])
    alpha = total / total_r
    keep = ran > float(np.float32(0.01)) * total_r / randoms[0].numel()
    return torch.where(keep, (rho - alpha * ran) / (par["bias"] * alpha * torch.where(keep, ran, torch.ones_like(ran))), torch.zeros_like(rho))


def _inverse_k2(geo):
    k = _waves(geo)
    k2 = k[0] ** 2 + k[1] ** 2 + k[2] ** 2
    return k, torch.where(k2 > 0, 1 / k2.clamp(min=1e-300), torch.zeros_like(k2))


def _iterate(ds, geo, beta, los):
    """Three iterations of the redshift-space correction."""
    k, ik2 = _inverse_k2(geo)
    x = _centres(geo)
    dr = ds
    for it in range(3):
        b = beta / (1 + beta) if it == 0 else beta
        spec = torch.fft.rfftn(dr) * ik2
        if los is not None:
            m = sum(k[a] ** 2 * los[a] for a in range(3))
            dr = ds - b * _inverse(spec * m, geo["grid"][0])
            continue
        s = torch.zeros_like(ds)
        for i in range(3):
            for j in range(i, 3):
                s += (2 if i != j else 1) * x[i] * x[j] * _inverse(spec * (k[i] * k[j]), geo["grid"][0])
        dr = ds - b * s / (x[0] ** 2 + x[1] ** 2 + x[2] ** 2)
    return dr


class _Operator:
    """The anisotropic 19-point operator on one grid: A v = diag v - near(v)."""

    def __init__(self, geo, beta, los):
        self.cell = [s / n for s, n in zip(geo["size"], geo["grid"])]
        x = _centres(geo) if los is None else [torch.tensor(float(v), device=DEV, dtype=F64) for v in los]
        self.p = [a / c for a, c in zip(x, self.cell)]
        s2 = sum((c * p) ** 2 for c, p in zip(self.cell, self.p))
        self.g = torch.where(s2 > 0, beta / s2.clamp(min=1e-300), torch.zeros_like(s2))
        self.local = los is None
        self.diag = sum(2 * (1 / c ** 2 + self.g * p * p) for c, p in zip(self.cell, self.p))

    def near(self, v):
        out, dim, cross, first = torch.zeros_like(v), [2, 1, 0], torch.zeros_like(v), torch.zeros_like(v)
        for a in range(3):
            up, dn = torch.roll(v, -1, dim[a]), torch.roll(v, 1, dim[a])
            out += (1 / self.cell[a] ** 2 + self.g * self.p[a] ** 2) * (up + dn)
            first += self.p[a] * (up - dn)
            for b in range(a + 1, 3):
                cross += self.p[a] * self.p[b] * (torch.roll(up, -1, dim[b]) + torch.roll(dn, 1, dim[b])
                                                  - torch.roll(dn, -1, dim[b]) - torch.roll(up, 1, dim[b]))
        out += 0.5 * self.g * cross
        return out + self.g * first if self.local else out

    def residual(self, v, f):
        return f - (self.diag * v - self.near(v))

    def jacobi(self, v, f, n):
        for _ in range(n):
            v = 0.6 * v + 0.4 * (f + self.near(v)) / self.diag
        return v


def _centre_los(geo, los):
    if los is not None:
        return list(los)
    c = [b + 0.5 * s for b, s in zip(geo["min"], geo["size"])]
    r = math.sqrt(sum(v * v for v in c))
    return [v / r for v in c]


def _spectral(f, geo, beta, los):
    """The operator with the line of sight fixed at the box centre's, inverted exactly (zero mean)."""
    d = _centre_los(geo, los)
    cell = [s / n for s, n in zip(geo["size"], geo["grid"])]
    p = [a / c for a, c in zip(d, cell)]
    g = beta / sum(v * v for v in d)
    t = [k * c for k, c in zip(_waves(geo), cell)]
    sym = sum((1 / cell[a] ** 2 + g * p[a] ** 2) * (2 - 2 * torch.cos(t[a])) for a in range(3))
    for a in range(3):
        for b in range(a + 1, 3):
            sym = sym + 2 * g * p[a] * p[b] * torch.sin(t[a]) * torch.sin(t[b])
    return _inverse(torch.where(sym > 0, torch.fft.rfftn(f) / torch.where(sym > 0, sym, torch.ones_like(sym)), 0), geo["grid"][0])


def _solve(f, geo, beta, los):
    """A phi = f minus the constant that makes it solvable, by Richardson steps with the fixed-LOS inverse."""
    phi = _spectral(f - f.mean(), geo, beta, los)
    if los is not None:
        return phi
    op, shift, norm = _Operator(geo, beta, los), f.mean(), torch.linalg.norm(f - f.mean())
    for _ in range(60):
        r = op.residual(phi, f - shift)
        shift = shift + r.mean()
        r = r - r.mean()
        if float(torch.linalg.norm(r) / norm) < 1e-10:
            break
        phi = phi + _spectral(r, geo, beta, los)
    return phi


def _restrict(v):
    for dim in range(3):
        even, odd = v.unfold(dim, 2, 2).unbind(-1)
        v = (even + 2 * odd + torch.roll(even, -1, dim)) / 4
    return v


def _prolong(v):
    for dim in range(3):
        v = torch.stack([(torch.roll(v, 1, dim) + v) / 2, v], dim + 1).flatten(dim, dim + 1)
    return v


def _full_multigrid(f, geo, beta, los):
    """The fixed schedule: six V-cycles per level, 5 + 5 damped Jacobi sweeps."""
    ops, fs = [_Operator(geo, beta, los)], [f]
    while min(geo["grid"]) > 4 and all(n % 2 == 0 for n in geo["grid"]):
        geo = dict(geo, grid=tuple(n // 2 for n in geo["grid"]))
        ops.append(_Operator(geo, beta, los))
        fs.append(_restrict(fs[-1]))

    def vcycle(level, v, rhs):
        v = ops[level].jacobi(v, rhs, 5)
        if level + 1 < len(ops):
            r = _restrict(ops[level].residual(v, rhs))
            v = v + _prolong(vcycle(level + 1, torch.zeros_like(r), r))
        return ops[level].jacobi(v, rhs, 5)

    v = torch.zeros_like(fs[-1])
    for level in range(len(ops) - 1, -1, -1):
        if level + 1 < len(ops):
            v = _prolong(v)
        for _ in range(6):
            v = vcycle(level, v, fs[level])
    return v


def _displacement(field, geo, potential):
    k, ik2 = _inverse_k2(geo)
    spec = 1j * torch.fft.rfftn(field)
    if not potential:
        spec = spec * ik2
    return [_inverse(spec * a, geo["grid"][0]) for a in k]


def _positions(xyz, psi, geo, f, los, rsd):
    """Shifted positions by trilinear read-out, in pieces."""
    nx, ny, nz = geo["grid"]
    out = []
    for part in zip(*(a.split(1 << 22) for a in xyz)):
        pos = [a.to(F64) for a in part]
        ax = []
        for p, n, s, b in zip(pos, geo["grid"], geo["size"], geo["min"]):
            u = (p - b) * (n / s)
            i = torch.floor(u)
            ax.append(((i.long() % n, 1 - (u - i)), ((i.long() + 1) % n, u - i)))
        shift = [torch.zeros_like(pos[0]) for _ in range(3)]
        for iz, wz in ax[2]:
            for iy, wy in ax[1]:
                for ix, wx in ax[0]:
                    cell, w = ix + nx * (iy + ny * iz), wx * wy * wz
                    for a in range(3):
                        shift[a] += w * psi[a].reshape(-1)[cell]
        if rsd:
            r = torch.sqrt(pos[0] ** 2 + pos[1] ** 2 + pos[2] ** 2)
            line = [a / r for a in pos] if los is None else list(los)
            dot = f * sum(s * l for s, l in zip(shift, line))
            shift = [s + dot * l for s, l in zip(shift, line)]
        out.append([p - s for p, s in zip(pos, shift)])
    return tuple(torch.cat([o[a] for o in out]) for a in range(3))


def _reconstructed_displacement(case, data, randoms):
    geo = _geometry(case, randoms)
    par = CONE if randoms else BOX
    beta = par["f"] / par["bias"]
    los = None if randoms or case.get("los", "z") == "local" else (0.0, 0.0, 1.0)
    ds = _delta(case, data, randoms, geo)
    recon = case.get("recon", "iterative")
    if recon == "iterative":
        field = _iterate(ds, geo, beta, los)
    else:
        field = (_full_multigrid if recon == "fmg" else _solve)(ds, geo, beta, los)
    return _displacement(field, geo, recon != "iterative"), geo, par["f"], los


def _distance_table(c):
    """Knots and comoving distances (Mpc) of a flat-table cosmology, 8-point Gauss-Legendre per interval."""
    f = np.float32
    h2 = f(f(c.h) * f(c.h))
    rho = f(3 * 100 ** 2 / (8 * np.pi * 6.67408e-11) * 6.582119514e-16 ** 3 * (1 / (1e-3 * 3.085677581491367e22)) ** 2
            * (1 / 1.782661907e-36) * (299792.458e3) ** 3)
    og = f((np.pi ** 2 / 15) * (2.725 * 8.6173303e-5) ** 4 / float(rho) * (float(f(c.T_cmb)) / 2.725) ** 4 / float(h2))
    on = f(float(f(c.Neff)) * (7 / 8 * (4 / 11) ** (4 / 3)) * float(og))
    ob, oc, ok = f(f(c.omega_b) / h2), f(f(c.omega_c) / h2), f(c.Omega_k0)
    ol = float(f(f(f(f(f(f(1) - ok) - ob) - oc) - on) - og))
    zk = np.linspace(c.z_tab_min, c.z_tab_max, c.z_tab_num)
    x, w = np.polynomial.legendre.leggauss(8)
    half = 0.5 * (zk[1:] - zk[:-1])
    z1 = 1 + 0.5 * (zk[1:] + zk[:-1])[:, None] + half[:, None] * x
    e = np.sqrt((float(on) + float(og)) * z1 ** 4 + (float(ob) + float(oc)) * z1 ** 3 + float(ok) * z1 ** 2 + ol)
    step = 299792.458 * half * ((1 / (float(f(f(c.h) * f(100))) * e)) @ w)
    return zk, np.concatenate([[0.0], np.cumsum(step)])


def _interp(x, xk, yk):
    xk, yk = torch.from_numpy(xk).to(DEV), torch.from_numpy(yk).to(DEV)
    i = (torch.searchsorted(xk, x, right=True) - 1).clamp(0, len(xk) - 2)
    return yk[i] + (x - xk[i]) / (xk[i + 1] - xk[i]) * (yk[i + 1] - yk[i])


def _exact_sky(case, seed):
    c = bh.Cosmology.desi()
    zk, rk = _distance_table(c)
    ra, dec, red = (a.to(F64) for a in _sky_catalog(case, seed))
    h = float(np.float32(c.h))
    r = _interp(red, zk, rk) * h
    a, d = torch.deg2rad(ra), torch.deg2rad(dec)
    xyz = (r * torch.cos(d) * torch.cos(a), r * torch.cos(d) * torch.sin(a), r * torch.sin(d))
    lon = torch.rad2deg(torch.atan2(xyz[1], xyz[0]))
    lat = torch.rad2deg(torch.atan2(xyz[2], torch.sqrt(xyz[0] ** 2 + xyz[1] ** 2)))
    dist = torch.sqrt(xyz[0] ** 2 + xyz[1] ** 2 + xyz[2] ** 2) / h
    return xyz, (torch.fmod(lon - 360, 360), lat, _interp(dist, rk, zk))


# the network: (skip or only input's channels, upsampled input's channels, output channels, level, inputs)
LAYERS = [
    (8, 0, 16, 0, -1, None), (16, 0, 16, 0, 0, None), (16, 0, 32, 1, -2, None), (32, 0, 32, 1, 2, None),
    (32, 0, 64, 2, -3, None), (64, 0, 64, 2, 4, None), (64, 0, 128, 3, -4, None), (128, 0, 128, 3, 6, None),
    (64, 128, 64, 2, 5, 7), (64, 0, 64, 2, 8, None), (32, 64, 32, 1, 3, 9), (32, 0, 32, 1, 10, None),
    (16, 32, 16, 0, 1, 11), (16, 0, 16, 0, 12, None),
]
N_PARAMS = sum(27 * (c1 + c2) * co + co for c1, c2, co, _, _, _ in LAYERS) + 17
TAPS = [(t // 9 - 1, t // 3 % 3 - 1, t % 3 - 1) for t in range(27)]


def _up(x):
    for dim in range(3):
        x = x.repeat_interleave(2, dim)
    return x


def _down(x):
    z, y, xx, c = x.shape
    return x.reshape(z // 2, 2, y // 2, 2, xx // 2, 2, c).sum(dim=(1, 3, 5))


def _network(par, feat, target, scale):
    """Loss and parameter gradients of one item ((z, y, x, channel) arrays)."""
    W, B, at, o = [], [], [], 0
    for c1, c2, co, _, _, _ in LAYERS:
        at.append(o)
        W.append(par[o:o + 27 * (c1 + c2) * co].reshape(27, c1 + c2, co))
        o += 27 * (c1 + c2) * co
        B.append(par[o:o + co])
        o += co
    head, bias = par[o:o + 16], par[o + 16]
    act, pooled = [], {}

    def inp(i):
        src = LAYERS[i][4]
        a = feat if src == -1 else pooled[-src - 2] if src < -1 else act[src]
        return a if LAYERS[i][5] is None else torch.cat([a, _up(act[LAYERS[i][5]])], -1)

    for i in range(len(LAYERS)):
        x = inp(i)
        out = sum(torch.roll(x, (-dz, -dy, -dx), (0, 1, 2)) @ W[i][t] for t, (dz, dy, dx) in enumerate(TAPS)) + B[i]
        act.append(torch.relu(out))
        if i in (1, 3, 5):
            pooled[(i - 1) // 2] = _down(act[i]) / 8
    diff = act[-1] @ head + bias - target
    loss, g = 0.0, torch.zeros_like(diff)
    for dim in range(3):
        d = torch.roll(diff, -1, dim) - diff
        loss = loss + (d * d).sum() * scale
        g += 2 * scale * (torch.roll(d, 1, dim) - d)
    grad = torch.zeros_like(par)
    grad[o:o + 16] = (act[-1] * g[..., None]).sum(dim=(0, 1, 2))
    grad[o + 16] = g.sum()
    up = {len(LAYERS) - 1: g[..., None] * head}
    for i in range(len(LAYERS) - 1, -1, -1):
        c1, c2, co, _, src, coarse = LAYERS[i]
        g, x = up.pop(i) * (act[i] > 0), inp(i)
        flat, dx = g.reshape(-1, co), torch.zeros_like(x)
        for t, (dz, dy, dxx) in enumerate(TAPS):
            n = at[i] + t * (c1 + c2) * co
            grad[n:n + (c1 + c2) * co] = (torch.roll(x, (-dz, -dy, -dxx), (0, 1, 2)).reshape(-1, c1 + c2).T @ flat).reshape(-1)
            dx += torch.roll(g, (dz, dy, dxx), (0, 1, 2)) @ W[i][t].T
        n = at[i] + 27 * (c1 + c2) * co
        grad[n:n + co] = flat.sum(0)
        if coarse is not None:
            up[src], up[coarse] = dx[..., :c1], _down(dx[..., c1:])
        elif src < -1:
            skip = 2 * (-src - 2) + 1
            up[skip] = up[skip] + _up(dx) / 8
        elif src >= 0:
            up[src] = dx
    return loss, grad


def _exact_train(case, seed):
    geo, beta = _train_geometry(case), CONE["f"] / CONE["bias"]
    fs, phis = _train_pairs(case, seed)
    par = _network_start(seed).to(F64)
    h = geo["size"][0] / geo["grid"][0]
    x, centre = _centres(geo), _centre_los(geo, None)
    r = torch.sqrt(x[0] ** 2 + x[1] ** 2 + x[2] ** 2)
    op = _Operator(geo, beta, None)
    loss, grad = 0.0, torch.zeros_like(par)
    for f, phi in zip(fs.to(F64), phis.to(F64)):
        s = torch.sqrt((f * f).mean())
        seed_phi = _spectral(f, geo, beta, None)
        res = op.residual(seed_phi, f)
        feat = torch.stack([f / s, seed_phi / (s * h * h), res / s, _spectral(res, geo, beta, None) / (s * h * h)]
                           + [(a / r - c).expand_as(f) for a, c in zip(x, centre)] + [(100 * h / r).expand_as(f)], -1)
        one, g = _network(par, feat, (phi - seed_phi) / (s * h * h), 1 / (3.0 * fs.numel()))
        loss, grad = loss + one, grad + g
    return {"loss": float(loss), "gradients": grad}


def exact(case, seed):
    kind = case["kind"]
    if kind == "sky":
        return _exact_sky(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "batch":
        (x, y, z, w), off = _batch_catalogs(case, seed)
        out = []
        for a, b in zip(off[:-1], off[1:]):
            cat = [v[a:b] for v in (x, y, z, w)]
            psi, geo, f, los = _reconstructed_displacement(case, cat, None)
            out.append(_positions(cat[:3], psi, geo, f, los, True))
        return tuple(torch.cat([o[k] for o in out]) for k in range(3))
    data, randoms = _catalogs(case, seed)
    psi, geo, f, los = _reconstructed_displacement(case, data, randoms)
    if kind == "readout":
        return tuple(_positions(randoms[:3], psi, geo, f, los, rsd) for rsd in (True, False))
    return _positions(data[:3], psi, geo, f, los, True)
