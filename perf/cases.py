"""Performance cases: the calls that reconstruction programs make through srf_amd's
public entry points, over the sizes they make them at.

Kinds of case, and what each stands for in use:

  project       Project / ProjectTof of one image along an event list that no plan was
                built for: one-shot simulations, line integrals, quality checks
  backproject   BackProject / BackProjectTof of event values into a fresh image, one-shot
  attenuation   AttenuationCorrect of a listmode: done once per scan, over all its events
  mlem          Mlem from listmode to image: plan construction, n_iter iterations, the
                image on the host; the ordinary whole call on a small scanner
  osem          one iteration (every subset) of an OsemEngine that a program built before
  autograd      forward and backward of the differentiable projector on a batch of images
                (the projector as a layer of a network that is being trained)
  sss           the single-scatter sinogram of a new emission estimate
  unet          the scatter surrogate's network on the features of N scans
  unet_train    gradients of one training batch of that network
  emap          the sensitivity image over all crystal pairs of a scanner
  psf           Richardson-Lucy deconvolution of a reconstructed image

Sizes are those of the benchmark and the tests where these have one (the 48 x 48 x 24
smoke grid, 64 x 64 x 32 MLEM, 256 x 256 x 128 TOF OSEM, 8 x 128 x 128 x 64 autograd, the
32 x 64 x 64 sinogram, the mCT's crystals on 200^3), and odd ones beside them.

exact() restates each path in 64-bit torch from its published formulas (the slab marcher of
srfnef/cc/siddon/siddon.cu.cc:12-656 and srfnef/cc/siddon_tof/siddon_tof.cu.cc:14-707, EM,
Klein-Nishina sums, convolutions) and shares no code with the package.
"""
import math
import os

import numpy as np
import torch

TOF_BIN = 3.66
TOF_SIGMA2 = 649.2          # 60 mm FWHM
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
WEIGHTS = os.path.join(ROOT, "srf_amd", "weights", "scatter_unet_128x128x64.npz")
WIDTHS = (16, 32, 64, 128)
MU_WATER = 0.0096
SSS_SPACING = 8.0
SSS_RADIUS, SSS_AXIAL, SSS_FOV = 424.0, 300.0, 256.0


def listed():
    return [
        # the smallest calls: a quick projection of a few thousand events, bound by launches
        _pr("project_small_tof", "project", 4096, (48, 48, 24), 2.0, True, 150.0, 80.0),
        # a whole OSEM subset projected without a plan (simulation of TOF data)
        _pr("project_tof_5e6", "project", 5_000_000, (256, 256, 128), 2.0, True),
        # the same direction back, ragged: a grid that no tile divides, fewer events
        _pr("backproject_tof_ragged", "backproject", 1_234_567, (181, 217, 91), 2.5, True),
        # attenuation factors of every event of a scan (7-column rows, non-TOF integrals)
        _pr("attenuation_3e6", "attenuation", 3_000_000, (200, 200, 109), 2.05, True),
        # the small-scanner MLEM of the configurations, listmode to image
        dict(_pr("mlem_1e6", "mlem", 1_000_000, (64, 64, 32), 3.4, False, 300.0, 110.0), n_iter=10),
        # two of the headline's subsets: TOF OSEM on 256 x 256 x 128, 5e6 events per subset
        dict(_pr("osem_tof_1e7", "osem", 10_000_000, (256, 256, 128), 2.0, True), n_sub=2),
        # the differentiable projector on 8 images
        dict(_pr("autograd_8x4e6", "autograd", 4_000_000, (128, 128, 64), 2.0, True, 300.0, 300.0), batch=8),
        # a full scatter estimate on the surrogate workload's grid
        {"name": "sss_128x128x64", "kind": "sss", "nx": 128, "ny": 128, "nz": 64, "voxel": 4.0, "n_rings": 32},
        # the surrogate network for the 32 scans of a batched reconstruction, and one training batch
        {"name": "unet_32", "kind": "unet", "samples": 32, "d": 32, "h": 64, "w": 64},
        {"name": "unet_train_4", "kind": "unet_train", "samples": 4, "d": 32, "h": 64, "w": 64},
        # the sensitivity image of an mCT-like scanner: 32448 crystals, 1.05e9 ordered pairs
        {"name": "emap_mct", "kind": "emap", "blocks": 48, "rings": 4, "by": 13, "bz": 13, "nx": 200, "nz": 200},
        # deconvolution on the mCT image grid
        {"name": "psf_200", "kind": "psf", "nx": 200, "ny": 200, "nz": 200, "voxel": 2.05, "n_iter": 10},
    ]


def _pr(name, kind, events, shape, voxel, tof, radius=424.0, axial=300.0):
    return {"name": name, "kind": kind, "events": events, "nx": shape[0], "ny": shape[1], "nz": shape[2],
            "voxel": voxel, "tof": tof, "radius": radius, "axial": axial}


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["project", "project", "backproject", "backproject", "attenuation", "mlem", "osem", "autograd",
                       "sss", "unet", "unet_train", "emap", "psf"])
    if kind in ("project", "backproject", "attenuation", "osem"):
        nx = rng.randint(48, 256)
        ny = nx if rng.random() < 0.5 else rng.randint(48, 256)
        c = {"kind": kind, "events": _log(rng, 4096, 5_000_000), "nx": nx, "ny": ny, "nz": rng.randint(24, 128),
             "voxel": rng.choice([2.0, 2.05, 2.5, 4.0]), "tof": rng.random() < 0.6, "radius": 424.0, "axial": 300.0}
        if kind == "attenuation":
            c["tof"] = True
        if kind == "osem":
            c["n_sub"] = rng.randint(1, 4)
            c["events"] = _log(rng, 100_000, 10_000_000)
        return c
    if kind == "mlem":
        return {"kind": kind, "events": _log(rng, 20_000, 2_000_000), "nx": rng.randint(40, 96),
                "ny": rng.randint(40, 96), "nz": rng.randint(16, 48), "voxel": 3.4, "tof": False, "radius": 300.0,
                "axial": 110.0, "n_iter": rng.randint(2, 10)}
    if kind == "autograd":
        return {"kind": kind, "events": _log(rng, 50_000, 4_000_000), "nx": rng.randint(48, 128),
                "ny": rng.randint(48, 128), "nz": rng.randint(24, 64), "voxel": 2.0, "tof": rng.random() < 0.6,
                "radius": 300.0, "axial": 300.0, "batch": rng.randint(1, 8)}
    if kind == "sss":
        return {"kind": kind, "nx": rng.randint(64, 128), "ny": rng.randint(64, 128), "nz": rng.randint(32, 64),
                "voxel": 4.0, "n_rings": rng.randint(1, 32)}
    if kind in ("unet", "unet_train"):
        return {"kind": kind, "samples": rng.randint(1, 32 if kind == "unet" else 4), "d": 8 * rng.randint(2, 4),
                "h": 8 * rng.randint(4, 8), "w": 8 * rng.randint(4, 8)}
    if kind == "emap":
        return {"kind": kind, "blocks": rng.randint(16, 48), "rings": rng.randint(1, 2), "by": rng.randint(4, 13),
                "bz": rng.randint(4, 9), "nx": rng.randint(64, 200), "nz": rng.randint(24, 100)}
    return {"kind": "psf", "nx": rng.randint(64, 200), "ny": rng.randint(64, 200), "nz": rng.randint(24, 200),
            "voxel": 2.05, "n_iter": rng.randint(2, 10)}


# ------------------------------------------------------------------ inputs --

def _dev():
    return torch.device("cuda", 0) if torch.cuda.is_available() else torch.device("cpu")


def _gen(seed, salt=0):
    return torch.Generator(device=_dev()).manual_seed(int(seed) * 1000 + salt)


def _rand(g, *shape, dtype=torch.float32):
    return torch.rand(shape, generator=g, device=_dev(), dtype=dtype)


def _shape(case):
    return [int(case["nx"]), int(case["ny"]), int(case["nz"])]


def _size(case):
    return [n * float(case["voxel"]) for n in _shape(case)]


def _smooth_field(g, shape, coarse):
    """Smooth positive random field of `shape` (batch, d, h, w) from noise on a coarse grid."""
    x = torch.rand((shape[0], 1) + tuple(max(2, n // coarse) for n in shape[1:]), generator=g, device=_dev())
    return torch.nn.functional.interpolate(x, size=shape[1:], mode="trilinear", align_corners=True)[:, 0]


def _body(shape, size, g):
    """Activity and mu-map of a water ellipsoid holding a few warmer ones, (nx, ny, nz) float32."""
    dev = _dev()
    ax = [torch.arange(n, device=dev, dtype=torch.float64) for n in shape]
    ax = [(a + 0.5) * (s / n) - s / 2 for a, n, s in zip(ax, shape, size)]

    def mask(c, r):
        q = [((a - float(ci)) / float(ri)) ** 2 for a, ci, ri in zip(ax, c, r)]
        return q[0][:, None, None] + q[1][None, :, None] + q[2][None, None, :] <= 1.0

    u = torch.rand(32, generator=g, device=dev, dtype=torch.float64).tolist()
    half = [s / 2 for s in size]
    r = [min(180.0, 0.9 * half[0]), min(120.0, 0.8 * half[1]), min(120.0, 0.95 * half[2])]
    body = mask((0, 0, 0), r)
    act, mu = body.to(torch.float32), body.to(torch.float32) * MU_WATER
    for k in range(4):
        c = [(2 * u[6 * k + i] - 1) * 0.5 * r[i] for i in range(3)]
        e = [(0.1 + 0.2 * u[6 * k + 3 + i]) * r[i] for i in range(3)]
        act[mask(c, e)] = 0.5 + 4.5 * u[6 * k]
    return act, mu, r


def _events(case, g, n):
    """n list-mode rows (6 or 7 columns): emission points in a body, random directions whose
    ends lie on the detector cylinder, TOF path difference with its noise; in random order."""
    dev, f = _dev(), torch.float64
    R, H = float(case["radius"]), float(case["axial"]) / 2
    half = [s / 2 for s in _size(case)]
    out = torch.empty((n, 7 if case["tof"] else 6), dtype=torch.float32, device=dev)
    axes = torch.tensor([min(180.0, 0.9 * half[0]), min(120.0, 0.8 * half[1]), min(0.9 * H, 0.95 * half[2])],
                        dtype=f, device=dev)
    for a in range(0, n, 1 << 22):
        m = min(1 << 22, n - a)
        v = torch.randn((m, 3), generator=g, device=dev, dtype=f)
        e = v / v.norm(dim=1, keepdim=True) * _rand(g, m, 1, dtype=f) ** (1.0 / 3.0) * axes
        phi = 2 * math.pi * _rand(g, m, dtype=f)
        c, s = torch.cos(phi), torch.sin(phi)
        b = e[:, 0] * c + e[:, 1] * s
        disc = torch.sqrt(b * b + R * R - e[:, 0] ** 2 - e[:, 1] ** 2)
        dp, dm = disc - b, disc + b                       # transaxial distances to the two ends
        lo = torch.maximum((-H - e[:, 2]) / dp, (e[:, 2] - H) / dm)
        hi = torch.minimum((H - e[:, 2]) / dp, (e[:, 2] + H) / dm)
        t = lo + (hi - lo) * _rand(g, m, dtype=f)         # axial slope: both ends inside the axial length
        rows = [e[:, 0] - dm * c, e[:, 1] - dm * s, e[:, 2] - dm * t, e[:, 0] + dp * c, e[:, 1] + dp * s,
                e[:, 2] + dp * t]
        if case["tof"]:
            noise = torch.randn(m, generator=g, device=dev, dtype=f) * (2 * math.sqrt(TOF_SIGMA2))
            rows.append((dp - dm) * torch.sqrt(1 + t * t) + noise)
        out[a:a + m] = torch.stack(rows, 1).to(torch.float32)
    return out


def _emap(case):
    """A smooth sensitivity image (nx, ny, nz), zero outside the transaxial field of view."""
    dev, n, s = _dev(), _shape(case), _size(case)
    ax = [((torch.arange(k, device=dev, dtype=torch.float64) + 0.5) / k - 0.5) * l for k, l in zip(n, s)]
    r2 = ax[0][:, None, None] ** 2 + ax[1][None, :, None] ** 2
    z = (1.0 - 0.8 * (ax[2].abs() / (s[2] / 2)))[None, None, :]
    e = (20.0 + r2 / 4.0e3) * z
    return torch.where(r2 <= (max(s[0], s[1]) / 2) ** 2, e, torch.zeros_like(e)).to(torch.float32).contiguous()


def _lists(case, seed):
    """(LORs, values, image) of the projector kinds."""
    g = _gen(seed, 1)
    n = int(case["events"])
    lors = _events(case, g, n)
    values = 1.0 + 9.0 * _rand(g, n)
    image, _, _ = _body(_shape(case), _size(case), g)
    image = (image + 0.05 * _rand(g, *_shape(case))).contiguous()
    return lors, values, image


def _perm(case, seed):
    return torch.randperm(int(case["events"]), generator=_gen(seed, 2), device=_dev())


def _images(case, seed):
    return (0.2 + _smooth_field(_gen(seed, 3), (int(case["batch"]),) + tuple(_shape(case)), 6)).contiguous()


def _sss_inputs(case, seed):
    g = _gen(seed, 4)
    act, mu, _ = _body(_shape(case), _size(case), g)
    em = act * (0.5 + _smooth_field(g, (1,) + tuple(_shape(case)), 8)[0])
    return em.contiguous(), mu.contiguous()


def _unet_inputs(case, seed):
    """Features (N V, 8) bf16 bits and targets (N V,) like a sinogram's line integrals."""
    N, dims = int(case["samples"]), (int(case["d"]), int(case["h"]), int(case["w"]))
    g = _gen(seed, 5)
    f = _smooth_field(g, (2 * N,) + dims, 6)
    e, m = 2.0 * f[:N], 4.0 * f[N:]
    a = torch.exp(-m)
    z = torch.zeros_like(e)
    x = torch.stack([e, a, e * a, 0.25 * m, z, z, z, z], -1).reshape(-1, 8).to(torch.bfloat16)
    t = (e * a * (0.8 + 0.4 * _smooth_field(g, (N,) + dims, 6))).reshape(-1).contiguous()
    return x.view(torch.int16).contiguous(), t, dims


def _psf_tables(case):
    """Patch weights (nx ny, 121) of a blur that widens with the radius, and the axial matrix."""
    nx, ny, nz = _shape(case)
    v = float(case["voxel"])
    x = ((np.arange(nx) + 0.5) - nx / 2) * v
    y = ((np.arange(ny) + 0.5) - ny / 2) * v
    r = np.sqrt(x[:, None] ** 2 + y[None, :] ** 2)
    sig = (1.8 + 0.006 * r).reshape(-1, 1, 1)
    o = np.arange(-5, 6)
    w = np.exp(-0.5 * v * v * (o[None, :, None] ** 2 + 1.2 * o[None, None, :] ** 2) / sig ** 2)
    ii = np.repeat(np.arange(nx), ny)[:, None, None] + o[None, :, None]
    jj = np.tile(np.arange(ny), nx)[:, None, None] + o[None, None, :]
    w = w * ((ii >= 0) & (ii < nx) & (jj >= 0) & (jj < ny))
    w = w / w.sum(axis=(1, 2), keepdims=True)
    w = np.where(w > 1e-6, w, 0.0).reshape(nx * ny, 121).astype(np.float32)
    k = np.arange(nz)
    kz = np.exp(-0.5 * ((k[:, None] - k[None, :]) * v) ** 2 / 2.2 ** 2)
    kz = kz / kz.sum(axis=0, keepdims=True)
    return w, np.where(kz > 1e-16, kz, 0.0).astype(np.float32)


def _psf_data(case, seed):
    g = _gen(seed, 6)
    act, _, _ = _body(_shape(case), _size(case), g)
    return (act + 0.05 + 0.1 * _rand(g, *_shape(case))).contiguous()


def _emap_scanner(case, seed):
    """Rings of blocks around the mCT's radius, the exact radius and axial pitch by the seed."""
    from srf_amd import scanner as S
    u = torch.rand(2, generator=torch.Generator().manual_seed(int(seed))).tolist()
    by, bz, radius = int(case["by"]), int(case["bz"]), 424.5 + 4.0 * u[0]
    width = 2 * math.pi * radius / int(case["blocks"])
    return S.PetEcatScanner(radius, radius + 20.0, int(case["rings"]), int(case["blocks"]), 0.0,
                            S.Block([20.0, 0.95 * width, 53.0 + u[1]], [1, by, bz]))


def _emap_config(case):
    from srf_amd.data import ImageConfig
    nx, nz = int(case["nx"]), int(case["nz"])
    return ImageConfig([nx, nx, nz], [0.0, 0.0, 0.0], [410.0, 410.0, 2.05 * nz])


# --------------------------------------------------------- prepare and run --

def prepare(case, seed):
    kind = case["kind"]
    st = {"case": dict(case)}
    if kind in ("project", "backproject", "attenuation", "mlem"):
        from srf_amd.data import Emap, Image, Listmode, Lors, Umap
        lors, values, image = _lists(case, seed)
        c0, size = [0.0, 0.0, 0.0], _size(case)
        st["lors"] = Lors(lors)
        st["listmode"] = Listmode(values, st["lors"])
        st["image"] = Image(image, c0, size)
        if kind == "attenuation":
            st["umap"] = Umap((image > 0.5).to(torch.float32) * MU_WATER, c0, size)
        if kind == "mlem":
            st["emap"] = Emap(_emap(case), c0, size)
    elif kind == "osem":
        from srf_amd.data import TofConfig
        from srf_amd.functions import OsemEngine
        lors, values, image = _lists(case, seed)
        tof = TofConfig(TOF_BIN, TOF_SIGMA2) if case["tof"] else None
        st["engine"] = OsemEngine(lors, values, _emap(case), _shape(case), [0.0, 0.0, 0.0] + _size(case),
                                  int(case["n_sub"]), _perm(case, seed), tof=tof, ratio_kind=1, eps=1e-5,
                                  zero_guard=1e8, tof_window=22.0 if case["tof"] else 0.0)
        st["x0"] = (image + 0.1).permute(2, 1, 0).contiguous()
    elif kind == "autograd":
        from srf_amd.autograd import Projector
        lors, values, _ = _lists(case, seed)
        st["images"], st["values"] = _images(case, seed), values
        st["projector"] = Projector(lors, _shape(case), [0.0, 0.0, 0.0], _size(case),
                                    tof=(TOF_BIN, TOF_SIGMA2) if case["tof"] else None)
    elif kind == "sss":
        from srf_amd.sss import SingleScatterSimulation, SssGeometry
        st["em"], st["mu"] = _sss_inputs(case, seed)
        st["sss"] = SingleScatterSimulation(SssGeometry(), _shape(case), [0.0, 0.0, 0.0], _size(case),
                                            rings=_rings(case))
    elif kind in ("unet", "unet_train"):
        from srf_amd.surrogate import UNet
        st["net"], _ = UNet.load(WEIGHTS)
        st["x"], st["t"], st["dims"] = _unet_inputs(case, seed)
    elif kind == "emap":
        st["scanner"], st["config"] = _emap_scanner(case, seed), _emap_config(case)
    elif kind == "psf":
        from srf_amd.psf import Deconvolute
        w, kz = _psf_tables(case)
        st["dec"] = Deconvolute(int(case["n_iter"]), None, None, None, w, kz)
        st["data"] = _psf_data(case, seed)
    return st


def _rings(case):
    n = int(case["n_rings"])
    return None if n == 32 else [(k * 32) // n for k in range(n)]


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "project":
        from srf_amd.data import TofConfig
        from srf_amd.functions import Project, ProjectTof
        op = ProjectTof("hip", TofConfig(TOF_BIN, TOF_SIGMA2)) if case["tof"] else Project("hip")
        return op(state["image"], state["lors"]).data
    if kind == "backproject":
        from srf_amd.data import TofConfig
        from srf_amd.functions import BackProject, BackProjectTof
        op = BackProjectTof("hip", TofConfig(TOF_BIN, TOF_SIGMA2)) if case["tof"] else BackProject("hip")
        return op(state["listmode"], state["image"]).data
    if kind == "attenuation":
        from srf_amd.corrections import AttenuationCorrect
        return AttenuationCorrect(state["umap"])(state["listmode"]).data
    if kind == "mlem":
        from srf_amd.functions import Mlem
        return Mlem(int(case["n_iter"]), state["emap"])(state["listmode"]).data
    if kind == "osem":
        eng = state["engine"]
        eng.x.copy_(state["x0"])
        eng.run(int(case["n_sub"]))
        return eng.x
    if kind == "autograd":
        x = state["images"].detach().requires_grad_(True)
        p = state["projector"](x)
        p.backward(state["values"].expand_as(p))
        return [p.detach(), x.grad]
    if kind == "sss":
        return state["sss"](state["em"], state["mu"])
    if kind == "unet":
        return state["net"].forward(state["x"], state["dims"], int(case["samples"]))
    if kind == "unet_train":
        net, N = state["net"], int(case["samples"])
        net.zero_grad()
        out = net.forward(state["x"], state["dims"], N)
        net.backward(net.loss_and_grad(out, state["t"], state["dims"], 1.0, N), state["dims"], N)
        return [out] + [l.gw for l in net.layers] + [l.gb for l in net.layers]
    if kind == "emap":
        from srf_amd.functions import crystal_pair_emap
        return crystal_pair_emap(state["scanner"], state["config"])
    return state["dec"].run(state["data"])


# -------------------------------------------------------------------- work --

def _march_work(n, case, tof, passes_lors=1):
    """One projection or backprojection of n events: LOR row, value, and the image once.  A ray
    crosses about 0.7 of the slabs of its dominant axis with 1.5 terms in each; a term is a
    multiply-add and its share (about 10 operations) of the slab's crossing fractions."""
    nx, ny, nz = int(case["nx"]), int(case.get("ny", case["nx"])), int(case["nz"])
    terms = n * 1.05 * max(nx, ny)
    return 4.0 * n * (6 + (1 if tof else 0) + 1) + 4.0 * nx * ny * nz, 12.0 * terms


def _unet_layers():
    L, c = [], 4
    for l, w in enumerate(WIDTHS):
        L += [(f"enc{l}a", l, 27, c, w), (f"enc{l}b", l, 27, w, w)]
        c = w
    for l in (2, 1, 0):
        L += [(f"dec{l}a", l, 27, WIDTHS[l + 1] + WIDTHS[l], WIDTHS[l]), (f"dec{l}b", l, 27, WIDTHS[l], WIDTHS[l])]
    return L + [("head", 0, 1, WIDTHS[0], 1)]


def work(case):
    kind = case["kind"]
    if kind in ("project", "backproject", "attenuation"):
        b, f = _march_work(int(case["events"]), case, case["tof"] and kind != "attenuation")
        return {"bytes": b + (8.0 * int(case["events"]) if kind == "attenuation" else 0.0), "flops": f}
    if kind in ("mlem", "osem"):
        n = int(case["events"])
        b, f = _march_work(n, case, case["tof"])
        it = 2 * int(case.get("n_iter", 1))
        nv = int(case["nx"]) * int(case["ny"]) * int(case["nz"])
        # with the TOF window about half of the TOF terms carry weight
        return {"bytes": it * (b + 8.0 * nv), "flops": it * f * (0.5 if case["tof"] else 1.0)}
    if kind == "autograd":
        b, f = _march_work(int(case["events"]), case, case["tof"])
        return {"bytes": 2 * int(case["batch"]) * b, "flops": 2 * int(case["batch"]) * f}
    if kind == "sss":
        step = SSS_SPACING
        pts = 0.25 * math.prod(s / step for s in _size(case))
        det = 128 * int(case["n_rings"])
        bins = 4096 * int(case["n_rings"])
        # line integrals from every detector to every point, then two pair terms per bin and point
        return {"bytes": 4.0 * (2 * math.prod(_shape(case)) + bins),
                "flops": det * pts * 12.0 * 0.5 * max(_shape(case)) + bins * pts * 40.0}
    if kind in ("unet", "unet_train"):
        V = int(case["samples"]) * int(case["d"]) * int(case["h"]) * int(case["w"])
        fl = sum(2.0 * (V >> (3 * l)) * t * ci * co for _, l, t, ci, co in _unet_layers())
        wb = sum(t * ci * co for _, _, t, ci, co in _unet_layers())
        if kind == "unet":
            return {"bytes": 16.0 * V + 4.0 * V + 2.0 * wb, "flops": fl}
        return {"bytes": 16.0 * V + 8.0 * V + 6.0 * wb, "flops": 3.0 * fl}
    if kind == "emap":
        n = (int(case["blocks"]) * int(case["rings"]) * int(case["by"]) * int(case["bz"]))
        b, f = _march_work(n * n, case, False)
        return {"bytes": 12.0 * n + 4.0 * int(case["nx"]) ** 2 * int(case["nz"]), "flops": f}
    nx, ny, nz = _shape(case)
    it = int(case["n_iter"])
    return {"bytes": it * 4.0 * (3.0 * nx * ny * nz + 121.0 * nx * ny),
            "flops": it * nx * ny * nz * (2 * 2 * 121.0 + 2 * 2.0 * nz)}


# ------------------------------------------------------------------- exact --

EXACT_SLABS = 6.0e9          # slab evaluations that take a few seconds
CHUNK = 1 << 25


def _march(lors, shape, size, tof, fwd):
    """Yields (rows, voxel (E, P, 3), weight (E, P, 3)): the terms of the projector (fwd) or the
    backprojector of each LOR; image element ix + nx (iy + ny iz)."""
    f = torch.float64
    nx, ny, nz = shape
    vx = size[0] / nx
    d = {"x": 1.0, "y": size[1] / ny / vx, "z": size[2] / nz / vx}
    step = max(1, CHUNK // max(nx, ny))
    for a in range(0, lors.shape[0], step):
        rows = torch.arange(a, min(a + step, lors.shape[0]), device=lors.device)
        r = lors[a:a + step].to(f)
        p = r[:, :6] / vx
        D = p[:, 3:6] - p[:, 0:3]
        tl = torch.sqrt(D[:, 0] ** 2 + D[:, 1] ** 2)
        L = torch.sqrt(tl ** 2 + D[:, 2] ** 2)
        live = tl >= 10.0
        if fwd and not tof:
            live &= tl >= D[:, 2].abs()
            xdom = D[:, 0].abs() >= D[:, 1].abs()
        else:
            xdom = D[:, 0].abs() > D[:, 1].abs()
        for xb in (True, False):
            s = torch.nonzero(live & (xdom == xb)).squeeze(1)
            if s.numel() == 0:
                continue
            i, j = (0, 1) if xb else (1, 0)
            np_, ns = (nx, ny) if xb else (ny, nx)
            ds = d["y"] if xb else 1.0
            p1, p2, s1, z1 = p[s, i, None], p[s, i + 3, None], p[s, j, None], p[s, 2, None]
            ks, kz = (D[s, j] / D[s, i])[:, None], (D[s, 2] / D[s, i])[:, None]
            Ls = L[s, None]
            ip = torch.arange(np_, device=lors.device)[None, :]
            lo = ip.to(f) - np_ / 2.0
            S0, S1 = ((s1 + ks * (q - p1)) / ds + ns / 2.0 for q in (lo, lo + 1))
            Z0, Z1 = ((z1 + kz * (q - p1)) / d["z"] + nz / 2.0 for q in (lo, lo + 1))
            sl, sh, zl, zh = torch.minimum(S0, S1), torch.maximum(S0, S1), torch.minimum(Z0, Z1), torch.maximum(Z0, Z1)
            c1, c2, e1, e2 = (torch.floor(t) for t in (sl, sh, zl, zh))
            bs, bz = c1 != c2, e1 != e2
            one = torch.ones((), dtype=f, device=lors.device)
            rs = torch.where(bs, (c2 - sl) / (sh - sl), one)
            rz = torch.where(bz, (e2 - zl) / (zh - zl), one)
            ok = (c1 >= torch.where(bs, -one, 0 * one)) & (c1 < ns) & (e1 >= torch.where(bz, -one, 0 * one)) & (e1 < nz)
            w = torch.sqrt(1.0 + ks ** 2 + kz ** 2) * vx
            if fwd:
                w = w / Ls / Ls
                if not tof:
                    ok &= torch.where(p1 < p2, lo + 1 <= p2, lo >= p2)
                elif xb:
                    ok &= torch.where(p2 > p1, lo > p1, torch.where(p2 < p1, lo + 1 < p1, True))
                else:
                    ok &= torch.where(p2 > p1, lo >= p1, torch.where(p2 < p1, lo + 1 <= p1, True))
            if tof:
                tb, t2 = TOF_BIN / vx, TOF_SIGMA2 / vx / vx
                tse = t2 + tb * tb / 12
                pc = ((ip - np_ // 2).to(f) + 0.5) * (1.0 if xb else d["y"])
                frac = (1.0 - r[s, 6, None] / vx / Ls) / 2
                q = ((pc - p1) / (p2 - p1) - frac) * Ls
                w = w * tb / math.sqrt(2 * math.pi * tse) * torch.exp(-q * q / (2 * tse))
            sgt = rs > rz
            both = bs & bz
            cells = [(c1, e1, torch.minimum(rs, rz), ok & (c1 >= 0) & (e1 >= 0)),
                     (torch.where(sgt, c1, c2), torch.where(sgt, e2, e1), (rs - rz).abs(),
                      ok & both & torch.where(sgt, (c1 >= 0) & (e2 < nz), (c2 < ns) & (e1 >= 0))),
                     (c2, e2, 1.0 - torch.where(both, torch.maximum(rs, rz), torch.minimum(rs, rz)),
                      ok & (bs | bz) & (c2 < ns) & (e2 < nz))]
            vox, wt = [], []
            for cs, cz, fr, on in cells:
                k = ip + nx * (cs.long() + ny * cz.long()) if xb else cs.long() + nx * (ip + ny * cz.long())
                vox.append(torch.where(on, k, torch.zeros_like(k)))
                wt.append(torch.where(on, w * fr, torch.zeros_like(fr)))
            yield rows[s], torch.stack(vox, -1), torch.stack(wt, -1)


def _fp64(img_xyz, lors, shape, size, tof):
    flat = img_xyz.to(torch.float64).permute(2, 1, 0).reshape(-1)
    out = torch.zeros(lors.shape[0], dtype=torch.float64, device=lors.device)
    for rows, v, w in _march(lors, shape, size, tof, True):
        out[rows] = (flat[v.reshape(-1)].reshape(w.shape) * w).sum((1, 2))
    return out


def _bp64(values, lors, shape, size, tof, fwd=False):
    flat = torch.zeros(shape[0] * shape[1] * shape[2], dtype=torch.float64, device=lors.device)
    for rows, v, w in _march(lors, shape, size, tof, fwd):
        flat.index_add_(0, v.reshape(-1), (values[rows].to(torch.float64)[:, None, None] * w).reshape(-1))
    return flat.reshape(shape[2], shape[1], shape[0]).permute(2, 1, 0)


def _conv64(x, w, b):
    """3x3x3 (or 1x1x1) convolution, zero padding: x (N, D, H, W, C), w (taps, cout, cin)."""
    if w.shape[0] == 1:
        return x @ w[0].t() + b
    N, D, H, W, _ = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    out = b
    for t in range(27):
        z, y, k = t // 9, (t // 3) % 3, t % 3
        out = out + xp[:, z:z + D, y:y + H, k:k + W] @ w[t].t()
    return out


def _unet64(x, P):
    act = lambda t: torch.nn.functional.leaky_relu(t, 0.01)
    skips = []
    for l in range(4):
        if l:
            N, D, H, W, C = x.shape
            x = x.reshape(N, D // 2, 2, H // 2, 2, W // 2, 2, C).mean((2, 4, 6))
        x = act(_conv64(x, *P[f"enc{l}a"]))
        x = act(_conv64(x, *P[f"enc{l}b"]))
        skips.append(x)
    for l in (2, 1, 0):
        for dim in (1, 2, 3):
            x = x.repeat_interleave(2, dim)
        x = act(_conv64(torch.cat([x, skips[l]], -1), *P[f"dec{l}a"]))
        x = act(_conv64(x, *P[f"dec{l}b"]))
    return _conv64(x, *P["head"])


def _exact_unet(case, seed):
    bits, target, dims = _unet_inputs(case, seed)
    N = int(case["samples"])
    z = np.load(WEIGHTS, allow_pickle=False)
    dev = bits.device
    train = case["kind"] == "unet_train"
    P = {n: tuple(torch.from_numpy(z[n + s]).to(dev, torch.float64).requires_grad_(train) for s in (".w", ".b"))
         for n, *_ in _unet_layers()}
    x = bits.view(torch.bfloat16).to(torch.float64)[:, :4].reshape((N,) + dims + (4,))
    if not train:
        return torch.cat([_unet64(x[i:i + 1], P).reshape(-1) for i in range(N)])
    out = []
    V = dims[0] * dims[1] * dims[2]
    for i in range(N):                                   # the loss is the sum of the samples' mean squares
        o = _unet64(x[i:i + 1], P).reshape(-1)
        ((o - target[i * V:(i + 1) * V].to(torch.float64)) ** 2).mean().backward()
        out.append(o.detach())
    gw, gb = [], []
    for n, _, t, ci, co in _unet_layers():               # stored padded: rows to 32, columns to 8
        full = torch.zeros((t, -(-co // 32) * 32, -(-ci // 8) * 8), dtype=torch.float64, device=dev)
        full[:, :co, :ci] = P[n][0].grad
        gw.append(full)
        gb.append(P[n][1].grad)
    return [torch.cat(out)] + gw + gb


def _exact_psf(case, seed):
    w, kz = _psf_tables(case)
    data = _psf_data(case, seed).to(torch.float64)
    nx, ny, nz = _shape(case)
    dev = data.device
    W = torch.from_numpy(w).to(dev, torch.float64).reshape(nx, ny, 121)
    K = torch.from_numpy(kz).to(dev, torch.float64)

    def taps(x, adjoint):
        out = torch.zeros_like(x)
        for o in range(121):
            a, b = o // 11 - 5, o % 11 - 5
            i0, i1, j0, j1 = max(0, -a), min(nx, nx - a), max(0, -b), min(ny, ny - b)
            if i0 >= i1 or j0 >= j1:
                continue
            wt = W[i0:i1, j0:j1, o, None]
            if adjoint:
                out[i0:i1, j0:j1] += wt * x[i0 + a:i1 + a, j0 + b:j1 + b]
            else:
                out[i0 + a:i1 + a, j0 + b:j1 + b] += wt * x[i0:i1, j0:j1]
        return out

    x = torch.ones_like(data)
    for _ in range(int(case["n_iter"])):
        c = taps(x @ K.t(), False)
        x = x * (taps(data / (c + 1e-16), True) @ K)
    return x


def _exact_sss(case, seed):
    em, mu = _sss_inputs(case, seed)
    shape, size, dev, f = _shape(case), _size(case), em.device, torch.float64
    v = float(case["voxel"])
    step = max(1, int(SSS_SPACING // v))
    cnt = [n // step for n in shape]
    k = torch.meshgrid(*(torch.arange(c, device=dev) for c in cnt), indexing="ij")
    k = [t.reshape(-1) for t in k]
    pos = torch.stack([(step * (t.to(f) + 0.5) * v - s / 2).to(torch.float32) for t, s in zip(k, size)], 1)
    m = mu[step * k[0] + step // 2, step * k[1] + step // 2, step * k[2] + step // 2]
    pos, m = pos[m != 0], m[m != 0].to(f)
    rings = _rings(case) or list(range(32))
    a = 2 * math.pi * torch.arange(128, device=dev, dtype=f) / 128
    det = torch.cat([torch.stack([SSS_RADIUS * torch.cos(a), SSS_RADIUS * torch.sin(a),
                                  torch.full_like(a, (r + 0.5) * SSS_AXIAL / 32 - SSS_AXIAL / 2), a], 1)
                     for r in rings]).to(torch.float32)
    nd, ns = det.shape[0], pos.shape[0]
    if 2.0 * nd * ns * max(shape) > 4.0 * EXACT_SLABS:
        return None
    E, M = torch.empty((nd, ns), dtype=f, device=dev), torch.empty((nd, ns), dtype=f, device=dev)
    fe, fm = (t.to(f).permute(2, 1, 0).reshape(-1) for t in (em, mu))
    few = max(1, CHUNK // (ns * max(shape)))
    for i in range(0, nd, few):
        n = min(few, nd - i)
        lors = torch.cat([det[i:i + n, None, :3].expand(n, ns, 3), pos[None].expand(n, ns, 3)], 2).reshape(-1, 6)
        L2 = ((lors[:, 3:6] - lors[:, 0:3]).to(f) ** 2).sum(1) / (v * v)
        e, u = (torch.zeros(n * ns, dtype=f, device=dev) for _ in range(2))
        for rows, vox, w in _march(lors, shape, size, False, True):
            e[rows] = (fe[vox.reshape(-1)].reshape(w.shape) * w).sum((1, 2))
            u[rows] = (fm[vox.reshape(-1)].reshape(w.shape) * w).sum((1, 2))
        E[i:i + n], M[i:i + n] = (e * L2).reshape(n, ns), (u * L2).reshape(n, ns)
    d = det.to(f)
    vec = d[:, None, :3] - pos[None].to(f)
    r = vec.norm(dim=2)
    g = (vec[:, :, 0] * torch.cos(d[:, 3])[:, None] + vec[:, :, 1] * torch.sin(d[:, 3])[:, None]) / r ** 3
    unit = vec / r[:, :, None]
    deg = torch.arange(181, device=dev, dtype=f) / 180.0 * math.pi
    Ep = 511.0 / (2.0 - torch.cos(deg))
    sig_kn = math.pi * (40.0 / 9.0 - 3.0 * math.log(3.0))
    # the path's own Klein-Nishina factor takes the angle in the place of its cosine
    kn = 1 / (2 - deg) ** 2 * ((1 + deg ** 2) / 2 + (1 - deg) ** 2 / 2 / (2 - deg)) / sig_kn
    s = math.sqrt(511.0) * 0.15
    Ei = torch.arange(400, 650, 5, device=dev, dtype=f)
    eff = torch.exp(-(Ei[None] - Ep[:, None]) ** 2 / 2 / s ** 2).sum(1)
    scale = 5 / math.sqrt(1022 * math.pi) / 0.15 * float(torch.exp(-(Ei - 511.0) ** 2 / 2 / s ** 2).sum()) / (4 * math.pi)
    bins = _sss_bins(len(rings)).to(dev)
    out = torch.empty(bins.shape[0], dtype=f, device=dev)
    nb = max(1, CHUNK // ns)
    for b in range(0, bins.shape[0], nb):
        A, B = bins[b:b + nb, 0], bins[b:b + nb, 1]
        cosv = -(unit[A] * unit[B]).sum(2)
        q = torch.clamp((torch.acos(cosv.clamp(-1, 1)) * (180.0 / math.pi)).long(), 0, 180)
        rr = 511.0 / Ep[q]
        I = torch.exp(-(M[A] + M[B] * rr)) * E[A] + torch.exp(-(M[A] * rr + M[B])) * E[B]
        out[b:b + nb] = (g[A] * g[B] * eff[q] * kn[q] * m * I).sum(1) * scale
    return out.reshape(len(rings), 64, 64)


def _sss_bins(n_rings):
    a = np.arange(64) * math.pi / 64
    s = (np.arange(64) + 0.5 - 32) * (2.0 * SSS_FOV / 64)
    A, S = np.meshgrid(a, s, indexing="ij")
    t = np.sqrt(np.maximum(SSS_RADIUS ** 2 - S ** 2, 0.0))
    psi = [np.arctan2(S * np.sin(A) + q * t * np.cos(A), S * np.cos(A) - q * t * np.sin(A)) for q in (-1, 1)]
    k = [np.mod(np.rint(p / (2 * math.pi) * 128), 128).astype(np.int64) for p in psi]
    ring = np.arange(n_rings)[:, None, None] * 128
    return torch.from_numpy(np.stack([ring + k[0][None], ring + k[1][None]], -1).reshape(-1, 2))


def _exact_em(case, seed, lors, values, x, subsets, kind, eps):
    shape, size = _shape(case), _size(case)
    emap = _emap(case).to(torch.float64)
    emap = torch.where(emap == 0, torch.full_like(emap, 1e8), emap)
    for idx in subsets:
        l, y = lors[idx], values[idx].to(torch.float64)
        p = _fp64(x, l, shape, size, case["tof"]) + eps
        q = torch.where(p == 0, torch.zeros_like(p), y / p) if kind else y / p
        x = x * _bp64(q, l, shape, size, case["tof"]) / emap
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind in ("unet", "unet_train"):
        return _exact_unet(case, seed)
    if kind == "psf":
        return _exact_psf(case, seed)
    if kind == "sss":
        return _exact_sss(case, seed)
    if kind == "emap":
        return None                                      # every pair of crystals: over the time
    n, shape, size = int(case["events"]), _shape(case), _size(case)
    passes = {"mlem": 2 * int(case.get("n_iter", 1)), "osem": 2, "autograd": 2 * int(case.get("batch", 1))}.get(kind, 1)
    if float(n) * max(shape[0], shape[1]) * passes > 3.0 * EXACT_SLABS:
        return None
    lors, values, image = _lists(case, seed)
    if kind == "project":
        return _fp64(image, lors, shape, size, case["tof"])
    if kind == "backproject":
        return _bp64(values, lors, shape, size, case["tof"])
    if kind == "attenuation":
        mu = ((image > 0.5).to(torch.float32) * MU_WATER)
        L2 = ((lors[:, 3:6].to(torch.float64) - lors[:, 0:3].to(torch.float64)) ** 2).sum(1)
        p = _fp64(mu, lors[:, :6], shape, size, False)
        return values.to(torch.float64) / torch.exp(-p * L2 / float(case["voxel"]))
    if kind == "mlem":
        eps = float(np.float32(float(values.mean().item()) * 1e-8))
        x = torch.ones(tuple(shape), dtype=torch.float64, device=lors.device)
        every = torch.arange(n, device=lors.device)
        return _exact_em(case, seed, lors, values, x, [every] * int(case["n_iter"]), 0, eps)
    if kind == "osem":
        m = n // int(case["n_sub"])
        perm = _perm(case, seed)
        subsets = [perm[k * m:(k + 1) * m] for k in range(int(case["n_sub"]))]
        x = (image + 0.1).to(torch.float64)
        return _exact_em(case, seed, lors, values, x, subsets, 1, 1e-5).permute(2, 1, 0)
    images = _images(case, seed)
    p = torch.stack([_fp64(i, lors, shape, size, case["tof"]) for i in images])
    g = _bp64(values, lors, shape, size, case["tof"], fwd=True)
    return [p, g[None].expand_as(images)]
