"""What a program built on dlux_amd spends its time in, as measurable cases.

Every case is one pass through the public API: a polychromatic PSF of an
aberrated telescope, a phase-retrieval step (PSF, loss, gradient), the matrix
Fourier transform of prepared wavefronts, an uneven batch of sources, a crowded
field through a detector, angular-spectrum propagation, and the detector chain
with its gradient.  Inputs are made from a seed on the GPU; ``exact`` restates
each path in 64-bit torch without the package.
"""

from __future__ import annotations

import functools
import math
from types import SimpleNamespace

import numpy as np
import torch

import dlux_amd as dl
from dlux_amd import layers, runtime
from dlux_amd.utils import propagation, units

DIAM = 1.0            # aperture diameter, metres
P_OUT = 2.5e-7        # focal pixel, radians: twice Nyquist at 1 um
DEV = "cuda"

# Relative 2-norm error bounds, about four times the largest seen against
# ``exact`` (or between orders of summation) over the listed and drawn sizes.
TOL = {
    "psf": {"fp32": 4e-6, "bf16x3": 8e-6},
    "fit": {"fp32": 4e-6, "bf16x3": 8e-6},
    "mft": {"fp32": 4e-6, "bf16x3": 2e-5},
    "batch": {"bf16x3": 1.2e-5},
    "scene": {"bf16x3": 8e-6},
    "asm": {"fp32": 2e-6},
    "detector": {"fp32": 5e-7},
    "detector_fit": {"fp32": 5e-7},
}


def listed():
    return [
        # one monochromatic PSF: the call an interactive user or an optimiser's inner
        # loop makes; launches and host latency
        dict(name="psf_mono_256", kind="psf", n_in=256, n_out=128, n_wl=1, n_zern=10,
             precision="fp32", spiders=False, tilted=False),
        # the broadband PSF of a spider-obstructed telescope in both arithmetic forms
        # (fp32 is the package's default)
        dict(name="psf_poly_512_bf16x3", kind="psf", n_in=512, n_out=256, n_wl=64, n_zern=36,
             precision="bf16x3", spiders=True, tilted=False),
        dict(name="psf_poly_512_fp32", kind="psf", n_in=512, n_out=256, n_wl=64, n_zern=36,
             precision="fp32", spiders=True, tilted=False),
        # an off-axis star on grids that are no multiple of a tile
        dict(name="psf_ragged_offaxis", kind="psf", n_in=401, n_out=173, n_wl=11, n_zern=21,
             precision="bf16x3", spiders=True, tilted=True),
        # phase retrieval: forward, Gaussian likelihood, gradient of the Zernike coefficients
        dict(name="fit_zernike_512", kind="fit", n_in=512, n_out=128, n_wl=16, n_zern=36,
             precision="bf16x3", wrt="coeffs"),
        # the same with a free OPD map, on an odd grid, in the default precision
        dict(name="fit_opd_map_300", kind="fit", n_in=300, n_out=101, n_wl=5, n_zern=10,
             precision="fp32", wrt="opd"),
        # fields a program already holds (a coronagraph's planes), propagated with a
        # sub-pixel shift per wavelength
        dict(name="mft_fields_512", kind="mft", n_in=512, n_out=256, n_wl=16,
             precision="fp32", shifted=True),
        # many sources of uneven pupil and image sizes, each at its own position and flux
        dict(name="batch_uneven_48x16", kind="batch", n_src=48, n_wl=16, n_max=1024,
             n_out_max=256, layout=5, precision="bf16x3"),
        # a crowded field through jitter, pixel response, downsampling and a bias
        dict(name="scene_24_stars", kind="scene", n_src=24, n_wl=8, n_in=512, n_out=256,
             n_zern=21, down=4, precision="bf16x3"),
        # near-field propagation of a padded wavefront
        dict(name="asm_1024_2048", kind="asm", n=1024, m=2048, batch=1, precision="fp32"),
        # a stack of oversampled frames through the detector, and its gradient
        dict(name="detector_64x1024", kind="detector", frames=64, n=1024, down=4, jitter=9,
             precision="fp32"),
        dict(name="detector_fit_24x512", kind="detector_fit", frames=24, n=512, down=2,
             jitter=9, precision="fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _side(rng, lo, hi):
    """A grid side: any integer half of the time, else a multiple of 16."""
    n = _log_int(rng, lo, hi)
    return n if rng.random() < 0.5 else max(16, 16 * round(n / 16))


def draw(rng):
    kind = rng.choice(["psf", "psf", "psf", "fit", "fit", "mft", "batch", "scene", "asm",
                       "detector", "detector_fit"])
    prec = rng.choice(["fp32", "bf16x3"])
    if kind == "psf":
        n_in = _side(rng, 128, 1024)
        n_out = _side(rng, 48, min(512, n_in))
        most = _mft_flops(512, 256) * 64 / _mft_flops(n_in, n_out)
        return dict(kind=kind, n_in=n_in, n_out=n_out,
                    n_wl=max(1, min(_log_int(rng, 1, 64), int(most))), n_zern=rng.randint(4, 36),
                    precision=prec, spiders=rng.random() < 0.5, tilted=rng.random() < 0.5)
    if kind == "fit":
        n_in = _side(rng, 128, 640)
        return dict(kind=kind, n_in=n_in, n_out=_side(rng, 48, min(192, n_in)),
                    n_wl=_log_int(rng, 1, 16), n_zern=rng.randint(4, 36), precision=prec,
                    wrt=rng.choice(["coeffs", "opd"]))
    if kind == "mft":
        return dict(kind=kind, n_in=_side(rng, 128, 640), n_out=_side(rng, 48, 320),
                    n_wl=_log_int(rng, 1, 24), precision=prec, shifted=rng.random() < 0.5)
    if kind == "batch":
        return dict(kind=kind, n_src=_log_int(rng, 8, 40), n_wl=_log_int(rng, 2, 16),
                    n_max=rng.choice([256, 400, 512, 1000]), n_out_max=rng.choice([64, 128, 250]),
                    layout=rng.randint(0, 1000), precision="bf16x3")
    if kind == "scene":
        down = rng.choice([2, 4])
        return dict(kind=kind, n_src=_log_int(rng, 3, 40), n_wl=_log_int(rng, 2, 10),
                    n_in=_side(rng, 192, 512), n_out=down * (_side(rng, 64, 256) // down),
                    n_zern=rng.randint(4, 36), down=down, precision="bf16x3")
    if kind == "asm":
        m = rng.choice([512, 1024, 2048])
        n = 2 * (_side(rng, m // 4, m) // 2)
        return dict(kind=kind, n=min(n, m), m=m, batch=rng.randint(1, 1 if m == 2048 else 3),
                    precision="fp32")
    down = rng.choice([2, 3, 4])
    n = down * 4 * max(8, _log_int(rng, 96, 1024) // (4 * down))
    frames = _log_int(rng, 1, 64 if kind == "detector" else 32)
    cap = (64 if kind == "detector" else 16) * 1024 * 1024 // (n * n)
    return dict(kind=kind, frames=max(1, min(frames, cap)), n=n, down=down,
                jitter=rng.choice([5, 7, 9, 11]), precision="fp32")


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _gen(seed, salt=0):
    return torch.Generator(device=DEV).manual_seed(1_000_003 * int(seed) + salt)


def _rng(seed, salt=0):
    return np.random.default_rng([int(seed), salt])


def _coords(n, d=DIAM):
    return (np.arange(n) - (n - 1) / 2.0) * (d / n)


@functools.lru_cache(maxsize=4)
def _pupil(n, n_zern, spiders):
    """(mask, Zernike basis) float32 on the GPU: a circular aperture, three 8-px
    vanes, Noll modes 2 .. n_zern + 1 on the unit disc."""
    x = _coords(n) / (DIAM / 2)
    xx, yy = np.meshgrid(x, x)
    r, th = np.hypot(xx, yy), np.arctan2(yy, xx)
    mask = (r < 1.0).astype(np.float32)
    if spiders:
        for a in np.deg2rad([0.0, 120.0, 240.0]):
            along, across = xx * np.cos(a) + yy * np.sin(a), -xx * np.sin(a) + yy * np.cos(a)
            mask[(along > 0) & (np.abs(across) < 8.0 / n)] = 0.0
    basis = np.empty((n_zern, n, n), np.float32)
    for i in range(n_zern):
        j = i + 2
        nn = int((math.sqrt(8 * j - 7) - 1) / 2)
        k = j - nn * (nn + 1) // 2 - 1
        m = 2 * ((k + 1) // 2) if nn % 2 == 0 else 2 * (k // 2) + 1
        rad = np.zeros_like(r)
        for s in range((nn - m) // 2 + 1):
            c = (-1) ** s * math.factorial(nn - s) / (
                math.factorial(s) * math.factorial((nn + m) // 2 - s)
                * math.factorial((nn - m) // 2 - s))
            rad += c * r ** (nn - 2 * s)
        if m == 0:
            z = math.sqrt(nn + 1) * rad
        else:
            z = math.sqrt(2 * (nn + 1)) * rad * (np.cos(m * th) if j % 2 == 0 else np.sin(m * th))
        basis[i] = z * (r <= 1.0)
    return torch.as_tensor(mask, device=DEV), torch.as_tensor(basis, device=DEV)


def _wavelengths(n, lo=0.8e-6, hi=1.2e-6):
    return np.array([1.0e-6]) if n == 1 else np.linspace(lo, hi, n)


def _system(case, coeffs, opd=None):
    mask, basis = _pupil(case["n_in"], case["n_zern"], bool(case.get("spiders")))
    chain = [("aperture", layers.TransmissiveLayer(mask, normalise=True))]
    if coeffs is not None:
        chain.append(("aberrations", layers.BasisLayer(basis, coeffs)))
    if opd is not None:
        chain.append(("map", layers.AberratedLayer(opd=opd)))
    return dl.AngularOpticalSystem(
        wf_npixels=case["n_in"], diameter=DIAM, layers=chain, psf_npixels=case["n_out"],
        psf_pixel_scale=float(units.rad2arcsec(P_OUT)), oversample=1)


def _batch_sources(case, seed):
    """Per-source sizes (fixed by the case) and position, flux (by the seed)."""
    fixed, rng = _rng(case["layout"], 1), _rng(seed, 2)
    sizes = [case["n_max"] // 4, case["n_max"] // 2, case["n_max"]]
    outs = [case["n_out_max"] // 4, case["n_out_max"] // 2, case["n_out_max"]]
    out = []
    for _ in range(case["n_src"]):
        out.append(dict(n_in=int(fixed.choice(sizes)), n_out=max(16, int(fixed.choice(outs))),
                        shift=rng.uniform(-9.7e-6, 9.7e-6, 2) / P_OUT,
                        flux=float(np.exp(rng.uniform(np.log(1e3), np.log(1e6))))))
    return out


def _inputs(case, seed):
    """The arrays of a case, for ``prepare`` and ``exact`` alike."""
    s = SimpleNamespace(case=case, kind=case["kind"], precision=case["precision"])
    kind = case["kind"]
    if kind in ("psf", "fit", "scene"):
        s.wls = _wavelengths(case["n_wl"]) if kind != "fit" else _wavelengths(
            case["n_wl"], 0.9e-6, 1.1e-6)
        s.weights = np.ones(len(s.wls)) / len(s.wls)
        s.coeffs = (30e-9 if kind != "fit" else 50e-9) * torch.randn(
            case["n_zern"], generator=_gen(seed), device=DEV)
        s.mask, s.basis = _pupil(case["n_in"], case["n_zern"], bool(case.get("spiders")))
        s.offset = _rng(seed, 3).uniform(-4e-6, 4e-6, 2) if case.get("tilted") else np.zeros(2)
    if kind == "fit":
        truth = 50e-9 * torch.randn(case["n_zern"], generator=_gen(seed, 1), device=DEV)
        s.flux = 1e6
        psf = _exact_psf(s.mask, _opd(s.basis, truth), s.wls, s.weights, case["n_out"])
        s.data = torch.poisson((s.flux * psf.clamp(min=0)).float(), generator=_gen(seed, 2))
        s.var = s.data.clamp(min=1.0)
        s.opd = torch.einsum("jyx,j->yx", s.basis, s.coeffs)
    if kind == "mft":
        s.wls = _wavelengths(case["n_wl"])
        n = case["n_in"]
        x = torch.as_tensor(_coords(n), device=DEV, dtype=torch.float32)
        amp = ((x[:, None] ** 2 + x[None, :] ** 2) < (DIAM / 2) ** 2).float() / n
        ph = torch.randn((case["n_wl"], 8, 8), generator=_gen(seed), device=DEV)
        ph = torch.nn.functional.interpolate(ph[:, None], (n, n), mode="bicubic")[:, 0]
        s.fields = torch.polar(amp.expand_as(ph).contiguous(), ph).contiguous()
        s.shift = _rng(seed, 4).uniform(-6, 6, (case["n_wl"], 2)) if case["shifted"] else \
            np.zeros((case["n_wl"], 2))
    if kind == "batch":
        s.wls = _wavelengths(case["n_wl"])
        s.sources = _batch_sources(case, seed)
        s.fields = []
        for i, src in enumerate(s.sources):
            n = src["n_in"]
            mask, basis = _pupil(n, 10, False)
            c = 30e-9 * torch.randn(10, generator=_gen(seed, 100 + i), device=DEV)
            ph = (2 * math.pi / 1e-6) * torch.einsum("jyx,j->yx", basis, c)
            s.fields.append(torch.polar(mask / mask.norm(), ph).contiguous())
    if kind == "scene":
        rng = _rng(seed, 5)
        half = 0.35 * case["n_out"] * P_OUT
        s.positions = rng.uniform(-half, half, (case["n_src"], 2))
        s.fluxes = np.exp(rng.uniform(np.log(1e3), np.log(1e6), case["n_src"]))
        s.resp = 0.9 + 0.2 * torch.rand((case["n_out"],) * 2, generator=_gen(seed, 1), device=DEV)
    if kind == "asm":
        n = case["n"]
        ph = torch.randn((case["batch"], 1, 16, 16), generator=_gen(seed), device=DEV)
        ph = torch.nn.functional.interpolate(ph, (n, n), mode="bicubic")[:, 0]
        s.fields = torch.polar(torch.ones_like(ph), ph).contiguous()
        s.z = float(_rng(seed, 6).uniform(1e-3, 100e-3))
        s.wl, s.dx = 1.0e-6, 2.0e-6
    if kind in ("detector", "detector_fit"):
        g = _gen(seed)
        n = case["n"]
        s.frames = torch.rand((case["frames"], n, n), generator=g, device=DEV)
        s.resp = 0.9 + 0.2 * torch.rand((n, n), generator=g, device=DEV)
        if kind == "detector_fit":
            s.cot = torch.randn((case["frames"],) + (n // case["down"],) * 2, generator=g,
                                device=DEV)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("psf", "scene"):
        s.system = _system(case, s.coeffs)
    if kind == "fit":
        if case["wrt"] == "coeffs":
            s.leaf = s.coeffs.clone().requires_grad_()
            s.system = _system(case, s.leaf)
        else:
            s.leaf = s.opd.clone().requires_grad_()
            s.system = _system(case, None, s.leaf)
    if kind == "batch":
        inst = []
        for i, src in enumerate(s.sources):
            for wl in s.wls:
                inst.append(dict(field=s.fields[i], wavelength=float(wl), n_out=src["n_out"],
                                 pixel_scale_in=DIAM / src["n_in"], pixel_scale_out=P_OUT,
                                 shift=(float(src["shift"][0]), float(src["shift"][1])),
                                 weight=src["flux"] / len(s.wls), out_index=i))
        s.batch = runtime.MftBatch(inst, n_outputs=len(s.sources))
    if kind == "scene":
        det = dl.LayeredDetector([layers.ApplyJitter(0.6), layers.ApplyPixelResponse(s.resp),
                                  layers.Downsample(case["down"]), layers.AddConstant(10.0)])
        stars = dl.PointSources(s.wls, position=s.positions, flux=s.fluxes)
        s.telescope = dl.Telescope(s.system, ("stars", stars), det)
    if kind == "asm":
        s.wf = dl.Wavefront.from_phasor(s.fields, np.full(case["batch"], s.wl), pixel_scale=s.dx)
    if kind in ("detector", "detector_fit"):
        tail = [layers.ApplySaturation(0.9 * case["down"] ** 2)] if kind == "detector" else []
        s.detector = dl.LayeredDetector(
            [layers.ApplyJitter(0.5, case["jitter"], 3), layers.ApplyPixelResponse(s.resp),
             layers.Downsample(case["down"])] + tail + [layers.AddConstant(0.01)])
        if kind == "detector_fit":
            s.frames.requires_grad_()
        s.psf = dl.PSF(s.frames, 1.0)
    return s


def run(s):
    if s.kind == "psf":
        with runtime.precision(s.precision):
            return s.system.propagate(s.wls, offset=s.offset, weights=s.weights)
    if s.kind == "fit":
        with runtime.precision(s.precision):
            psf = s.system.propagate(s.wls, weights=s.weights)
            loss = 0.5 * torch.sum((s.flux * psf - s.data) ** 2 / s.var)
            (grad,) = torch.autograd.grad(loss, s.leaf)
        return {"psf": psf.detach(), "grad": grad}
    if s.kind == "mft":
        return propagation.MFT(s.fields, s.wls, DIAM / s.case["n_in"], s.case["n_out"], P_OUT,
                               shift=s.shift, precision=s.precision)
    if s.kind == "batch":
        return s.batch()
    if s.kind == "scene":
        with runtime.precision(s.precision):
            return s.telescope.model()
    if s.kind == "asm":
        return s.wf.propagate_ASM(s.z, s.case["m"]).phasor
    image = s.detector(s.psf)
    if s.kind == "detector":
        return image
    (grad,) = torch.autograd.grad(image, s.frames, s.cot)
    return {"image": image.detach(), "grad": grad}


# ---------------------------------------------------------------------------
# floors, tolerances, 64-bit values
# ---------------------------------------------------------------------------


def _mft_flops(n_in, n_out):
    """Real operations of one two-sided transform.  The kernel of each axis is a
    cosine and a sine on symmetric grids, so a quarter of the 8 (N_out N_in^2 +
    N_out^2 N_in) of the plain complex products is needed."""
    return 2.0 * (n_out * n_in ** 2 + n_out ** 2 * n_in)


def work(case):
    k = case["kind"]
    if k in ("psf", "fit"):
        n, m = case["n_in"], case["n_out"]
        f = _mft_flops(n, m) * case["n_wl"]
        if k == "psf":
            return {"bytes": 4.0 * ((case["n_zern"] + 1) * n * n + m * m),
                    "flops": f + 2.0 * case["n_zern"] * n * n}
        planes = case["n_zern"] + 1 if case["wrt"] == "coeffs" else 3
        return {"bytes": 4.0 * (planes * n * n + 4 * m * m), "flops": 2 * f}
    if k == "mft":
        n, m = case["n_in"], case["n_out"]
        return {"bytes": 8.0 * case["n_wl"] * (n * n + m * m),
                "flops": _mft_flops(n, m) * case["n_wl"]}
    if k == "batch":
        src = _batch_sources(case, 0)
        return {"bytes": float(sum(8 * s["n_in"] ** 2 + 4 * s["n_out"] ** 2 for s in src)),
                "flops": sum(_mft_flops(s["n_in"], s["n_out"]) for s in src) * case["n_wl"]}
    if k == "scene":
        n, m = case["n_in"], case["n_out"]
        return {"bytes": 4.0 * ((case["n_zern"] + 1) * n * n + m * m + (m // case["down"]) ** 2),
                "flops": _mft_flops(n, m) * case["n_wl"] * case["n_src"]}
    if k == "asm":
        n, m, b = case["n"], case["m"], case["batch"]
        return {"bytes": 8.0 * b * (n * n + m * m), "flops": 20.0 * b * m * m * math.log2(m)}
    px = case["frames"] * case["n"] ** 2
    small = px / case["down"] ** 2
    if k == "detector":
        return {"bytes": 4.0 * (px + small + case["n"] ** 2), "flops": 4.0 * case["jitter"] * px}
    return {"bytes": 4.0 * (2 * px + 2 * small + case["n"] ** 2),
            "flops": 8.0 * case["jitter"] * px}


def tolerance(case):
    return {"rel": TOL[case["kind"]][case["precision"]]}


def _opd(basis, coeffs):
    return torch.einsum("jyx,j->yx", basis.double(), coeffs.double())


def _kernel(n_in, n_out, wl, shift=0.0):
    """(n_out, n_in) complex128 exp(-2 pi i a_k b_l) of the centred grids."""
    a = (torch.arange(n_in, device=DEV, dtype=torch.float64) - (n_in - 1) / 2.0 - shift) / n_in
    b = (torch.arange(n_out, device=DEV, dtype=torch.float64) - (n_out - 1) / 2.0 - shift) * (
        P_OUT * DIAM / wl)
    t = torch.outer(b, a)
    return torch.polar(torch.ones_like(t), -2 * math.pi * (t - torch.round(t)))


def _exact_mft(field, wl, n_out, shift=(0.0, 0.0)):
    n = field.shape[-1]
    norm = n_out * P_OUT * DIAM / wl / (n * n_out)
    wx = _kernel(n, n_out, wl, float(shift[0]))
    wy = wx if shift[0] == shift[1] else _kernel(n, n_out, wl, float(shift[1]))
    return norm * (wy @ field @ wx.T)


def _exact_psf(mask, opd, wls, weights, n_out, tilt=(0.0, 0.0)):
    n = mask.shape[-1]
    amp = mask.double() / mask.double().norm()
    x = torch.as_tensor(_coords(n), device=DEV)
    path = opd.double() + tilt[0] * x[None, :] + tilt[1] * x[:, None]
    out = 0.0
    for wl, w in zip(wls, weights):
        field = torch.polar(amp, 2 * math.pi / wl * path) if not path.requires_grad else \
            amp * torch.exp(2j * math.pi / wl * path)
        out = out + w * _exact_mft(field, float(wl), n_out).abs() ** 2
    return out


def _exact_detector(img, sigma, size, resp, down, bias, full=None):
    g = np.exp(-0.5 * (np.linspace(-5.0, 5.0, size * 3) / sigma) ** 2).reshape(size, 3).sum(1)
    f = torch.as_tensor(g / g.sum(), device=DEV)
    h = size // 2
    x = torch.nn.functional.pad(img, (h, h, h, h))
    n = img.shape[-1]
    x = sum(f[i] * x[..., i:i + n, :] for i in range(size))
    x = sum(f[i] * x[..., i:i + n] for i in range(size))
    x = x * resp.double()
    x = x.reshape(x.shape[:-2] + (n // down, down, n // down, down)).sum((-3, -1))
    return (x if full is None else x.clamp(max=full)) + bias


def exact(case, seed):
    s = _inputs(case, seed)
    k = case["kind"]
    if k == "psf":
        return _exact_psf(s.mask, _opd(s.basis, s.coeffs), s.wls, s.weights, case["n_out"],
                          s.offset)
    if k == "fit":
        if case["wrt"] == "coeffs":
            leaf = s.coeffs.double().requires_grad_()
            opd = torch.einsum("jyx,j->yx", s.basis.double(), leaf)
        else:
            opd = leaf = s.opd.double().requires_grad_()
        psf = _exact_psf(s.mask, opd, s.wls, s.weights, case["n_out"])
        loss = 0.5 * torch.sum((s.flux * psf - s.data.double()) ** 2 / s.var.double())
        (grad,) = torch.autograd.grad(loss, leaf)
        return {"psf": psf.detach(), "grad": grad}
    if k == "mft":
        return torch.stack([_exact_mft(f.to(torch.complex128), float(wl), case["n_out"], sh)
                            for f, wl, sh in zip(s.fields, s.wls, s.shift)])
    if k == "batch":
        out = []
        for f, src in zip(s.fields, s.sources):
            f = f.to(torch.complex128)
            out.append(sum(src["flux"] / len(s.wls) * _exact_mft(
                f, float(wl), src["n_out"], src["shift"]).abs() ** 2 for wl in s.wls))
        return out
    if k == "scene":
        opd = _opd(s.basis, s.coeffs)
        img = sum(_exact_psf(s.mask, opd, s.wls, s.weights * fl, case["n_out"], pos)
                  for pos, fl in zip(s.positions, s.fluxes))
        return _exact_detector(img, 0.6, 9, s.resp, case["down"], 10.0)
    if k == "asm":
        n, m = case["n"], case["m"]
        x = torch.nn.functional.pad(s.fields.to(torch.complex128), ((m - n) // 2,) * 4)
        spec = torch.fft.fft2(torch.fft.ifftshift(x, dim=(-2, -1)))
        f = torch.fft.fftfreq(m, s.dx, device=DEV, dtype=torch.float64)
        arg = s.wl ** -2 - f[:, None] ** 2 - f[None, :] ** 2
        t = s.z * torch.sqrt(arg.clamp(min=0))
        h = torch.polar((arg > 0).double(), 2 * math.pi * (t - torch.round(t)))
        return torch.fft.fftshift(torch.fft.ifft2(spec * h), dim=(-2, -1))
    full = 0.9 * case["down"] ** 2 if k == "detector" else None
    img = s.frames.double().requires_grad_(k == "detector_fit")
    out = _exact_detector(img, 0.5, case["jitter"], s.resp, case["down"], 0.01, full)
    if k == "detector":
        return out
    (grad,) = torch.autograd.grad(out, img, s.cot.double())
    return {"image": out.detach(), "grad": grad}
