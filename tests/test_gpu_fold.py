"""The folded contractions at the sizes where their tiles, stages and rules can
go wrong, against the FP64 oracle: sides of one to a few rows, odd and even,
either side of a 16-k stage, a 32-row block and a 64- or 128-column tile; every
width of both stages; each loader (aligned runs, single values, missing planes,
a phase plane, a tilt, a field with and without shifts, a folded pupil in
memory); the gradient's epilogues; uneven batches whose tile groups are not full.

Bounds.  The split form drops 2^-18 of a product's terms twice over (each
operand's third part); 3 * 2^-18 per term and contraction covers that and the
carrying of a table value's rest to its neighbour.  The hardware sine and cosine are good to 1.3e-7.  float32 sums of
K terms round by 2^-24 of the running sum each.  Independent errors of the K =
N_in terms of a contraction add in quadrature against a sum that adds
coherently at the peak, so relative to it a field is off by
sigma = sqrt(2) 3 2^-18 / sqrt(N_in) (split) + 2^-24 sqrt(N_in) + 2e-7, and an
intensity by twice that; 6 sigma of the largest of all pixels.
"""

import numpy as np
import pytest

from oracle import dlux_oracle as orc

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

P_OUT = 2.1e-7


@pytest.fixture(scope="module")
def rt():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dlux_amd import runtime
    return runtime


def _sigma(n, prec):
    split = np.sqrt(2) * 3 * 2.0 ** -18 / np.sqrt(n) if prec == "bf16x3" else 0.0
    return split + 2.0 ** -24 * np.sqrt(n) + 2e-7


def _err(x, ref):
    x = x.detach().cpu().numpy() if isinstance(x, torch.Tensor) else np.asarray(x)
    return float(np.max(np.abs(x - ref)) / max(np.max(np.abs(ref)), 1e-300))


def _planes(n, planes, seed, offset):
    """float32 device planes and their float64 values; `offset` floats into a buffer."""
    rng = np.random.default_rng(seed)
    make = {"amp": lambda: rng.uniform(0.5, 1.0, (n, n)),
            "opd": lambda: 3e-8 * rng.standard_normal((n, n)),
            "phase": lambda: 0.2 * rng.standard_normal((n, n))}
    dev, ref = {}, {}
    for k in ("amp", "opd", "phase"):
        if k in planes:
            a = make[k]().astype(np.float32)
            buf = torch.zeros(n * n + offset, device="cuda")
            buf[offset:] = torch.as_tensor(a.reshape(-1)).cuda()
            dev[k], ref[k] = buf[offset:].view(n, n), a.astype(np.float64)
    return dev, ref


def _pupil(n, ref, wl, tilt):
    x = (np.arange(n) - (n - 1) / 2) / n
    path = tilt[0] * x[None, :] + tilt[1] * x[:, None] + ref.get("opd", 0.0)
    return ref.get("amp", 1.0) * np.exp(1j * (2 * np.pi * path / wl + ref.get("phase", 0.0))) \
        * np.ones((n, n)) / n ** 2


# n, m, wavelengths: the stage-1 kernel (rows x columns) and the stage-2 rows they take
PSF = [(1, 1, 1), (2, 3, 1), (3, 2, 2), (16, 33, 1), (31, 64, 3), (33, 17, 2), (64, 40, 3),
       (65, 129, 2), (130, 101, 17),            # 16 x 32, 32 rows
       (400, 60, 64),                           # 32 x 32
       (130, 100, 66), (136, 100, 64),          # 32 x 64 (and a second chunk of two)
       (200, 150, 40), (202, 131, 40),          # 32 x 128, 64 rows
       (130, 270, 40),                          # 32 x 64 (float32) or 32 x 128 (split)
       (128, 600, 2), (130, 600, 14), (200, 600, 16),   # folded pupil in memory, 32 / 64 / 128
       (40, 600, 2)]                            # in the loader: no room for the folded pupil


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("n,m,nwl", PSF)
def test_psf_sizes(rt, n, m, nwl, prec):
    print(f"[fold-psf] n={n} m={m} nwl={nwl} {prec}", flush=True)
    dev, ref = _planes(n, "amp opd", n + m, 0)
    wls, w = np.linspace(0.8e-6, 1.2e-6, nwl), np.linspace(0.5, 1.5, nwl)
    out = rt.psf_poly(n, m, wls, w, 1.0 / n, P_OUT, scale=1.0 / n ** 2, precision=prec, **dev)
    exact = sum(wi * np.abs(orc.mft(_pupil(n, ref, wl, (0, 0)), wl, 1.0 / n, m, P_OUT)) ** 2
                for wl, wi in zip(wls, w))
    assert _err(out, exact) < 12 * _sigma(n, prec)


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("tilt", [(0.0, 0.0), (3e-7, -2e-7)])
@pytest.mark.parametrize("planes,n,offset", [("amp opd", 72, 1), ("amp opd", 67, 0), ("amp", 72, 0),
                                             ("opd", 72, 0), ("opd", 67, 2), ("none", 40, 0),
                                             ("phase", 72, 0), ("amp opd phase", 67, 1)])
def test_psf_loaders(rt, planes, n, offset, tilt, prec):
    print(f"[fold-loader] {planes} n={n} offset={offset} tilt={tilt} {prec}", flush=True)
    dev, ref = _planes(n, planes, n, offset)
    m, wls = 45, np.array([0.9e-6, 1.1e-6])
    out = rt.psf_poly(n, m, wls, [0.4, 0.6], 1.0 / n, P_OUT, scale=1.0 / n ** 2, precision=prec,
                      tilt=tilt, **dev)
    exact = sum(wi * np.abs(orc.mft(_pupil(n, ref, wl, tilt), wl, 1.0 / n, m, P_OUT)) ** 2
                for wl, wi in zip(wls, (0.4, 0.6)))
    assert _err(out, exact) < 12 * _sigma(n, prec)


# n, m, wavelengths, offset of the planes in floats
PHASE = [(64, 40, 3, 0), (61, 40, 3, 0), (64, 40, 3, 1),   # loader, 16 x 32: runs and single values
         (400, 60, 64, 0), (136, 100, 64, 0), (130, 100, 66, 0),   # 32 x 32, 32 x 64
         (200, 150, 40, 0), (202, 131, 40, 0),                     # 32 x 128
         (300, 101, 5, 0), (512, 128, 2, 1), (264, 280, 2, 0)]     # folded pupil in memory


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("planes", ["amp opd phase", "phase", "none"])
@pytest.mark.parametrize("n,m,nwl,offset", PHASE)
def test_phase_and_missing_planes(rt, n, m, nwl, offset, planes, prec):
    """Pupils outside the fast loader, at every width and written first."""
    print(f"[fold-phase] {planes} n={n} m={m} nwl={nwl} offset={offset} {prec}", flush=True)
    dev, ref = _planes(n, planes, n + m, offset)
    wls, w = np.linspace(0.8e-6, 1.2e-6, nwl), np.linspace(0.5, 1.5, nwl)
    tilt = (3e-7, -2e-7) if nwl % 2 else (0.0, 0.0)
    out = rt.psf_poly(n, m, wls, w, 1.0 / n, P_OUT, scale=1.0 / n ** 2, tilt=tilt, precision=prec,
                      **dev)
    exact = sum(wi * np.abs(orc.mft(_pupil(n, ref, wl, tilt), wl, 1.0 / n, m, P_OUT)) ** 2
                for wl, wi in zip(wls, w))
    assert _err(out, exact) < 12 * _sigma(n, prec)


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("shifted", [False, True])
@pytest.mark.parametrize("n,m,b", [(1, 2, 1), (5, 3, 2), (33, 31, 2), (72, 45, 3), (130, 100, 66),
                                   (400, 60, 64), (200, 150, 40), (202, 131, 40), (40, 600, 1)])
def test_mft_sizes(rt, n, m, b, shifted, prec):
    print(f"[fold-mft] n={n} m={m} b={b} shifted={shifted} {prec}", flush=True)
    rng = np.random.default_rng(n + m)
    f = (rng.uniform(0.5, 1, (b, n, n)) * np.exp(0.2j * rng.standard_normal((b, n, n)))
         / n ** 2).astype(np.complex64)
    wls = np.linspace(0.8e-6, 1.2e-6, b)
    sx, sy = (rng.uniform(-3, 3, b), rng.uniform(-3, 3, b)) if shifted else (np.zeros(b),) * 2
    out = rt.mft(torch.as_tensor(f).cuda(), wls, 1.0 / n, m, P_OUT, shift_x=sx, shift_y=sy,
                 precision=prec).cpu().numpy()
    for i in sorted({0, b // 2, b - 1}):
        exact = orc.mft(f[i].astype(complex), wls[i], 1.0 / n, m, P_OUT, shift=(sx[i], sy[i]))
        assert _err(out[i], exact) < 8 * _sigma(n, prec)


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
@pytest.mark.parametrize("n,m,nwl", [(2, 3, 1), (33, 17, 2), (64, 40, 3), (131, 100, 5),
                                     (300, 101, 2), (200, 150, 40)])
def test_gradient_sizes(rt, n, m, nwl, prec):
    """dL/dOPD, dL/dphase and dL/damp of a random cotangent against autograd in complex128."""
    print(f"[fold-grad] n={n} m={m} nwl={nwl} {prec}", flush=True)
    dev, ref = _planes(n, "amp opd phase" if nwl == 2 else "amp opd", n + m, 0)
    wls, w = np.linspace(0.8e-6, 1.2e-6, nwl), np.linspace(0.5, 1.5, nwl) / nwl
    g = np.random.default_rng(m).standard_normal((m, m)).astype(np.float32)
    got = rt.psf_poly_vjp(n, m, wls, w, 1.0 / n, P_OUT, torch.as_tensor(g).cuda(),
                          scale=1.0 / n ** 2, precision=prec, need_phase=True, need_amp=True, **dev)
    leaf = {k: torch.zeros((n, n), dtype=torch.float64) + torch.as_tensor(
        ref.get(k, np.zeros((n, n)))) for k in ("opd", "phase", "amp")}
    for t in leaf.values():
        t.requires_grad_()
    loss = 0.0
    for wl, wi in zip(wls, w):
        P = leaf["amp"] / n ** 2 * torch.exp(1j * (2 * np.pi / wl * leaf["opd"] + leaf["phase"]))
        W = torch.as_tensor(orc.transfer_matrix(wl, n, 1.0 / n, m, P_OUT).T.copy())
        c = orc.calc_nfringes(wl, n, 1.0 / n, m, P_OUT) / (n * m)
        E = c * (W @ P @ W.T)
        loss = loss + wi * torch.sum(torch.as_tensor(g.astype(np.float64)) * E.abs() ** 2)
    loss.backward()
    for x, k in zip(got, ("opd", "phase", "amp")):
        # four contractions, incoherent against the cotangent: sqrt(2) more terms, no common peak
        assert _err(x, leaf[k].grad.numpy()) < 24 * np.sqrt(2) * _sigma(1, prec) / np.sqrt(min(n, m)) \
            + 12 * _sigma(n, "fp32"), k


def test_batch_partial_groups(rt):
    """Every tile width with shared fields, so groups of 4, 2 and 1 tiles are left partly filled."""
    print("[fold-batch]", flush=True)
    rng = np.random.default_rng(3)
    inst, exact = [], {}
    for o, (n, m, k) in enumerate([(16, 20, 1), (33, 20, 5), (130, 64, 6), (130, 100, 3),
                                   (200, 130, 2), (33, 260, 3), (200, 64, 9), (1, 1, 1)]):
        f = (rng.uniform(0.5, 1, (n, n)) * np.exp(0.2j * rng.standard_normal((n, n)))
             / n ** 2).astype(np.complex64)
        t = torch.as_tensor(f).cuda()
        for _ in range(k):
            wl, wt = float(rng.uniform(0.8e-6, 1.2e-6)), float(rng.uniform(0.5, 1.5))
            sh = tuple(rng.uniform(-2, 2, 2)) if rng.random() < 0.7 else (0.0, 0.0)
            inst.append(dict(field=t, wavelength=wl, n_out=m, pixel_scale_in=1.0 / n,
                             pixel_scale_out=P_OUT, shift=sh, weight=wt, out_index=o))
            E = orc.mft(f.astype(complex), wl, 1.0 / n, m, P_OUT, shift=sh)
            exact[o] = exact.get(o, 0.0) + wt * np.abs(E) ** 2
    for _ in range(2):   # tables generated, then from the cache
        for o, x in enumerate(rt.mft_batched_psf(inst, n_outputs=len(exact))):
            n = [d["field"].shape[0] for d in inst if d["out_index"] == o][0]
            assert _err(x, exact[o]) < 12 * _sigma(n, "bf16x3"), o


@pytest.mark.parametrize("prec", ["fp32", "bf16x3"])
def test_noalloc_smallest_pupil_largest_image(rt, prec):
    """A geometry whose plain buffers fit the 64 MiB array and whose padded ones exceed it."""
    import ctypes
    from dlux_amd import _lib
    n, m = 2, 4050
    print(f"[fold-noalloc] n={n} m={m} {prec}", flush=True)
    dev, _ = _planes(n, "amp opd", 5, 0)
    wls, w = np.array([0.9e-6, 1.1e-6]), np.array([0.4, 0.6])
    ref = rt.psf_poly(n, m, wls, w, 1.0 / n, P_OUT, scale=0.25, precision=prec, **dev)
    out = torch.full((m, m), float("nan"), device="cuda")
    g = rt.geom(n, m)
    st = _lib.load().dlx_psf_poly_noalloc(
        ctypes.byref(g), 2, _lib.dptr(wls), _lib.dptr(w), 1.0 / n, P_OUT, 0.0, 0.0, 0.0,
        dev["amp"].data_ptr(), dev["opd"].data_ptr(), None, 0.25, out.data_ptr(),
        rt._prec_code(prec), rt.stream_handle())
    _lib.check(st, "dlx_psf_poly_noalloc")
    assert _err(out, ref.double().cpu().numpy()) < 12 * _sigma(n, prec)


def _unfolded_split(f, wl, m, shift):
    """The transform as split operands of the unfolded complex form give it: the
    field, the kernels and the intermediate each hi + lo in bf16, products hi hi
    + hi lo + lo hi, sums in 64 bits."""
    def split(x):
        x = x.float()
        hi = x.bfloat16().float()
        return hi.double(), (x - hi).bfloat16().double()

    def real_nt(a, b):
        (ah, al), (bh, bl) = split(a), split(b)
        return al @ bh.T + ah @ bl.T + ah @ bh.T

    def nt(a, b):
        return torch.complex(real_nt(a.real, b.real) - real_nt(a.imag, b.imag),
                             real_nt(a.real, b.imag) + real_nt(a.imag, b.real))

    n = f.shape[-1]
    wx, wy = (torch.as_tensor(orc.transfer_matrix(wl, n, 1.0 / n, m, P_OUT, shift=s).T.copy()).cuda()
              for s in shift)
    c = orc.calc_nfringes(wl, n, 1.0 / n, m, P_OUT) / (n * m)
    return c * nt(wy, nt(f, wx).T)


@pytest.mark.parametrize("white", [False, True])
@pytest.mark.parametrize("n,m,shift", [(64, 64, (10.0, -7.0)), (256, 256, (20.0, -30.0)),
                                       (131, 101, (0.0, 0.0))])
def test_split_error_not_above_the_unfolded_form(rt, n, m, shift, white):
    """The folds add mirrored values before the split, so its rounding errors
    meet at the peak; the products and the tables must make up for that.  Rms
    over fields of the 2-norm error of the field and of its intensity against
    complex128, beside that of the unfolded split form with exact sums."""
    print(f"[fold-split-error] n={n} m={m} shift={shift} white={white}", flush=True)
    x = (torch.arange(n, device="cuda") - (n - 1) / 2) / n * 2
    yy, xx = torch.meshgrid(x, x, indexing="ij")
    err = torch.zeros(2, 2, dtype=torch.float64)
    for seed in range(6):
        g = torch.Generator(device="cuda").manual_seed(seed)
        if white:
            f = torch.complex(*torch.randn((2, n, n), generator=g, device="cuda")) / n ** 2
        else:
            c = 0.2 * torch.randn(5, generator=g, device="cuda")
            ph = c[0] * xx + c[1] * yy + c[2] * (2 * xx ** 2 - 1) + c[3] * xx * yy + c[4] * yy ** 3
            f = torch.polar((xx ** 2 + yy ** 2 < 1).float() / n ** 2, ph)
        wl = 0.8e-6 + 0.07e-6 * seed
        ref = torch.as_tensor(orc.mft(f.cpu().numpy().astype(complex), wl, 1.0 / n, m, P_OUT,
                                      shift=shift)).cuda()
        got = rt.mft(f, wl, 1.0 / n, m, P_OUT, shift_x=shift[0], shift_y=shift[1],
                     precision="bf16x3")
        plain = _unfolded_split(f.to(torch.complex128), wl, m, shift)
        for i, e in enumerate((got.to(torch.complex128), plain)):
            for j, (a, b) in enumerate(((e, ref), (e.abs() ** 2, ref.abs() ** 2))):
                err[i, j] += float(torch.linalg.vector_norm(a - b) / torch.linalg.vector_norm(b)) ** 2
    err = (err / 6).sqrt()
    print(err.tolist(), flush=True)
    assert bool((err[0] <= err[1]).all())
