"""Every transform length of the LDS FFT (2 to 8192: one to four stages, radices
2 to 16, one to eight rows per workgroup, padded rows skipped or, as in unpadded
fields and those whose half is no multiple of the row count, not) against
complex128 transforms.

Bound: a Cooley-Tukey transform of M points in unit roundoff u = 2^-24 has a
2-norm error below log2(M) eta with eta = mu + gamma_4 (sqrt 2 + mu) < 8 u per
radix-2 level (mu <= u: twiddles rounded from double), and higher radices round
less; a 2-D transform has 2 log2(M) levels.  The angular spectrum runs two of
them with a transfer function of error 1.3e-7 per element between.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

U = 2.0 ** -24


@pytest.fixture(scope="module")
def rt():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dlux_amd import runtime
    return runtime


def _field(b, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.complex(*torch.randn((2, b, n, n), generator=g, device="cuda")).contiguous()


def _pad(x, m):
    p = (m - x.shape[-1]) // 2
    return torch.nn.functional.pad(x, (p, p, p, p))


def _shift(x, inverse=False):
    f = torch.fft.ifftshift if inverse else torch.fft.fftshift
    return f(x, dim=(-2, -1))


def _rel(x, ref):
    return float(torch.linalg.vector_norm(x.to(ref.dtype) - ref) / torch.linalg.vector_norm(ref))


SIZES = [(2, 2), (2, 4), (4, 8), (6, 16), (20, 32), (64, 64), (96, 128), (130, 256),
         (254, 256), (256, 256), (256, 512), (300, 512), (512, 512), (512, 1024),
         (1000, 1024), (1024, 1024), (1024, 2048), (600, 2048), (1002, 2048), (2048, 2048),
         (2048, 4096), (130, 8192)]


@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("n,m", SIZES)
def test_fft2_every_length(rt, n, m, inverse):
    print(f"[fft-size] n={n} m={m} inverse={inverse}", flush=True)
    x = _field(2 if m <= 2048 else 1, n, n + m)
    out = rt.fft2(x, m, inverse=inverse)
    z = _shift(_pad(x.to(torch.complex128), m), inverse=True)
    ref = _shift(torch.fft.ifft2(z) * m if inverse else torch.fft.fft2(z) / m)
    assert _rel(out, ref) < 2 * np.log2(m) * 8 * U


@pytest.mark.parametrize("n,m", SIZES)
def test_asm_every_length(rt, n, m):
    print(f"[asm-size] n={n} m={m}", flush=True)
    x = _field(1, n, n + m)
    wl, dx, z = 1e-6, 3e-6, 0.01
    out = rt.asm_prop(x, [wl], dx, z, m)
    f = torch.fft.fftfreq(m, dx, dtype=torch.float64, device="cuda")
    arg = 1 / wl ** 2 - f[None, :] ** 2 - f[:, None] ** 2
    t = z * torch.sqrt(arg.clamp(min=0))
    h = torch.where(arg > 0, torch.polar(torch.ones_like(t), 2 * np.pi * (t - torch.round(t))), 0)
    spec = torch.fft.fft2(_shift(_pad(x.to(torch.complex128), m), inverse=True))
    ref = _shift(torch.fft.ifft2(spec * h))
    assert _rel(out, ref) < 4 * np.log2(m) * 8 * U + 1.3e-7


def _rnd(x):
    return x.float().double()


def _fma(a, b, c):
    return _rnd(a * b + c)


def _dft4(x, sgn):
    a0, a1 = _rnd(x[0] + x[2]), _rnd(x[0] - x[2])
    a2, d = _rnd(x[1] + x[3]), _rnd(x[1] - x[3])
    a3 = torch.stack([-sgn * d[1], sgn * d[0]])
    return [_rnd(a0 + a2), _rnd(a1 + a3), _rnd(a0 - a2), _rnd(a1 - a3)]


def _rows_radix8(x, sgn):
    """The transform of rows (real and imaginary planes first) in radix-8 stages and
    one of the rest, float32 arithmetic with fused multiply-adds, twiddles rounded
    from double."""
    m, p = x.shape[-1], 1
    h = _rnd(torch.tensor(0.5, dtype=torch.float64, device=x.device).sqrt())
    while p < m:
        rad = min(8, m // p)
        n = m // rad
        j = torch.arange(n, device=x.device)
        k = j % p
        v = [x[..., r * n:(r + 1) * n] for r in range(rad)]
        for r in range(1, rad if p > 1 else 1):
            t = 2 * np.pi * (r * k).double() / (p * rad)
            c, s = _rnd(torch.cos(t)), _rnd(sgn * torch.sin(t))
            v[r] = torch.stack([_fma(v[r][0], c, -_rnd(v[r][1] * s)),
                                _fma(v[r][0], s, _rnd(v[r][1] * c))])
        if rad == 2:
            y = [_rnd(v[0] + v[1]), _rnd(v[0] - v[1])]
        elif rad == 4:
            y = _dft4(v, sgn)
        else:
            e, o = _dft4(v[0::2], sgn), _dft4(v[1::2], sgn)
            t1 = _rnd(torch.stack([o[1][0] - sgn * o[1][1], o[1][1] + sgn * o[1][0]]))
            t2 = torch.stack([-sgn * o[2][1], sgn * o[2][0]])
            t3 = _rnd(torch.stack([-o[3][0] - sgn * o[3][1], sgn * o[3][0] - o[3][1]]))
            y = [_rnd(e[0] + o[0]), _fma(t1, h, e[1]), _rnd(e[2] + t2), _fma(t3, h, e[3]),
                 _rnd(e[0] - o[0]), _fma(-t1, h, e[1]), _rnd(e[2] - t2), _fma(-t3, h, e[3])]
        out = torch.empty_like(x)
        for q in range(rad):
            out[..., (j - k) * rad + k + q * p] = y[q]
        x, p = out, p * rad
    return x


@pytest.mark.parametrize("m", [128, 256, 1024, 2048, 4096])
def test_fft2_error_not_above_radix8(rt, m):
    """Wider radices save passes through LDS, not digits: the error against
    complex128 is no larger than that of the same transform in radix-8 stages (the
    rms of 2 m^2 errors has a standard error of 1 / (2 m), the ratio of two sqrt(2)
    of it: three of those)."""
    print(f"[fft-radix8] m={m}", flush=True)
    x = _field(1, m, m)[0]
    z = _shift(x.to(torch.complex128), inverse=True)
    ref = torch.fft.fft2(z)
    r = torch.stack([z.real, z.imag])
    r = _rows_radix8(_rows_radix8(r, -1.0).transpose(1, 2).contiguous(), -1.0).transpose(1, 2)
    plain = _rel(torch.complex(r[0].contiguous(), r[1].contiguous()), ref)
    got = _rel(rt.fft2(x, m), _shift(ref) / m)
    print(got, plain, flush=True)
    assert got <= plain * (1 + 1.5 * np.sqrt(2) / m)
