"""Every transform length of the LDS FFT (2 to 8192: one to four stages, radices
2 to 16, one to four rows per workgroup, padded rows skipped or not) against
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
         (256, 512), (300, 512), (512, 1024), (1000, 1024), (1024, 2048), (600, 2048),
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
