"""GPU: the register FFT passes of grid lengths that are not powers of two,
against the FP64 restatement (oracle), every supported length.

Tolerance: an FP32 FFT of length n has a relative error of about
eps log2(n) / 2 (eps = 6e-8), twice for a 2-D grid and three times for a 3-D
one, plus the taps' rounding: below 1e-6 for n <= 480; 2e-6 is asserted."""
import re
from pathlib import Path

import numpy as np
import pytest


pytestmark = pytest.mark.gpu
HEADER = Path(__file__).resolve().parents[1] / "powergrid_amd" / "csrc" / "pg_fftmix.h"
LENGTHS = [int(a) for a in re.findall(r"\bf\((\d+),", HEADER.read_text())]
TOL = 2e-6


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def _check(orc, N, Nz, M, nc, L, seed):
    import powergrid_amd as P
    rng = np.random.default_rng(seed)
    kx, ky = (rng.uniform(-N / 2, N / 2 - 1e-2, M).astype(np.float32) for _ in range(2))
    kz = rng.uniform(-Nz / 2, Nz / 2 - 1e-2, M).astype(np.float32) if Nz > 1 \
        else np.zeros(M, np.float32)
    t = np.linspace(1e-3, 9e-3, M).astype(np.float32)
    n = N * N * Nz
    fm = rng.uniform(-300, 300, n).astype(np.float32)
    sens = (rng.standard_normal((nc, n)) + 1j * rng.standard_normal((nc, n))).astype(np.complex64)
    x = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)
    y = (rng.standard_normal(nc * M) + 1j * rng.standard_normal(nc * M)).astype(np.complex64)
    A = P.SENSE(P.TimeSegmentation(P.Gnufft(M, 2.0, N, N, Nz, kx, ky, kz), fm, t, M, n, L), sens,
                M, n, nc)
    G = orc.Gnufft(M, 2.0, N, N, Nz, kx, ky, kz, prec="d")
    O = orc.SENSE(orc.TimeSegmentation(G, fm, t, M, n, L), sens.astype(complex).ravel(), M, n, nc)
    assert _rel(A * x, O * x.astype(complex)) < TOL
    assert _rel(A / y, O / y.astype(complex)) < TOL


@pytest.mark.parametrize("n", LENGTHS)
def test_every_length(orc, n):
    # one coil and segment (several columns a block), and more segments than
    # a block of the adjoint y pass holds lines
    _check(orc, n // 2, 1, 61, 1, 1, n)
    if n <= 120:
        _check(orc, n // 2, 1, 61, 2, 9, n + 1)


@pytest.mark.parametrize("N,Nz", [(12, 10), (18, 14), (20, 6), (26, 8)])
def test_three_dimensions(orc, N, Nz):
    _check(orc, N, Nz, 83, 3, 2, N)


# image sizes of both kinds of y FFT, Nz up to and past the matrix-core z
# stage's 32; the last has more planes (512 coils x 16 segments x 10) than one
# grid dimension holds
@pytest.mark.parametrize("N,Nz,nc,L", [(12, 8, 8, 2), (20, 36, 4, 4), (8, 10, 5, 4),
                                       (10, 10, 512, 16)])
def test_stack_planes(orc, N, Nz, nc, L):
    import powergrid_amd as P
    rng = np.random.default_rng(N)
    m = 7
    kx, ky = (rng.uniform(-N / 2, N / 2 - 1e-2, m * Nz).astype(np.float32) for _ in range(2))
    kz = np.repeat(np.arange(Nz) - Nz / 2.0, m).astype(np.float32)
    M, n = m * Nz, N * N * Nz
    t = np.linspace(1e-3, 9e-3, M).astype(np.float32)
    fm = rng.uniform(-300, 300, n).astype(np.float32)
    sens = (rng.standard_normal((nc, n)) + 1j * rng.standard_normal((nc, n))).astype(np.complex64)
    x = (rng.standard_normal(n) + 1j * rng.standard_normal(n)).astype(np.complex64)
    y = (rng.standard_normal(nc * M) + 1j * rng.standard_normal(nc * M)).astype(np.complex64)
    Gg = P.Gnufft(M, 2.0, N, N, Nz, kx, ky, kz)
    assert P.zclasses(Gg) == Nz
    A = P.SENSE(P.TimeSegmentation(Gg, fm, t, M, n, L), sens, M, n, nc)
    G = orc.Gnufft(M, 2.0, N, N, Nz, kx, ky, kz, prec="d")
    O = orc.SENSE(orc.TimeSegmentation(G, fm, t, M, n, L), sens.astype(complex).ravel(), M, n, nc)
    assert _rel(A * x, O * x.astype(complex)) < TOL
    assert _rel(A / y, O / y.astype(complex)) < TOL
