"""GPU: the 2-D spread on the matrix cores against the FP64 restatement
(oracle): every width of its coil chunks and remainder of its segment chunks,
complex segment weights, value rows (no segments, or few coils of several),
patches of one to eight wavefronts and in parts, grids whose rows end in a
partial strip, and, of every width and kind of rows, grids large enough for
the rows gathered in LDS.

Tolerance 2e-6: FP32 sums of products of two taps and a weight (each rounded,
eps = 6e-8) and a 2-D FFT, below 1e-6 in relative 2-norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 2e-6


def _complex(rng, *shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)


@pytest.mark.parametrize("N,M,nc,L,interp,centre", [
    (16, 300, 1, 1, 1, 0.0), (16, 300, 5, 3, 1, 0.0), (18, 300, 8, 4, 1, 0.3),
    (16, 300, 9, 5, 1, 0.0), (22, 900, 16, 7, 1, 0.6), (16, 300, 17, 1, 1, 0.0),
    (16, 300, 17, 3, 1, 0.0), (16, 300, 33, 2, 1, 0.0), (16, 300, 40, 1, 1, 0.0),
    (16, 300, 3, 4, 2, 0.0), (16, 300, 11, 3, 2, 0.0), (16, 300, 19, 4, 3, 0.0),
    (16, 9000, 4, 2, 1, 0.7), (66, 2000, 33, 16, 1, 0.2), (110, 1500, 7, 24, 1, 0.5),
    # value rows for few coils of several segments, real and complex weights
    (16, 300, 1, 8, 1, 0.0), (16, 300, 11, 5, 1, 0.3), (16, 300, 17, 12, 1, 0.0),
    (16, 300, 2, 7, 2, 0.0),
    # gathered: values in two and four column tiles, compact rows in one, two
    # and four, with real and complex weights
    (182, 2000, 16, 1, 1, 0.3), (64, 2000, 40, 4, 1, 0.3), (210, 2000, 8, 9, 1, 0.3),
    (110, 1500, 16, 11, 1, 0.3), (66, 2000, 32, 17, 1, 0.3), (210, 2000, 8, 9, 2, 0.3),
    (110, 1500, 16, 11, 2, 0.3), (66, 2000, 64, 9, 2, 0.3)])
def test_adjoint(orc, N, M, nc, L, interp, centre):
    import powergrid_amd as P
    rng = np.random.default_rng(M + nc + L)
    kx, ky = rng.uniform(-N / 2, N / 2, M), rng.uniform(-N / 2, N / 2, M)
    kx[:int(centre * M)] *= 0.08  # crowd the central patches
    ky[:int(centre * M)] *= 0.08
    kx, ky, kz = kx.astype(np.float32), ky.astype(np.float32), np.zeros(M, np.float32)
    n = N * N
    t = np.linspace(1e-3, 9e-3, M).astype(np.float32)
    # (min-max weights of many segments are determined by many turns only)
    turn = 700 if interp == 1 or L < 7 else 4000
    fm = rng.uniform(-turn, turn, n).astype(np.float32)
    sens, y = _complex(rng, nc, n), _complex(rng, nc * M)
    A = P.SENSE(P.TimeSegmentation(P.Gnufft(M, 2.0, N, N, 1, kx, ky, kz), fm, t, M, n, L,
                                   interptype=interp), sens, M, n, nc)
    G = orc.Gnufft(M, 2.0, N, N, 1, kx, ky, kz, prec="d")
    O = orc.SENSE(orc.TimeSegmentation(G, fm, t, M, n, L, interptype=interp),
                  sens.astype(complex).ravel(), M, n, nc)
    x = A / y
    orc.set_threads(8)
    try:
        ref = O / y.astype(complex)
    finally:
        orc.set_threads(1)
    assert np.linalg.norm(x - ref) / np.linalg.norm(ref) < TOL
    assert np.array_equal(x, A / y)  # deterministic


@pytest.mark.parametrize("M", [300, 301, 302, 303])
def test_infinite_sample(orc, M):
    """the spatial spread of an infinite sample is infinite in its window, also
    where it is the last entry of a patch"""
    import powergrid_amd as P
    rng = np.random.default_rng(M)
    N = 16
    kx, ky = (rng.uniform(-N / 2, N / 2, M).astype(np.float32) for _ in range(2))
    kz = np.zeros(M, np.float32)
    d = _complex(rng, M)
    d[-1], kx[-1], ky[-1] = np.inf + 1j, 0.3, -0.7
    G = P.Gnufft(M, 2.0, N, N, 1, kx, ky, kz)
    x = G.adjointSpatialInterp(d).real
    ref = orc.grid_adjoint(d.astype(complex), kx, ky, kz, N, N, 1, G.grid_size, 2.0, 4.0).real
    assert np.isinf(ref).sum() == 64
    assert np.array_equal(x[np.isinf(ref)], ref[np.isinf(ref)])
