"""GPU: gridding on the full 3-D grid (trajectories that are not stacks of
2-D ones) against the FP64 restatement (oracle): every chunk width of the
patch spread, patches summed in parts, runs of patches without a sample,
ragged items, windows past the grid's edges, 6, 8 and 12 taps, and few samples
on a large grid (the gather).

Tolerance 2e-6: FP32 sums of products of three taps (each rounded, eps = 6e-8)
and a 3-D FFT, below 1e-6 in relative 2-norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 2e-6


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def _traj(rng, N, Nz, M, centre):
    k = [rng.uniform(-N / 2, N / 2, M), rng.uniform(-N / 2, N / 2, M),
         rng.uniform(-Nz / 2, Nz / 2, M)]
    for a in k:
        a[:int(centre * M)] *= 0.05  # crowd the central patches
        a[-1] = -N / 2 - 1.7 if a is k[0] else a[-1]  # a window partly off the grid
    k[1][-2] = N  # and one wholly off it
    return [a.astype(np.float32) for a in k]


def _complex(rng, *shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)


@pytest.mark.parametrize("N,Nz,M,nc,L,width,centre", [
    (12, 10, 301, 1, 1, 4.0, 0.0), (12, 10, 301, 4, 2, 4.0, 0.0), (12, 10, 301, 9, 1, 4.0, 0.0),
    (12, 10, 65, 8, 2, 4.0, 0.0), (12, 10, 301, 17, 1, 4.0, 0.0), (12, 10, 301, 33, 1, 4.0, 0.0),
    (10, 4, 97, 13, 5, 3.0, 0.2), (16, 16, 5000, 6, 3, 4.0, 0.5), (16, 16, 9000, 3, 1, 4.0, 0.5),
    # most patches met by no sample, in every chunk width; the last two gathered
    (26, 20, 100, 3, 1, 4.0, 0.8), (26, 20, 100, 11, 1, 4.0, 0.8), (26, 20, 100, 7, 5, 4.0, 0.8),
    (22, 24, 100, 4, 3, 3.0, 0.8), (32, 32, 600, 12, 1, 4.0, 0.0), (32, 32, 600, 24, 2, 3.0, 0.0)])
def test_operator(orc, N, Nz, M, nc, L, width, centre):
    import powergrid_amd as P
    rng = np.random.default_rng(M + nc)
    k = _traj(rng, N, Nz, M, centre)
    n = N * N * Nz
    t = np.linspace(1e-3, 9e-3, M).astype(np.float32)
    fm = rng.uniform(-300, 300, n).astype(np.float32)
    sens, x, y = _complex(rng, nc, n), _complex(rng, n), _complex(rng, nc * M)
    Gg = P.Gnufft(M, 2.0, N, N, Nz, *k, kernel_width=width)
    assert P.zclasses(Gg) == 0
    A = P.SENSE(P.TimeSegmentation(Gg, fm, t, M, n, L), sens, M, n, nc)
    G = orc.Gnufft(M, 2.0, N, N, Nz, *k, width, prec="d")
    O = orc.SENSE(orc.TimeSegmentation(G, fm, t, M, n, L), sens.astype(complex).ravel(), M, n, nc)
    assert _rel(A * x, O * x.astype(complex)) < TOL
    assert _rel(A / y, O / y.astype(complex)) < TOL
    assert np.array_equal(A / y, A / y)  # deterministic


@pytest.mark.parametrize("gridos,width", [(2.0, 4.0), (2.0, 3.0), (3.0, 4.0)])
def test_spatial_interpolation(orc, gridos, width):
    import powergrid_amd as P
    rng = np.random.default_rng(3)
    N, Nz, M = 12, 8, 400
    k = _traj(rng, N, Nz, M, 0.3)
    Gg = P.Gnufft(M, gridos, N, N, Nz, *k, kernel_width=width)
    grid, d = _complex(rng, Gg.grid_size), _complex(rng, M)
    geo = (*k, N, N, Nz)
    assert _rel(Gg.forwardSpatialInterp(grid),
                orc.grid_forward(grid.astype(complex), *geo, gridos, width)) < TOL
    assert _rel(Gg.adjointSpatialInterp(d),
                orc.grid_adjoint(d.astype(complex), *geo, Gg.grid_size, gridos, width)) < TOL


@pytest.mark.parametrize("gridos,width", [(2.0, 4.0), (2.0, 3.0), (3.0, 4.0)])
def test_values_not_finite(orc, gridos, width):
    """reach the points of their windows alone, in patches summed whole and in
    parts; the others keep their sums"""
    import powergrid_amd as P
    rng = np.random.default_rng(4)
    N, Nz, M = 12, 8, 1500
    k = _traj(rng, N, Nz, M, 0.5)
    d = _complex(rng, M)
    d[3], d[700], d[1000], d[1300] = np.nan, 1 + 1j * np.inf, -np.inf, 2 + 1j * np.nan
    Gg = P.Gnufft(M, gridos, N, N, Nz, *k, kernel_width=width)
    x = Gg.adjointSpatialInterp(d)
    ref = orc.grid_adjoint(d.astype(complex), *k, N, N, Nz, Gg.grid_size, gridos, width)
    for a, b in ((x.real, ref.real), (x.imag, ref.imag)):
        ok = np.isfinite(b)
        assert 0 < ok.sum() < ok.size
        assert np.array_equal(np.isnan(a), np.isnan(b))
        assert np.array_equal(a[np.isinf(b)], b[np.isinf(b)])
        assert _rel(a[ok], b[ok]) < TOL


def test_dense_plan(orc):
    """more than 8.4 million (sample, patch) entries: longer parts, and a
    workspace of at most 65536 partial patches (16 KB for 32 grids each; one for
    every 256 entries would be 5.2 GB here)"""
    import powergrid_amd as P
    from powergrid_amd import serve
    rng = np.random.default_rng(11)
    N, M = 16, 600_000
    k = [rng.uniform(-N / 2, N / 2, M).astype(np.float32) for _ in range(3)]
    d = _complex(rng, M)
    Gg = P.Gnufft(M, 2.0, N, N, N, *k)
    ref = orc.grid_adjoint(d.astype(complex), *k, N, N, N, Gg.grid_size, 2.0, 4.0)
    assert _rel(Gg.adjointSpatialInterp(d), ref) < TOL
    del Gg
    M = 4_000_000
    k = [rng.uniform(-N / 2, N / 2, M).astype(np.float32) for _ in range(3)]
    free = serve.mem_info()[0]
    A = P.SENSE(P.Gnufft(M, 2.0, N, N, N, *k), _complex(rng, 8, N ** 3), M, N ** 3, 8)
    A / np.ones(8 * M, np.complex64)
    assert free - serve.mem_info()[0] < 4 << 30


def test_many_blocks():
    """more (tile, coil) blocks than one launch can have"""
    import powergrid_amd as P
    rng = np.random.default_rng(13)
    N, M, nc = 8, 2_200_000, 256
    k = [rng.uniform(-N / 2, N / 2, M).astype(np.float32) for _ in range(3)]
    n = N ** 3
    G = P.Gnufft(M, 2.0, N, N, N, *k)
    maps, x = _complex(rng, 4, n), _complex(rng, n)
    ref = (P.SENSE(G, maps, M, n, 4) * x).reshape(4, M)
    y = (P.SENSE(G, np.tile(maps, (nc // 4, 1)), M, n, nc) * x).reshape(nc, M)
    for c in (*range(8), *range(nc - 8, nc)):
        assert np.array_equal(y[c], ref[c % 4])
