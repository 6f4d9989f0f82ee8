"""GPU: interpolation by patches on the matrix cores against the FP64
restatement (oracle): each width of its coil chunks with partial last ones,
odd and even segment counts, complex segment weights, patches of one to
several wavefronts, samples at the grid's edges, class planes, and the calls
that it does not serve (fewer coils, segments or samples: the tiled form).  It
is asked for wherever it can serve (interp_lds4 3): at these sizes the tiles
are the faster form, as the last test shows.

Tolerance 2e-6: FP32 sums of products of two taps, a grid value and a weight
(each rounded, eps = 6e-8) after a 2-D FFT, below 1e-6 in relative 2-norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 2e-6


def _complex(rng, *shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)


@pytest.mark.parametrize("N,Nz,M,nc,L,interp,centre,patches", [
    (32, 1, 900, 8, 8, 1, 0.0, True), (30, 1, 900, 9, 9, 1, 0.3, True),
    (32, 1, 900, 16, 6, 1, 0.0, True), (26, 1, 600, 17, 7, 1, 0.0, True),
    (32, 1, 650, 33, 6, 1, 0.5, True), (32, 1, 900, 8, 11, 2, 0.0, True),
    (32, 1, 900, 12, 6, 2, 0.4, True), (26, 1, 600, 32, 7, 3, 0.0, True),
    (16, 8, 1800, 8, 8, 1, 0.2, True), (32, 1, 900, 7, 10, 1, 0.0, False),
    (32, 1, 900, 16, 5, 1, 0.0, False), (32, 1, 300, 8, 8, 1, 0.0, False),
    (16, 1, 3000, 8, 8, 1, 0.6, False)])
def test_forward(orc, N, Nz, M, nc, L, interp, centre, patches):
    import powergrid_amd as P
    rng = np.random.default_rng(M + nc + L)
    kx, ky = rng.uniform(-N / 2, N / 2, M), rng.uniform(-N / 2, N / 2, M)
    kx[:int(centre * M)] *= 0.2  # crowd the central patches
    ky[:int(centre * M)] *= 0.2
    kx[-1] = -N / 2
    ky[-1] = N / 2
    kz = rng.integers(0, Nz, M) - Nz // 2
    kx, ky, kz = (a.astype(np.float32) for a in (kx, ky, kz))
    n = N * N * Nz
    t = np.linspace(1e-3, 9e-3, M).astype(np.float32)
    # (min-max weights of few turns a segment are not determined: at 700 rad/s
    # and 11 segments the oracle's in FP32 and in FP64 differ by 0.4)
    turn = 700 if interp == 1 else 4000
    fm = rng.uniform(-turn, turn, n).astype(np.float32)
    sens, x = _complex(rng, nc, n), _complex(rng, n)
    A = P.SENSE(P.TimeSegmentation(P.Gnufft(M, 2.0, N, N, Nz, kx, ky, kz), fm, t, M, n, L,
                                   interptype=interp), sens, M, n, nc)
    G = orc.Gnufft(M, 2.0, N, N, Nz, kx, ky, kz, prec="d")
    O = orc.SENSE(orc.TimeSegmentation(G, fm, t, M, n, L, interptype=interp),
                  sens.astype(complex).ravel(), M, n, nc)
    P.set_tuning("interp_lds4", 3)
    try:
        y, again = A * x, A * x
    finally:
        P.set_tuning("interp_lds4", 1)
    orc.set_threads(8)
    try:
        ref = O * x.astype(complex)
    finally:
        orc.set_threads(1)
    assert np.linalg.norm(y - ref) / np.linalg.norm(ref) < TOL
    assert np.array_equal(y, again)  # deterministic
    # which form ran: the tiled one alone differs in its last bits
    P.set_tuning("interp_lds4", 2)
    try:
        tiled = A * x
    finally:
        P.set_tuning("interp_lds4", 1)
    assert np.array_equal(y, tiled) != patches


@pytest.mark.parametrize("M,nc,L,interp,width", [
    (900, 8, 8, 1, 3.0), (900, 16, 6, 2, 3.0), (600, 8, 8, 1, 6.0), (600, 16, 6, 2, 6.0)])
def test_widths(orc, M, nc, L, interp, width):
    """6 taps, and 12, whose windows meet up to 16 patches"""
    import powergrid_amd as P
    rng = np.random.default_rng(M + nc)
    N = 32
    n = N * N
    kx, ky = (rng.uniform(-N / 2, N / 2, M).astype(np.float32) for _ in range(2))
    kz = np.zeros(M, np.float32)
    t = np.linspace(1e-3, 9e-3, M).astype(np.float32)
    fm = rng.uniform(-4000, 4000, n).astype(np.float32)
    sens, x = _complex(rng, nc, n), _complex(rng, n)
    A = P.SENSE(P.TimeSegmentation(P.Gnufft(M, 2.0, N, N, 1, kx, ky, kz, kernel_width=width), fm,
                                   t, M, n, L, interptype=interp), sens, M, n, nc)
    G = orc.Gnufft(M, 2.0, N, N, 1, kx, ky, kz, width, prec="d")
    O = orc.SENSE(orc.TimeSegmentation(G, fm, t, M, n, L, interptype=interp),
                  sens.astype(complex).ravel(), M, n, nc)
    y = {}
    try:
        for form in (3, 2):
            P.set_tuning("interp_lds4", form)
            y[form] = A * x
    finally:
        P.set_tuning("interp_lds4", 1)
    ref = O * x.astype(complex)
    assert not np.array_equal(y[3], y[2])  # by patches
    assert np.linalg.norm(y[3] - ref) / np.linalg.norm(ref) < TOL


def test_form_independent_of_earlier_calls():
    """a batch whose partial sums do not fit its own share of the plan's
    workspace keeps its form, and so its bits, when a larger batch on the same
    plan has grown that workspace"""
    import powergrid_amd as P
    rng = np.random.default_rng(5)
    N, M, nc, L = 32, 1500, 12, 6
    n = N * N
    kx, ky = (rng.uniform(-N / 2, N / 2, M).astype(np.float32) for _ in range(2))
    t = np.linspace(1e-3, 9e-3, M).astype(np.float32)
    fm = rng.uniform(-700, 700, n).astype(np.float32)
    x, sens = _complex(rng, n), _complex(rng, 32, n)
    G = P.Gnufft(M, 2.0, N, N, 1, kx, ky, np.zeros(M, np.float32))
    A = P.SENSE(P.TimeSegmentation(G, fm, t, M, n, L), sens[:nc], M, n, nc)
    P.set_tuning("interp_lds4", 3)
    try:
        fresh = A * x
        P.SENSE(P.TimeSegmentation(G, fm, t, M, n, 8), sens, M, n, 32) * x
        again = A * x
    finally:
        P.set_tuning("interp_lds4", 1)
    assert np.array_equal(again, fresh)


@pytest.mark.parametrize("N,M,nc,L,interp,patches", [
    (64, 4096, 17, 8, 1, False), (64, 8192, 8, 8, 1, False), (128, 16384, 8, 8, 2, False),
    (128, 32768, 8, 8, 1, True), (128, 16384, 16, 6, 1, True), (96, 16384, 32, 12, 2, True)])
def test_rule(N, M, nc, L, interp, patches):
    """which form a batch takes by default; both sides of the rule measured"""
    import powergrid_amd as P
    rng = np.random.default_rng(7)
    n = N * N
    kx, ky = (rng.uniform(-N / 2, N / 2, M).astype(np.float32) for _ in range(2))
    t = np.linspace(1e-3, 9e-3, M).astype(np.float32)
    fm = rng.uniform(-4000, 4000, n).astype(np.float32)
    A = P.SENSE(P.TimeSegmentation(P.Gnufft(M, 2.0, N, N, 1, kx, ky, np.zeros(M, np.float32)),
                                   fm, t, M, n, L, interptype=interp), _complex(rng, nc, n), M, n,
                nc)
    x = _complex(rng, n)
    y = {}
    try:
        for form in (3, 2, 1):
            P.set_tuning("interp_lds4", form)
            y[form] = A * x
    finally:
        P.set_tuning("interp_lds4", 1)
    assert not np.array_equal(y[3], y[2])
    assert np.array_equal(y[1], y[3 if patches else 2])
    assert np.linalg.norm(y[3] - y[2]) / np.linalg.norm(y[2]) < TOL


@pytest.mark.parametrize("L", [1, 2, 4])
def test_many_blocks(L):
    """more (block of samples, coil) blocks than one launch can have: the
    gather, and tiles of all and of four segments"""
    import ctypes as C

    import powergrid_amd as P
    from powergrid_amd._lib import check, lib
    rng = np.random.default_rng(17)
    N, M, nc = 8, 2_200_000, 512
    n = N * N
    kx, ky = (rng.uniform(-N / 2, N / 2, M).astype(np.float32) for _ in range(2))
    G = P.Gnufft(M, 2.0, N, N, 1, kx, ky, np.zeros(M, np.float32))
    if L > 1:
        t = np.linspace(1e-3, 9e-3, M).astype(np.float32)
        G = P.TimeSegmentation(G, rng.uniform(-700, 700, n).astype(np.float32), t, M, n, L)
    maps, x = _complex(rng, 4, n), _complex(rng, n)
    ref = (P.SENSE(G, maps, M, n, 4) * x).reshape(4, M)
    out = P.DeviceArray(nc * M)
    A = P.SENSE(G, np.tile(maps, (nc // 4, 1)), M, n, nc)
    A.forward(P.DeviceArray.from_host(x), out=out)
    y = np.empty(M, np.complex64)
    for c in (0, 1, 250, 490, 510, 511):
        check(lib().pg_memcpy_dtoh(y.ctypes.data_as(C.c_void_p),
                                   C.c_void_p(out.ptr.value + 8 * M * c), 8 * M, None))
        assert np.array_equal(y, ref[c % 4])
