"""GPU: the FP32 exact DFT on the matrix cores (Gdft and GdftR2 through SENSE)
against the FP64 restatement (oracle), at the edges of its tiles: one to 33
coils (8 and 16 a product, 16 a launch layer), outputs and inputs that fill no
tile, input slices.

Tolerance: the FP32 phase of a pair, P revolutions, is rounded to 2^-24 P a
few times, so a term is off by up to 2 pi 2^-23 (P + 1) relative; the sums add
less."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("M,n,Nz,nc,r2", [
    (1, 4, 1, 1, False), (63, 6, 1, 1, False), (65, 8, 1, 8, False), (130, 10, 1, 9, False),
    (1000, 12, 4, 17, False), (4099, 16, 1, 33, False), (333, 6, 6, 3, True),
    (333, 6, 6, 18, True), (5000, 40, 1, 2, False)])
def test_sense_dft(orc, M, n, Nz, nc, r2):
    import powergrid_amd as P
    rng = np.random.default_rng(M)
    N = n * n * Nz
    k = [rng.uniform(-n / 2, n / 2, M).astype(np.float32) for _ in range(3)]
    t = rng.uniform(0, 0.01, M).astype(np.float32)
    r = [rng.uniform(-0.5, 0.5, N).astype(np.float32) for _ in range(3)]
    fm = rng.uniform(-700, 700, N).astype(np.float32)

    def cplx(*s):
        return (rng.standard_normal(s) + 1j * rng.standard_normal(s)).astype(np.complex64)

    sens, x, y = cplx(nc, N), cplx(N), cplx(M * nc)
    dims = (n, n, Nz) if r2 else ()
    D = (P.GdftR2 if r2 else P.Gdft)(M, N, *k, *r, fm, t, *dims)
    Do = (orc.GdftR2 if r2 else orc.Gdft)(M, N, *k, *r, fm, t, *dims, prec="d")
    A = P.SENSE(D, sens, M, N, nc)
    O = orc.SENSE(Do, sens.astype(complex).ravel(), M, N, nc)
    turns = 3 * (n / 2) * 0.5 + 700 * 0.01 / (2 * np.pi)
    tol = 2 * np.pi * 2.0 ** -23 * (turns + 1)
    assert _rel(A * x, O * x.astype(complex)) < tol
    assert _rel(A / y, O / y.astype(complex)) < tol
