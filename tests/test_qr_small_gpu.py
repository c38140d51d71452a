"""QR of calls that hold small matrices (qlt_block_qr): a call of small matrices
only, many small ones beside larger ones (which take different kernels), a few
beside larger ones (which share one), and shapes on both sides of the lines
between them.

Compared with LAPACK's factors; the bound is the one of the blocked QR's tests, 100 m eps
max(1, sqrt n) for matrices of condition below 10."""
import numpy as np
import pytest

from tensortoolkit_amd import decompose as DEC

pytestmark = pytest.mark.gpu


def _well_conditioned(rng, m, n, cplx):
    def draw(a, b):
        return rng.standard_normal((a, b)) + (1j * rng.standard_normal((a, b)) if cplx else 0)
    k = min(m, n)
    u, v = np.linalg.qr(draw(m, k))[0], np.linalg.qr(draw(n, k))[0]
    return (u * np.linspace(1.0, 5.0, k)) @ v.conj().T


SMALL = [(1, 1), (2, 2), (3, 1), (1, 7), (4, 4), (6, 5), (2, 60), (1, 300), (64, 2), (256, 4), (1500, 1)]
EDGE = [(6, 8), (6, 9), (8, 8), (8, 9), (9, 9), (11, 11), (12, 12), (13, 13), (4, 64), (1024, 3), (1025, 3), (3072, 1),
        (1, 128), (1, 129), (1, 300), (1, 301), (1, 1400), (1, 1401), (1, 2048), (1, 2049), (24, 24), (24, 25), (25, 24),
        (25, 25)]
BATCHES = {
    "small": SMALL,
    "one": [(2, 2)],
    "one_edge": [(6, 9)],
    "many_small": [(1 + i % 5, 1 + i % 7) for i in range(600)],
    "many_edge": EDGE * 45,
    "few_beside_large": [(40, 33)] + SMALL + [(90, 17)],
    "many_beside_large": [(1 + i % 4, 1 + i % 3) for i in range(520)] + [(40, 33), (17, 70)],
    "beside_too_tall": [(2050, 3), (3, 3), (40, 20)],
    "edge": EDGE,
}


@pytest.mark.parametrize("batch", list(BATCHES))
@pytest.mark.parametrize("dtype", ["f64", "c128"])
def test_small_matrices_match_lapack(qlt, dtype, batch):
    rng = np.random.default_rng(20261203 + len(batch))
    mats = [_well_conditioned(rng, m, n, dtype == "c128") for m, n in BATCHES[batch]]
    print(f"case: small qr {dtype} {batch}", flush=True)
    eps = np.finfo(np.float64).eps
    for a, (q, r) in zip(mats, DEC.block_qr_dense(mats, dtype)):
        m, n = a.shape
        qn, rn = np.linalg.qr(a)
        tol = 100 * m * eps * max(1.0, np.sqrt(n))
        assert np.max(np.abs(r - rn)) <= 5 * tol
        assert np.max(np.abs(q - qn)) <= tol
        assert not np.any(np.tril(r, -1))
