"""The blocked QR at the sizes where its branches change (qlt_block_qr):
columns around multiples of the 16-column block, wide matrices whose last
panel holds columns past the last reflector, rows around the panel's register
capacities, and matrices too tall for it in the same batch as small ones.

Q and R are compared with LAPACK's (same reflector convention).  Householder
QR is backward stable with a constant of about m n eps, which the condition
number of Q's and R's dependence on A multiplies: the matrices are scaled
orthonormal bases plus noise, condition below 10, so 100 m eps max(1, sqrt n)
bounds both factors' entries."""
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


SHAPES = {
    "columns": [(40, 15), (40, 16), (40, 17), (33, 32), (33, 33), (64, 48), (64, 49)],
    "wide": [(1, 16), (1, 17), (15, 40), (16, 16), (16, 33), (17, 18), (17, 64), (31, 130)],
    "mixed": [(1, 1), (2, 1), (300, 3), (257, 129), (5, 290)],
    "rows512": [(511, 20), (512, 17), (513, 18)],
    "rows1024": [(1024, 17), (1025, 33)],
    "rows1536": [(1536, 16), (1537, 20), (30, 30)],
    "rows2048": [(2048, 18), (2049, 17), (12, 40)],
}


@pytest.mark.parametrize("group", list(SHAPES))
@pytest.mark.parametrize("dtype", ["f64", "c128"])
def test_blocked_qr_matches_lapack(qlt, dtype, group):
    rng = np.random.default_rng(20261202 + len(group))
    mats = [_well_conditioned(rng, m, n, dtype == "c128") for m, n in SHAPES[group]]
    print(f"case: blocked qr {dtype} {SHAPES[group]}", flush=True)
    eps = np.finfo(np.float64).eps
    for a, (q, r) in zip(mats, DEC.block_qr_dense(mats, dtype)):
        m, n = a.shape
        qn, rn = np.linalg.qr(a)
        tol = 100 * m * eps * max(1.0, np.sqrt(n))
        assert np.max(np.abs(r - rn)) <= 5 * tol
        assert np.max(np.abs(q - qn)) <= tol
        assert np.max(np.abs(q.conj().T @ q - np.eye(q.shape[1]))) <= tol
        assert not np.any(np.tril(r, -1))


@pytest.mark.parametrize("dtype", ["f64", "c128"])
def test_blocked_qr_zero_columns_and_rows(qlt, dtype):
    """Zero columns take no reflector, zero trailing rows stay zero in Q."""
    rng = np.random.default_rng(9)
    a = _well_conditioned(rng, 70, 40, dtype == "c128")
    a[:, [0, 15, 16, 39]] = 0.0
    b = np.zeros((20, 18), dtype=a.dtype)
    b[:9, :9] = _well_conditioned(rng, 9, 9, dtype == "c128")
    for x, (q, r) in zip((a, b), DEC.block_qr_dense([a, b], dtype)):
        assert np.linalg.norm(q @ r - x) <= 1e-13 * np.linalg.norm(x)
        assert np.max(np.abs(q.conj().T @ q - np.eye(q.shape[1]))) <= 1e-12
