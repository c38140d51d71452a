"""Native grouped GEMM at the edges of its tiles and steps: one block of m x k
times k x n with extents around the 16-row / 16-column MFMA blocks, the 32-row
and 32- / 64-column tiles, the n <= 4 and n <= 16 classes, and contracted extents
around the 4-k, 8-k and 16-k steps; operands in every memory order, so that
blocks contiguous in either axis, affine and not affine in k all occur; every
element type; alpha and beta.

An inner product of length k computed in FP64, in any order, is within
2 k eps sum |a b| (complex: 4 products); entries are uniform in [-1, 1), so
relative to the block's Frobenius norm (about sqrt(m n k) / 3) 64 k eps bounds
it; single precision adds its rounding, 2^-24 per entry of inputs already
rounded."""
import numpy as np
import pytest

from tensortoolkit_amd import capi
from tensortoolkit_amd.blocksparse import IN, OUT, BlockSparseTensor, ContractionPlan, Index

pytestmark = pytest.mark.gpu

CODE = {"f64": capi.QLT_F64, "c128": capi.QLT_C128, "f32": capi.QLT_F32, "c64": capi.QLT_C64}
NP = {"f64": np.float64, "c128": np.complex128, "f32": np.float32, "c64": np.complex64}


def _index(n, d):
    return Index(((0,),), (n,), d)


def _draw(rng, shape, dtype):
    x = rng.uniform(-1, 1, shape)
    if dtype in ("c128", "c64"):
        x = x + 1j * rng.uniform(-1, 1, shape)
    return x.astype(NP[dtype])


def _run(rng, dtype, a_dims, b_dims, a_ctr, b_ctr, a_sav, b_sav, alpha, beta):
    wide = "c128" if dtype in ("c128", "c64") else "f64"
    a = BlockSparseTensor.allowed_blocks([_index(d, IN) for d in a_dims], (0,), wide)
    b_idx = [_index(d, OUT) for d in b_dims]
    b = BlockSparseTensor.allowed_blocks(b_idx, (0,), wide)
    x, y = _draw(rng, a_dims, dtype), _draw(rng, b_dims, dtype)
    plan = ContractionPlan(a, b, a_ctr, b_ctr, a_sav, b_sav)
    ref = np.tensordot(x.astype(a.np_dtype), y.astype(a.np_dtype), axes=(a_ctr, b_ctr))
    fa, fb = sorted(a_sav), sorted(b_sav)
    ref = np.transpose(ref, [fa.index(v) for v in a_sav] + [len(fa) + fb.index(v) for v in b_sav]).reshape(-1)
    c0 = _draw(rng, ref.size, dtype)
    da, db, dc = (capi.DeviceBuffer.from_numpy(v) for v in (x.reshape(-1), y.reshape(-1), c0))
    al, be = np.array([np.real(alpha), np.imag(alpha)]), np.array([np.real(beta), np.imag(beta)])
    capi.check(capi.lib().qlt_contract_execute(plan.handle, CODE[dtype], capi.QLT_MODE_NATIVE, da.ptr, db.ptr, dc.ptr,
                                               capi.f64(al), capi.f64(be), None))
    capi.check(capi.lib().qlt_device_sync())
    got = dc.to_numpy(NP[dtype], ref.size).astype(a.np_dtype)
    exp = alpha * ref + beta * c0.astype(a.np_dtype)
    k = int(np.prod([a_dims[v] for v in a_ctr]))
    tol = 64 * k * np.finfo(np.float64).eps + (2.0 ** -23 if dtype in ("f32", "c64") else 0.0)
    scale = np.linalg.norm(alpha * ref) + np.linalg.norm(beta * c0)
    assert np.linalg.norm(got - exp) <= tol * scale, (a_dims, b_dims, a_ctr, b_ctr)


@pytest.mark.parametrize("dtype", ["f64", "c128", "f32", "c64"])
@pytest.mark.parametrize("order", ["mk_kn", "km_kn", "mk_nk", "km_nk"])
def test_tile_and_step_edges(qlt, dtype, order):
    rng = np.random.default_rng(17)
    print(f"case: tile edges {dtype} {order}", flush=True)
    left, right = order.split("_")
    cases = [(m, n, k) for m in (1, 16, 33) for n in (5, 16, 17, 33, 65) for k in (1, 4, 9, 16, 17)]
    cases += [(15, 31, 3), (17, 32, 8), (31, 64, 5), (32, 15, 33), (64, 97, 31), (65, 6, 130), (130, 70, 40), (40, 130, 600)]
    for m, n, k in cases:
        a_dims, a_ctr, a_sav = ((m, k), [1], [0]) if left == "mk" else ((k, m), [0], [1])
        b_dims, b_ctr, b_sav = ((k, n), [0], [1]) if right == "kn" else ((n, k), [1], [0])
        alpha, beta = (1.0, 0.0) if (m + n + k) % 2 else (-0.5, 2.0)
        _run(rng, dtype, a_dims, b_dims, a_ctr, b_ctr, a_sav, b_sav, alpha, beta)


@pytest.mark.parametrize("dtype", ["f64", "c128", "f32", "c64"])
def test_blocks_not_affine_in_k(qlt, dtype):
    """Contracted axes that do not merge into one stride (either operand, or
    both), with saved axes in cyclic order."""
    rng = np.random.default_rng(23)
    print(f"case: not affine in k {dtype}", flush=True)
    for p, q, s in ((3, 5, 7), (4, 4, 4), (2, 9, 6), (7, 3, 11)):
        # A (k0 m0 k1 m1), B (n0 k1 n1 k0): neither merges
        _run(rng, dtype, (p, 6, q, 7), (s, q, 5, p), [0, 2], [3, 1], [1, 3], [0, 2], 1.0, 0.0)
        # A merges (m0 m1 | k0 k1), B does not, saved axes reversed
        _run(rng, dtype, (5, 4, p, q), (q, s, p, 3), [2, 3], [2, 0], [1, 0], [3, 1], 1.5, -0.25)
        # n <= 16 on the same layouts
        _run(rng, dtype, (p, 9, q, 5), (3, q, 4, p), [0, 2], [3, 1], [3, 1], [2, 0], 1.0, 0.5)
