"""GPU: qlt_block_svd at the edges of its column pairs (32 columns, odd
counts), of the row groups of its Gram (64) and update (32) steps, and with
transposed working matrices, against numpy in FP64.  A pair counts as
orthogonal below M eps, so values, reconstruction and orthogonality are held
to a few times M eps (relative to the norm)."""
import ctypes as C

import numpy as np
import pytest

from tensortoolkit_amd import capi

pytestmark = pytest.mark.gpu

BATCHES = [[(1, 1), (2, 2), (3, 2)], [(31, 31), (33, 32), (32, 33)], [(65, 17), (64, 16), (63, 18)],
           [(97, 33), (33, 129), (5, 4)]]


@pytest.mark.parametrize("dtype", ["f64", "c128"])
@pytest.mark.parametrize("shapes", BATCHES)
def test_svd_edges(qlt, dtype, shapes):
    print(f"case: svd edges {dtype} {shapes}", flush=True)
    lib = capi.lib()
    code, npt = (capi.QLT_C128, np.complex128) if dtype == "c128" else (capi.QLT_F64, np.float64)
    rng = np.random.default_rng(sum(m * n for m, n in shapes))
    mats = []
    for m, n in shapes:
        x = rng.uniform(-1, 1, (m, n))
        mats.append(x + 1j * rng.uniform(-1, 1, (m, n)) if dtype == "c128" else x)
    rows, cols = np.array([m for m, _ in shapes]), np.array([n for _, n in shapes])
    k = np.minimum(rows, cols)
    ao, uo, so, vo = (np.concatenate([[0], np.cumsum(z)]).astype(np.int64) for z in (rows * cols, rows * k, k, k * cols))
    a = capi.DeviceBuffer.from_numpy(np.concatenate([m.reshape(-1) for m in mats]))
    esz = np.dtype(npt).itemsize
    u, s, v = (capi.DeviceBuffer(int(z)) for z in (uo[-1] * esz, so[-1] * 8, vo[-1] * esz))
    capi.check(lib.qlt_block_svd(code, len(mats), capi.i64(rows), capi.i64(cols), a.ptr, capi.i64(ao[:-1]), u.ptr,
                                 capi.i64(uo[:-1]), s.ptr, capi.i64(so[:-1]), v.ptr, capi.i64(vo[:-1]), None, None))
    capi.check(lib.qlt_device_sync())
    U, S, V = u.to_numpy(npt), s.to_numpy(np.float64), v.to_numpy(npt)
    for i, A in enumerate(mats):
        m, n = A.shape
        Ui, Si = U[uo[i]:uo[i + 1]].reshape(m, k[i]), S[so[i]:so[i + 1]]
        Vi = V[vo[i]:vo[i + 1]].reshape(k[i], n)
        tol = 8 * max(16, m, n) * np.finfo(np.float64).eps
        ref = np.linalg.svd(A, compute_uv=False)
        assert np.all(np.abs(Si - ref) <= tol * ref[0])
        assert np.linalg.norm((Ui * Si) @ Vi - A) <= tol * np.linalg.norm(A)
        # the smallest values of these matrices are within 10^3 of the largest: U = X / sigma
        long = Ui.conj().T @ Ui, Vi @ Vi.conj().T
        cond = ref[0] / ref[-1]
        assert max(np.linalg.norm(g - np.eye(k[i])) for g in long) <= tol * np.sqrt(k[i]) * max(1.0, cond)
