"""GPU: qlt_block_svd of a batch in which one matrix holds a NaN: the call
returns, and the other matrices get the factors they get without it, bit for
bit.  (The column order of a matrix is a permutation whatever its norms.)"""
import ctypes as C

import numpy as np
import pytest

from tensortoolkit_amd import capi

pytestmark = pytest.mark.gpu


def _svd(lib, code, npt, mats):
    rows, cols = [m.shape[0] for m in mats], [m.shape[1] for m in mats]
    k = [min(m.shape) for m in mats]
    off = lambda sizes: np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
    ao, uo, so, vo = (off([r * c for r, c in zip(rows, cols)]), off([r * x for r, x in zip(rows, k)]), off(k),
                      off([x * c for x, c in zip(k, cols)]))
    a = capi.DeviceBuffer.from_numpy(np.concatenate([m.reshape(-1) for m in mats]))
    esz = np.dtype(npt).itemsize
    u, s, v = capi.DeviceBuffer(int(uo[-1]) * esz), capi.DeviceBuffer(int(so[-1]) * 8), capi.DeviceBuffer(int(vo[-1]) * esz)
    sweeps = C.c_int32(0)
    status = lib.qlt_block_svd(code, len(mats), capi.i64(np.array(rows)), capi.i64(np.array(cols)), a.ptr,
                               capi.i64(ao[:-1]), u.ptr, capi.i64(uo[:-1]), s.ptr, capi.i64(so[:-1]), v.ptr,
                               capi.i64(vo[:-1]), C.byref(sweeps), None)
    capi.check(lib.qlt_device_sync())
    U, S, V = u.to_numpy(npt), s.to_numpy(np.float64), v.to_numpy(npt)
    return status, [(U[uo[i]:uo[i + 1]], S[so[i]:so[i + 1]], V[vo[i]:vo[i + 1]]) for i in range(len(mats))]


@pytest.mark.parametrize("dtype", ["f64", "c128"])
@pytest.mark.parametrize("shape", [(40, 33), (12, 70), (2, 2)])
def test_nan_matrix_leaves_the_others_alone(qlt, dtype, shape):
    print(f"case: svd with a NaN matrix {dtype} {shape}", flush=True)
    lib = capi.lib()
    code, npt = (capi.QLT_C128, np.complex128) if dtype == "c128" else (capi.QLT_F64, np.float64)
    rng = np.random.default_rng(shape[0])

    def draw(m, n):
        x = rng.uniform(-1, 1, (m, n))
        return np.ascontiguousarray(x + 1j * rng.uniform(-1, 1, (m, n)) if dtype == "c128" else x)

    mats = [draw(35, 20), draw(*shape), draw(18, 50)]
    status, want = _svd(lib, code, npt, mats)
    assert status == 0
    mats[1][1, 0] = np.nan
    status, got = _svd(lib, code, npt, mats)
    assert status == 0
    for i in (0, 2):
        for g, w in zip(got[i], want[i]):
            np.testing.assert_array_equal(g, w)
    assert np.isnan(got[1][1]).any()
