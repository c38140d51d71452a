"""GPU: qlt_lanczos_update_extend (w += scale V c2, then the Lanczos extension
of the updated w) against qlt_basis_update followed by qlt_lanczos_extend, bit
for bit, and against numpy in FP64; qlt_basis_dot over more than one sweep of
basis vectors.  Edges: no elements, one element, one more than the grid of
the reductions covers in a step (512 x 256), active vectors on both sides of
the sweeps of 8 and 16, a full arena (no slot to store to), w = 0."""
import ctypes as C

import numpy as np
import pytest

from tensortoolkit_amd import capi

pytestmark = pytest.mark.gpu

K_MAX = 20


def _dev(a):
    return capi.DeviceBuffer.from_numpy(np.ascontiguousarray(a))


@pytest.mark.parametrize("dtype", ["f64", "c128"])
@pytest.mark.parametrize("n,m,zero", [(0, 1, False), (1, 1, False), (255, 8, False), (131073, 9, False),
                                      (131073, 16, False), (3001, 17, False), (3001, K_MAX, False), (513, 3, True)])
def test_update_extend_matches_update_then_extend(qlt, dtype, n, m, zero):
    print(f"case: update+extend {dtype} n={n} m={m} zero={zero}", flush=True)
    lib = capi.lib()
    cplx = dtype == "c128"
    code, npt = (capi.QLT_C128, np.complex128) if cplx else (capi.QLT_F64, np.float64)
    ldv = n + 3
    rng = np.random.default_rng(17 * n + m)

    def draw(*shape):
        x = rng.uniform(-1, 1, shape)
        return (x + 1j * rng.uniform(-1, 1, shape)) if cplx else x

    V, w, c2 = draw(K_MAX, ldv), draw(max(n, 1)), draw(K_MAX)
    if zero:
        w[:], c2[:] = 0, 0
    c1 = rng.uniform(-1, 1, 2 * K_MAX)
    pairs = np.stack([c2.real, c2.imag], axis=1).reshape(-1)
    dc1, dc2 = _dev(c1), _dev(pairs)
    out = []
    for fused in (False, True):
        dV, dw, dcount = _dev(V), _dev(w), _dev(np.array([m], dtype=np.int32))
        dal, dbe = _dev(np.full(K_MAX, 7.0)), _dev(np.full(K_MAX, 7.0))
        dwork = capi.DeviceBuffer(8 * (2 * 512 * K_MAX + 1))
        if fused:
            capi.check(lib.qlt_lanczos_update_extend(code, n, K_MAX, dcount.ptr, dc1.ptr, -1.0, dc2.ptr, dw.ptr,
                                                     dV.ptr, ldv, dal.ptr, dbe.ptr, dwork.ptr, None))
        else:
            capi.check(lib.qlt_basis_update(code, n, K_MAX, dcount.ptr, -1.0, dc2.ptr, dV.ptr, ldv, dw.ptr, None))
            capi.check(lib.qlt_lanczos_extend(code, n, K_MAX, dcount.ptr, dc1.ptr, dw.ptr, dV.ptr, ldv, dal.ptr,
                                              dbe.ptr, dwork.ptr, None))
        capi.check(lib.qlt_device_sync())
        out.append((dw.to_numpy(npt), dV.to_numpy(npt).reshape(K_MAX, ldv), dal.to_numpy(np.float64),
                    dbe.to_numpy(np.float64), int(dcount.to_numpy(np.int32)[0])))
    for a, b in zip(*out):
        np.testing.assert_array_equal(a, b)
    got_w, got_V, al, be, count = out[1]
    assert count == min(m + 1, K_MAX)
    ref = w[:n] - c2[:m] @ V[:m, :n]
    beta = np.linalg.norm(ref)
    # m + 1 roundings of terms of size below 2 each, n of them in the norm
    assert np.linalg.norm(got_w[:n] - ref) <= 1e-15 * 4 * (m + 1) * np.sqrt(n + 1)
    assert abs(be[m - 1] - beta) <= 1e-13 * (1.0 + beta) and al[m - 1] == c1[2 * (m - 1)]
    keep = np.ones(K_MAX, dtype=bool)
    keep[m - 1] = False
    assert np.all(al[keep] == 7.0) and np.all(be[keep] == 7.0)
    want = V.copy()
    if m < K_MAX:
        want[m, :n] = got_w[:n] * (1.0 / be[m - 1] if be[m - 1] > 0 else 0.0)
        np.testing.assert_allclose(got_V[m, :n], want[m, :n], rtol=1e-15, atol=0)
        want[m, :n] = got_V[m, :n]
    np.testing.assert_array_equal(got_V, want)
    # the products of the whole arena with the vector (20 = 16 + 4 vectors)
    dout, dwork = capi.DeviceBuffer(16 * K_MAX), capi.DeviceBuffer(8 * (2 * 512 * K_MAX + 1))
    dV, dw, dcount = _dev(V), _dev(w), _dev(np.array([m], dtype=np.int32))
    capi.check(lib.qlt_basis_dot(code, n, K_MAX, dcount.ptr, dV.ptr, ldv, dw.ptr, dout.ptr, dwork.ptr, None))
    capi.check(lib.qlt_device_sync())
    o = dout.to_numpy(np.float64)
    o = o[0::2] + 1j * o[1::2]
    assert np.linalg.norm(o[:m] - V[:m, :n].conj() @ w[:n]) <= 4e-15 * (n + 1) * np.sqrt(m)
    assert np.all(o[m:] == 0)
