"""Native contractions onto narrow outputs (n <= 16) on every path that they
may take: 32-row tiles whose four waves share the contracted extent, 32-row tiles of
a wave each (many rows, few 16-k steps), and the n <= 4 row class, each with and
without k-slices; both sides of the lines between them; and plans that hold
blocks of all tile classes at once, so that they run in one launch.  The tile count of
a plan says which path its blocks took.

A sum of k products in FP64, in any order, is within 2 k eps sum |a b| (complex:
4 products each); entries are uniform in [-1, 1), so 64 k eps of the output's
Frobenius norm (about sqrt(m n k) / 3) bounds it; single precision adds 2^-23 of
the stored result, its inputs being rounded already."""
import numpy as np
import pytest

from tensortoolkit_amd import capi
from tensortoolkit_amd.blocksparse import IN, OUT, BlockSparseTensor, ContractionPlan, Index

pytestmark = pytest.mark.gpu

CODE = {"f64": capi.QLT_F64, "c128": capi.QLT_C128, "f32": capi.QLT_F32, "c64": capi.QLT_C64}
NP = {"f64": np.float64, "c128": np.complex128, "f32": np.float32, "c64": np.complex64}
DTYPES = ["f64", "c128", "f32", "c64"]


def _draw(rng, n, dtype):
    x = rng.uniform(-1, 1, n)
    if dtype in ("c128", "c64"):
        x = x + 1j * rng.uniform(-1, 1, n)
    return x.astype(NP[dtype])


def _execute(rng, dtype, plan, a, b, reference, k, alpha, beta):
    """reference(x, y): the raw result of raw operands in FP64 / complex128."""
    wide = np.complex128 if dtype in ("c128", "c64") else np.float64
    x, y = _draw(rng, a.raw_size, dtype), _draw(rng, b.raw_size, dtype)
    ref = reference(x.astype(wide), y.astype(wide))
    assert ref.size == plan.info.c_raw_size
    c0 = _draw(rng, ref.size, dtype)
    da, db, dc = (capi.DeviceBuffer.from_numpy(v) for v in (x, y, c0))
    al, be = np.array([np.real(alpha), np.imag(alpha)]), np.array([np.real(beta), np.imag(beta)])
    capi.check(capi.lib().qlt_contract_execute(plan.handle, CODE[dtype], capi.QLT_MODE_NATIVE, da.ptr, db.ptr, dc.ptr,
                                               capi.f64(al), capi.f64(be), None))
    capi.check(capi.lib().qlt_device_sync())
    got = dc.to_numpy(NP[dtype], ref.size).astype(wide)
    tol = 64 * k * np.finfo(np.float64).eps + (2.0 ** -23 if dtype in ("f32", "c64") else 0.0)
    scale = np.linalg.norm(alpha * ref) + np.linalg.norm(beta * c0)
    assert np.linalg.norm(got - (alpha * ref + beta * c0.astype(wide))) <= tol * scale


def _diagonal(shapes, order):
    """Block q: m_q x k_q ("km": stored k_q x m_q) times k_q x n_q."""
    qns = tuple((q,) for q in range(len(shapes)))
    ms, ks, ns = (tuple(s[i] for s in shapes) for i in range(3))
    left = [Index(qns, ms, IN), Index(qns, ks, OUT)] if order == "mk" else [Index(qns, ks, IN), Index(qns, ms, OUT)]
    a = BlockSparseTensor.allowed_blocks(left, (0,))
    b = BlockSparseTensor.allowed_blocks([Index(qns, ks, IN), Index(qns, ns, OUT)], (0,))
    plan = ContractionPlan(a, b, [1 if order == "mk" else 0], [0])

    def reference(x, y):
        out, xo, yo = [], 0, 0
        for m, k, n in shapes:
            blk = x[xo:xo + m * k].reshape((m, k) if order == "mk" else (k, m))
            out.append(((blk if order == "mk" else blk.T) @ y[yo:yo + k * n].reshape(k, n)).reshape(-1))
            xo, yo = xo + m * k, yo + k * n
        return np.concatenate(out)

    return plan, a, b, reference


def _tasks(m, n, tasks, k):
    """One output block of `tasks` tasks of contracted extent k."""
    q = tuple((j,) for j in range(tasks))
    mid, aux = Index(q, (k,) * tasks, OUT), Index(q, (1,) * tasks, IN)
    a = BlockSparseTensor.allowed_blocks([Index(((0,),), (m,), IN), aux, mid], (0,))
    b = BlockSparseTensor.allowed_blocks([mid.inverse(), aux.inverse(), Index(((0,),), (n,), OUT)], (0,))
    plan = ContractionPlan(a, b, [2, 1], [0, 1])

    def reference(x, y):
        return np.einsum("tmk,tkn->mn", x.reshape(tasks, m, k), y.reshape(tasks, k, n)).reshape(-1)

    return plan, a, b, reference


def _run(rng, dtype, made, k, tiles, alpha=1.0, beta=0.0):
    plan, a, b, reference = made
    assert plan.info.n_panel_tiles == 0
    if tiles is not None:
        assert plan.info.n_tiles == tiles
    _execute(rng, dtype, plan, a, b, reference, k, alpha, beta)


def _ceil(x, y):
    return -(-x // y)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("order", ["mk", "km"])
def test_tiles_of_a_wave_each(qlt, dtype, order):
    rng = np.random.default_rng(31)
    print(f"case: a tile per wave {dtype} {order}", flush=True)
    for m, n, k in ((32737, 5, 1), (32768, 8, 4), (32800, 16, 15), (32897, 11, 16), (65540, 6, 17), (65505, 16, 32)):
        _run(rng, dtype, _diagonal([(m, k, n)], order), k, _ceil(m, 128))
        _run(rng, dtype, _diagonal([(m, k, n)], order), k, _ceil(m, 128), -0.5, 2.0)
    # 9 short tasks, a step each
    _run(rng, dtype, _tasks(294912, 5, 9, 1), 9, _ceil(294912, 128), -1.0, 0.0)
    # one tile short of the line: the waves share each tile
    _run(rng, dtype, _diagonal([(32736, 16, 7)], order), 16, _ceil(32736, 32), 1.5, -0.25)
    _run(rng, dtype, _diagonal([(65504, 17, 7)], order), 17, _ceil(65504, 32))


@pytest.mark.parametrize("dtype", DTYPES)
def test_sliced_tiles_of_a_wave_each(qlt, dtype):
    """Few rows of 16 steps beside many of one step: two k-slices for the few."""
    rng = np.random.default_rng(33)
    print(f"case: k-sliced tiles of a wave each {dtype}", flush=True)
    shapes = [(1100001, 1, 5), (100, 250, 9), (129, 256, 16)]
    tiles = _ceil(1100001, 128) + 2 + 4
    _run(rng, dtype, _diagonal(shapes, "mk"), 256, tiles, 1.0, 0.0)
    _run(rng, dtype, _diagonal(shapes, "km"), 256, tiles, 0.75, -1.5)


@pytest.mark.parametrize("dtype", DTYPES)
def test_sliced_row_class(qlt, dtype):
    """n <= 4 blocks of many short tasks: the row class, cut into k-slices of 8 steps."""
    rng = np.random.default_rng(35)
    print(f"case: k-sliced row class {dtype}", flush=True)
    alpha, beta = (0.5 - 1.5j, 2.0 + 0.25j) if dtype in ("c128", "c64") else (1.5, -0.75)
    for m, n, tasks, k in ((100, 3, 40, 1), (1025, 1, 20, 3), (7, 4, 64, 1), (2050, 2, 17, 2)):
        tiles = _ceil(m, 1024) * _ceil(tasks, 8)
        assert tiles > 1
        _run(rng, dtype, _tasks(m, n, tasks, k), tasks * k, tiles)
        _run(rng, dtype, _tasks(m, n, tasks, k), tasks * k, tiles, alpha, beta)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("order", ["mk", "km"])
def test_row_class_edges(qlt, dtype, order):
    """n in 1 .. 4 around the contracted extent up to which the row class takes them."""
    rng = np.random.default_rng(37)
    print(f"case: row class edges {dtype} {order}", flush=True)
    for n in (1, 2, 3, 4):
        for m in (1, 31, 1030):
            for k in (5, 63, 64, 65, 130):
                tiles = _ceil(m, 1024) if k <= 64 else _ceil(m, 32)
                _run(rng, dtype, _diagonal([(m, k, n)], order), k, tiles, *((1.0, 0.0) if k % 2 else (-0.5, 2.0)))


@pytest.mark.parametrize("dtype", ["f64", "c64"])
def test_long_sums_over_many_rows_stay_with_the_row_class(qlt, dtype):
    rng = np.random.default_rng(39)
    print(f"case: long sums over many rows {dtype}", flush=True)
    m = 255 * 1024 + 1
    _run(rng, dtype, _diagonal([(m, 66, 2)], "km"), 66, 256)
    _run(rng, dtype, _diagonal([(m - 1, 66, 2)], "km"), 66, _ceil(m - 1, 32), 1.0, 0.5)
    _run(rng, dtype, _diagonal([(m, 66, 2)], "mk"), 66, _ceil(m, 32))
    # 70 tasks of k = 1 in 22 row tiles (1540 steps, in slices of at least 8), and in 21: 32-row
    # tiles whose chains of 70 steps are cut into slices of 32 at least
    _run(rng, dtype, _tasks(21 * 1024 + 1, 3, 70, 1), 70, 22 * 9, -1.0, 0.5)
    _run(rng, dtype, _tasks(21 * 1024, 3, 70, 1), 70, 21 * 32 * 3)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("order", ["mk", "km"])
def test_every_class_in_one_plan(qlt, dtype, order):
    """Blocks of n <= 4, n <= 16, 32 x 32 and 32 x 64 tiles together, ragged, some
    k-sliced; then with a block of wave tiles beside them."""
    rng = np.random.default_rng(41)
    print(f"case: every class in one plan {dtype} {order}", flush=True)
    alpha, beta = (0.5 - 1.5j, 2.0 + 0.25j) if dtype in ("c128", "c64") else (1.5, -0.75)
    shapes = [(70, 40, 3), (33, 17, 10), (50, 30, 20), (65, 9, 50), (31, 200, 16), (1030, 64, 1), (130, 33, 97),
              (5, 300, 4), (40, 1500, 33), (64, 1500, 64), (17, 1500, 12)]
    for extra in ([], [(90000, 16, 6)]):
        _run(rng, dtype, _diagonal(shapes + extra, order), 1500, None)
        _run(rng, dtype, _diagonal(shapes + extra, order), 1500, None, alpha, beta)
