"""Forward and dX of rows that start off a chunk boundary, against the oracle:
every dtype at the edges of the kernels' chunks, stages and tiles, and for a
Float32 and a 6-bit store the larger tile shapes.  Products and sums are f64
there, so an output may differ from the oracle's f64 sum by its one rounding
to f32 (2^-24 relative, doubled for the oracle's own) and by the two f64
summation orders: at most K roundings of 2^-53 of the sum of magnitudes each."""
import numpy as np
import pytest

import pywelvet
from oracle import DTYPE_NAMES
from test_gpu_dense import oracle_weights

pytestmark = pytest.mark.gpu

# (out, in, batch): one code; inside a chunk; chunk and stage edges (16, 32,
# 64, 128 elements) on either side; batch on both sides of the row-product /
# MFMA border (4, 5) and of the 16-row tile
EDGES = [(1, 1, 1), (3, 2, 5), (17, 3, 4), (15, 31, 2), (16, 33, 16), (33, 63, 17), (5, 129, 3), (18, 127, 6),
         (31, 257, 20), (2, 1027, 1), (9, 515, 33)]


@pytest.fixture(scope="module", autouse=True)
def device():
    pywelvet.init()


def within(got, want, A, Wd, k, what):
    """got, want [m][n] for sums over k of A [m][k] * Wd [k][n]."""
    bound = 2.0 ** -23 * np.abs(want) + k * 2.0 ** -52 * (np.abs(A.astype(np.float64)) @ np.abs(Wd)) + 1e-45
    bad = ~(np.abs(got.astype(np.float64) - want) <= bound)
    assert not bad.any(), (what, np.argwhere(bad)[:4], got[bad][:4], want[bad][:4])


def check(oracle, dtype, out, inn, batch, path=0):
    rng = np.random.default_rng(dtype * 1000 + out * 31 + inn * 7 + batch)
    W = rng.normal(0, 0.5, (out, inn)).astype(np.float32)
    x = rng.normal(0, 1, (batch, inn)).astype(np.float32)
    gy = rng.normal(0, 1, (batch, out)).astype(np.float32)
    Wd = oracle_weights(oracle, dtype, W)
    tag = (DTYPE_NAMES[dtype], out, inn, batch)
    with pywelvet.Session(W, batch=batch, act=-1, dtype=dtype) as s:
        pywelvet.set_forward_path(path)
        try:
            pre, post = s.execute(x)
        finally:
            pywelvet.set_forward_path(0)
        dX, _ = s.backward(x, pre, gy)
    ref = x.astype(np.float64) @ Wd.T
    within(pre, ref, x, Wd.T, inn, ("pre",) + tag)
    assert np.array_equal(pre, post)
    if path == 0:
        within(dX, gy.astype(np.float64) @ Wd, gy, Wd, out, ("dX",) + tag)


def chunk(dtype):
    bits = pywelvet.DTYPE_BITS[dtype]
    return 32 if bits <= 6 else max(1, 128 // bits)


@pytest.mark.parametrize("dtype", range(34), ids=DTYPE_NAMES)
def test_ragged_edges(oracle, dtype):
    for out, inn, batch in EDGES:
        if inn % chunk(dtype):
            check(oracle, dtype, out, inn, batch)


@pytest.mark.parametrize("dtype", range(34), ids=DTYPE_NAMES)
def test_element_wise_path_takes_aligned_rows(oracle, dtype):
    """set_forward_path(3) runs the same kernels on any shape."""
    for out, inn, batch in ((24, 128, 2), (40, 96, 9)):
        check(oracle, dtype, out, inn, batch, path=3)


@pytest.mark.parametrize("dtype", [1, 27])
@pytest.mark.parametrize("out,inn,batch", [(1000, 333, 290), (333, 1001, 260), (700, 1001, 600)])
def test_ragged_large_tiles(oracle, dtype, out, inn, batch):
    check(oracle, dtype, out, inn, batch)


def test_ragged_nonfinite_weights_stay_in_their_columns(oracle):
    """An Inf or NaN weight reaches only the outputs that use it, though the
    kernels decode the neighbouring rows' codes past a row's end."""
    rng = np.random.default_rng(5)
    W = rng.normal(0, 1, (20, 37)).astype(np.float32)
    W[3, 0], W[9, 36], W[12, 5] = np.inf, -np.inf, np.nan
    for batch in (1, 3, 18):
        x = rng.normal(0, 1, (batch, 37)).astype(np.float32)
        gy = rng.normal(0, 1, (batch, 20)).astype(np.float32)
        with pywelvet.Session(W, batch=batch, act=-1, dtype=1) as s:
            pre, _ = s.execute(x)
            dX, _ = s.backward(x, pre, gy)
        good = [o for o in range(20) if o not in (3, 9, 12)]
        assert np.isfinite(pre[:, good]).all() and not np.isfinite(pre[:, [3, 9, 12]]).any()
        good = [i for i in range(37) if i not in (0, 5, 36)]
        assert np.isfinite(dX[:, good]).all() and not np.isfinite(dX[:, [0, 5, 36]]).any()


@pytest.mark.parametrize("dtype", range(34), ids=DTYPE_NAMES)
@pytest.mark.parametrize("batch", [5, 6, 7, 8])
def test_ragged_long_rows_small_batch(oracle, dtype, batch):
    """Batch 5 to 8 of long rows as row products in two halves (an odd batch's
    halves share a row); 515 columns for Complex64, which takes them there."""
    for out, inn in ((5, 3075), (9, 515)):
        if inn % chunk(dtype):
            check(oracle, dtype, out, inn, batch)


def test_ragged_batch_5_costs_little_more_than_batch_4():
    """One MFMA chain per 16 x 16 outputs took three times batch 4's row
    products at 4095 -> 100; two halves of them take 1.2 times."""
    import time

    from devmem import DeviceArray, hip
    W = np.random.default_rng(1).normal(0, 1, (100, 4095)).astype(np.float32)
    best = {}
    for batch in (4, 5):
        d_x, d_pre, d_post = (DeviceArray((batch, n), 0.5) for n in (4095, 100, 100))
        with pywelvet.Session(W, batch=batch, act=-1, dtype=1) as s:
            t = []
            for _ in range(8):
                hip().hipDeviceSynchronize()
                t0 = time.perf_counter()
                for _ in range(100):
                    s.forward_device(d_x.ptr, d_pre.ptr, d_post.ptr)
                hip().hipDeviceSynchronize()
                t.append((time.perf_counter() - t0) / 100)
        best[batch] = min(t)
    print({b: "%.1f us" % (t * 1e6) for b, t in best.items()}, flush=True)
    assert best[5] < 2 * best[4]


@pytest.mark.parametrize("dtype", [1, 0, 14, 27])
@pytest.mark.parametrize("out,inn,batch", [(16, 4095, 16), (16, 4097, 16), (17, 33, 31), (17, 41, 25), (777, 11, 8)])
def test_ragged_dx_few(oracle, dtype, out, inn, batch):
    """dX of few rows or few outputs, on both sides of where its kernels change
    (16 rows and 65536 outputs, 1024 outputs)."""
    if inn % chunk(dtype):
        check(oracle, dtype, out, inn, batch)


@pytest.mark.parametrize("batch", [5, 6, 7, 8])
def test_ragged_swiglu_halves(batch):
    """SwiGLU's Up projection reads h and overwrites it: a row in both halves of
    an odd batch is stored once.  g and u are f64 sums rounded once, so h is
    within a few f32 roundings of silu(g) u."""
    rng = np.random.default_rng(batch)
    G, U = (rng.normal(0, 0.02, (37, 3075)).astype(np.float32) for _ in range(2))
    D = rng.normal(0, 0.2, (3075, 37)).astype(np.float32)
    x = rng.normal(0, 1, (batch, 3075)).astype(np.float32)
    xd = x.astype(np.float64)
    g, u = xd @ G.astype(np.float64).T, xd @ U.astype(np.float64).T
    ref = g / (1 + np.exp(-g)) * u
    for _ in range(5):
        h, _ = pywelvet.swiglu_forward(G, U, D, x, dtype=1)
        assert np.all(np.abs(h - ref) <= 1e-6 * (np.abs(ref) + np.abs(u) + np.abs(g)) + 1e-30)
