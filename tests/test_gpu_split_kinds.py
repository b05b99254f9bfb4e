"""The split-x bf16 GEMM's kinds for batches above 16 (BFloat16, Float16,
Float32, Int4, Uint8) against the oracle: edges of the batch and of the k stage
(64), weights of one sign, non-finite operands, and both ends of the float
range (the tiles' edges: test_gpu_split_tiles.py).  The products of BFloat16, Int4 and Float16's and Float32's higher
parts are exact; the dropped ones of the lower parts are at most 3.9 2^-23 of
a product (Float16 1.7), and the sums are fp32, so an output is within 1e-5 of
the sum of magnitudes, as for the other kinds."""
import numpy as np
import pytest

import pywelvet
from oracle import DTYPE_NAMES
from test_gpu_dense import check_forward, elementwise_bound, oracle_weights

pytestmark = pytest.mark.gpu
KINDS = [3, 2, 1, 14, 13]
# (out, in, batch): K of one piece, inside a stage, 31.5 stages, whole stage
# pairs; columns past a tile; batch at both sides of the 32- and 64-row tiles
SHAPES = [(40, 32, 17), (129, 96, 32), (257, 2016, 33), (300, 1024, 64), (100, 512, 65), (8200, 128, 20),
          (1000, 640, 130)]


@pytest.fixture(scope="module", autouse=True)
def device():
    pywelvet.init()


@pytest.mark.parametrize("dtype", KINDS, ids=[DTYPE_NAMES[d] for d in KINDS])
def test_split_kinds(oracle, dtype):
    rng = np.random.default_rng(40 + dtype)
    for out, inn, batch in SHAPES:
        W = rng.normal(0, 0.1, (out, inn)).astype(np.float32)
        x = rng.normal(0, 1, (batch, inn)).astype(np.float32)
        check_forward(oracle, dtype, W, x)
        check_forward(oracle, dtype, W, x, act=2, bias=rng.normal(0, 0.1, out))
    # K % 16 == 8: the half formats' rows are chunks, the x pieces are not
    if dtype in (2, 3):
        W = rng.normal(0, 0.1, (70, 72)).astype(np.float32)
        check_forward(oracle, dtype, W, rng.normal(0, 1, (40, 72)).astype(np.float32))


@pytest.mark.parametrize("lo,hi", [(0.5, 0.75), (-0.75, -0.5), (-0.05, 3.0), (0.25, 0.25)])
def test_uint8_offsets(oracle, lo, hi):
    """Uint8 ranges without 0, with an outlier on one side, and of no width (96
    outputs: the fp32 MFMA; test_gpu_sum_error.py has such ranges on the
    split-x GEMM)."""
    rng = np.random.default_rng(3)
    W = rng.normal(0, 0.01, (96, 256)).astype(np.float32) + np.float32((lo + hi) / 2 if lo * hi > 0 else 0)
    W = np.clip(W, lo, hi)
    W[0, 0], W[-1, -1] = lo, hi
    x = rng.normal(0, 1, (40, 256)).astype(np.float32)
    pre, _ = pywelvet.forward(W, x, dtype=13)
    Wd = oracle_weights(oracle, 13, W)
    ref = x.astype(np.float64) @ Wd.T
    assert np.all(np.abs(pre - ref) <= elementwise_bound(Wd, x, 1e-5))


@pytest.mark.parametrize("dtype", [3, 2, 1, 13])
@pytest.mark.parametrize("batch", [20, 70])
@pytest.mark.parametrize("out", [40, 520])
def test_split_kinds_nonfinite(oracle, dtype, batch, out):
    """Infinities and NaN in x (all kinds) and W (the float ones): the class
    of every output is that of the whole operands' product.  K = 80 ends
    inside a k stage, which then holds the next row's first weights.  520
    outputs: Float32 and Uint8, on the fp32 MFMA at 40, are split there too."""
    rng = np.random.default_rng(batch + dtype)
    W = rng.choice(np.float32([-1.0, -0.5, 0.5, 1.0, 0.0]), (out, 80)).astype(np.float32)
    W[0, 0], W[0, 1] = 1.0, -1.0
    x = rng.choice(np.float32([-2.0, -1.0, 1.0, 0.0, 0.37]), (batch, 80)).astype(np.float32)
    x[3, 5], x[4, 6], x[5, 7], x[6, 1], x[6, 2] = np.inf, -np.inf, np.nan, np.inf, -np.inf
    if dtype != 13:
        W[7, 3], W[9, 0], W[11, 79], W[13, 4] = np.inf, -np.inf, np.inf, np.nan
    pre, _ = pywelvet.forward(W, x, dtype=dtype)
    Wd = oracle_weights(oracle, dtype, W)
    with np.errstate(invalid="ignore"):
        ref = np.array([[np.sum(x[m].astype(np.float64) * Wd[n]) for n in range(out)] for m in range(batch)])
    assert np.array_equal(np.isnan(pre), np.isnan(ref))
    assert np.array_equal(pre[np.isinf(ref)], ref[np.isinf(ref)].astype(np.float32))
    ok = np.isfinite(ref)
    assert np.allclose(pre[ok], ref[ok], rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("inn", [64, 128])
def test_noalloc_keeps_the_batches_it_took(oracle, inn):
    """A batch whose split-x plan needs more partial tiles than the fixed
    64 MiB takes the fp32 MFMA plan there (Float32 128 -> 4096 b3584: 80
    against 64 MiB; one k stage, on 32-row tiles, fits)."""
    from test_zz_no_alloc import run
    rng = np.random.default_rng(9)
    W = rng.normal(0, 0.1, (4096, inn)).astype(np.float32)
    x = rng.normal(0, 1, (3584, inn)).astype(np.float32)
    with pywelvet.Session(W, batch=1, act=-1, dtype=1) as s:
        got, _ = run(s, 3584, x, True)
    ref = x.astype(np.float64) @ W.astype(np.float64).T
    assert np.all(np.abs(got - ref) <= elementwise_bound(W.astype(np.float64), x, 1e-5))


@pytest.mark.parametrize("dtype", [3, 1], ids=[DTYPE_NAMES[d] for d in (3, 1)])
def test_nan_redo_is_bounded(dtype):
    """The recomputation of NaN sums costs a small multiple of the product: a
    NaN at the end of every row of x next to nothing (such rows need no walk
    over K), one in every row of W a wave-wide walk per output.  The limits
    leave a factor of three over what is measured; a serial walk per output
    takes hundreds of times the product."""
    import time

    from devmem import DeviceArray, hip
    n, batch = 2048, 512
    rng = np.random.default_rng(5)
    W = rng.normal(0, 0.1, (n, n)).astype(np.float32)
    x = rng.normal(0, 1, (batch, n)).astype(np.float32)
    d_x, d_pre, d_post = DeviceArray((batch, n)), DeviceArray((batch, n)), DeviceArray((batch, n))

    def best(W, x):
        d_x.upload(x)
        with pywelvet.Session(W, batch=batch, act=-1, dtype=dtype) as s:
            t = []
            for _ in range(6):
                hip().hipDeviceSynchronize()
                t0 = time.perf_counter()
                s.forward_device(d_x.ptr, d_pre.ptr, d_post.ptr)
                hip().hipDeviceSynchronize()
                t.append(time.perf_counter() - t0)
        return min(t), d_pre.download()

    xn, Wn = x.copy(), W.copy()
    xn[:, -1] = np.nan
    Wn[:, -1] = np.nan
    plain, _ = best(W, x)
    in_x, got = best(W, xn)
    assert np.isnan(got).all()
    in_w, got = best(Wn, x)
    assert np.isnan(got).all()
    print(f"plain {plain * 1e6:.0f} us, NaN in x {in_x * 1e6:.0f}, in W {in_w * 1e6:.0f}", flush=True)
    assert in_x < 4 * plain
    assert in_w < 60 * plain


@pytest.mark.parametrize("scale,big", [(0.01, 1e37), (1.0, 1e37), (1e38, 1e-3), (1e-44, 1e30), (-0.5, 3e37)])
def test_int4_extremes(oracle, scale, big):
    """Int4 stores at both ends of the float range, mounted from native bytes:
    sums of 16 code x pass the largest float where those of the decoded
    weights do not, a sixteenth of a small scale is no float, and codes whose
    value is infinite."""
    rng = np.random.default_rng(3)
    raw, _ = oracle.pack(14, rng.normal(0, 1, (70, 128)).astype(np.float32))
    x = rng.normal(0, 1, (40, 128)).astype(np.float32)
    if scale == 1e38:  # fp32 sums of its finite values (up to 3e38 |x|, 128 of them) stay below 3.4e38
        x *= np.float32(1e-3)
    x[:, 9] = big * rng.choice([-1.0, 0.5, 1.0], 40)
    Wd = oracle.decode_f64(14, raw, scale, 70 * 128).reshape(70, 128)
    with pywelvet.Session((70, 128), batch=40, dtype=14, native=(raw, scale)) as s:
        pre, _ = s.execute(x)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = np.array([[np.sum(x[m].astype(np.float64) * Wd[n]) for n in range(70)] for m in range(40)])
        ref32 = ref.astype(np.float32)
        assert np.array_equal(np.isnan(pre), np.isnan(ref32))
        assert np.array_equal(pre[np.isinf(ref32)], ref32[np.isinf(ref32)])
        ok = np.isfinite(ref32)
        bound = elementwise_bound(np.where(np.isfinite(Wd), Wd, 0), x, 1e-5)
    assert np.all(np.abs(pre[ok] - ref[ok]) <= bound[ok] + 1.5e-45)


def test_int4_pair_extremes(oracle):
    """SwiGLU's Gate and Up in one launch with sums of 16 code x past the
    largest float: g and u are small, h their product."""
    rng = np.random.default_rng(4)
    G, U = (rng.normal(0, 1e-36, (70, 128)).astype(np.float32) for _ in range(2))
    D = rng.normal(0, 0.1, (128, 70)).astype(np.float32)
    x = np.zeros((40, 128), np.float32)
    x[:, 5], x[:, 77] = 2e37, -1e37
    pre, _ = pywelvet.swiglu_forward(G, U, D, x, dtype=14)

    def decoded(W):
        raw, s = oracle.pack(14, W)
        return oracle.decode_f64(14, raw, s, W.size).reshape(W.shape)

    g, u = (x.astype(np.float64) @ decoded(W).T for W in (G, U))
    ref = g / (1 + np.exp(-g)) * u
    assert np.all(np.abs(pre - ref) <= 1e-5 * (np.abs(ref) + np.abs(u) + np.abs(g) + 1))
