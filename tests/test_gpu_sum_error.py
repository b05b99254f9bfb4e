"""How far sums over a long K are from 64 bits (2-norm of the difference over
2-norm of the result), which the element-wise tolerances do not see.  A GEMM's
fp32 chains end at its shares of K (they are added in f64): c products of
random sign in one chain of fp32 additions, each rounded to 2^-24 / 2 at most
of a partial sum that grows as the root of its length, end within 2^-24
sqrt(c / 2) of the result (a mean over the outputs; about a third of it is
measured)."""
import numpy as np
import pytest

import pywelvet
from test_gpu_dense import oracle_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    pywelvet.init()


def chain_bound(products):
    return 2.0 ** -24 * np.sqrt(products / 2)


def error(got, ref):
    return np.linalg.norm(got - ref) / np.linalg.norm(ref)


@pytest.mark.parametrize("dtype,batch", [(1, 17), (1, 64), (2, 13), (2, 33), (3, 13), (3, 33), (8, 33), (13, 33),
                                         (15, 33), (27, 64)])
def test_long_k_few_outputs(oracle, dtype, batch):
    """128 outputs over K = 11008: one k stage of 64 per share in the kernels
    without stage sums, forward and (K = rows) dX."""
    rng = np.random.default_rng(dtype * 100 + batch)
    W = rng.normal(0, 0.1, (128, 11008)).astype(np.float32)
    x = rng.normal(0, 1, (batch, 11008)).astype(np.float32)
    pre, _ = pywelvet.forward(W, x, dtype=dtype)
    Wd = oracle_weights(oracle, dtype, W)
    assert error(pre, x.astype(np.float64) @ Wd.T) <= chain_bound(64)
    V = np.ascontiguousarray(W.T)
    with pywelvet.Session(V, batch=batch, dtype=dtype) as s:
        dX, _ = s.backward(np.zeros((batch, 128), np.float32), x, x)
    Vd = oracle_weights(oracle, dtype, V)
    assert error(dX, x.astype(np.float64) @ Vd) <= chain_bound(64)


@pytest.mark.parametrize("dtype", [4, 5, 9, 16, 26, 2])
@pytest.mark.parametrize("inn,out,batch", [(1024, 1024, 512), (4096, 512, 250), (2048, 4096, 120), (1024, 3000, 100)])
def test_stage_sums(oracle, dtype, inn, out, batch):
    """32-row tiles above batch 32 (K = 4 to 8 stages a share): a stage rounds
    its sum four times (16 products a step; the products of x's and w's lower
    parts weigh 2^-8) and the tile's sum once, n stages a share and the
    output's own rounding on top."""
    rng = np.random.default_rng(dtype * 100 + batch)
    W = rng.normal(0, 2.0 if dtype == 16 else 0.1, (out, inn)).astype(np.float32)
    x = rng.normal(0, 1, (batch, inn)).astype(np.float32)
    pre, _ = pywelvet.forward(W, x, dtype=dtype)
    Wd = oracle_weights(oracle, dtype, W)
    stages = -(-(-(-batch // 32) * -(-out // 128) * (inn // 64)) // 512)  # a share of 512 blocks' equal ones
    assert error(pre, x.astype(np.float64) @ Wd.T) <= 2.0 ** -24 * np.sqrt((4 + stages + 1) / 2)


@pytest.mark.parametrize("lo,hi", [(-3.0, 0.05), (-0.05, 3.0), (0.5, 0.75), (-0.05, 0.05)])
def test_uint8_decoded_values(oracle, lo, hi):
    """Uint8 multiplies the decoded values fl32(fl32(q scale) + min): with a
    range far to one side of most weights their rounding is 1e-6 of them, and
    products of unrounded q scale + min are that far off.  Six products a
    weight, 24 roundings a stage, three stages a share."""
    rng = np.random.default_rng(17)
    W = np.clip(rng.normal(0, 0.01, (2065, 2032)).astype(np.float32) + np.float32(max(lo, 0)), lo, hi)
    W[0, 0], W[-1, -1] = lo, hi
    x = rng.normal(0, 1, (70, 2032)).astype(np.float32)
    pre, _ = pywelvet.forward(W, x, dtype=13)
    Wd = oracle_weights(oracle, 13, W)
    assert error(pre, x.astype(np.float64) @ Wd.T) <= chain_bound(72)


@pytest.mark.parametrize("dtype", [1, 13])
def test_short_k_many_outputs(oracle, dtype):
    """Six-product kinds at K = 16 and more tiles than 64-row ones start at: two
    steps of 16 products, the low parts' sum and the output's rounding."""
    rng = np.random.default_rng(dtype)
    W = rng.normal(0, 0.1, (8200, 16)).astype(np.float32)
    x = rng.normal(0, 1, (1100, 16)).astype(np.float32)
    pre, _ = pywelvet.forward(W, x, dtype=dtype)
    Wd = oracle_weights(oracle, dtype, W)
    assert error(pre, x.astype(np.float64) @ Wd.T) <= 2.0 ** -24 * np.sqrt((2 + 1 + 1) / 2)
