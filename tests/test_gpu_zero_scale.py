"""A store whose scale is 0 decodes as one of scale 1 (native_codec.cpp
weight_at) in every product, as in the decoded values that it exports: native
bytes mounted with scale 0 against the oracle's decode of them."""
import numpy as np
import pytest

import pywelvet
from oracle import DTYPE_NAMES
from parity import tol_for_k
from test_gpu_dense import elementwise_bound

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    pywelvet.init()


def _check(oracle, dtype, out, inn, batch):
    rng = np.random.default_rng(dtype * 1000 + out + batch)
    W = rng.normal(0, 0.1, (out, inn)).astype(np.float32)
    raw, _ = oracle.pack(dtype, W)
    Wd = oracle.decode_f64(dtype, raw, 0.0, W.size).reshape(W.shape)
    x = rng.normal(0, 1, (batch, inn)).astype(np.float32)
    gy = rng.normal(0, 1, (batch, out)).astype(np.float32)
    with pywelvet.Session((out, inn), batch=batch, dtype=dtype, native=(raw, 0.0)) as s:
        pre, _ = s.execute(x)
        dX, _ = s.backward(x, gy, gy)
    assert np.all(np.abs(pre - x.astype(np.float64) @ Wd.T) <= elementwise_bound(Wd, x, tol_for_k(inn)))
    assert np.all(np.abs(dX - gy.astype(np.float64) @ Wd) <= elementwise_bound(Wd.T, gy, tol_for_k(out)))


@pytest.mark.parametrize("dtype", range(34), ids=DTYPE_NAMES)
@pytest.mark.parametrize("batch", [1, 2, 5, 16, 17, 40])
def test_zero_scale_is_one(oracle, dtype, batch):
    for out, inn in ((70, 256), (33, 50)):
        _check(oracle, dtype, out, inn, batch)


def test_zero_scale_uint8_split(oracle):
    """Uint8 at the sizes where it takes the split-x GEMM (1024 units)."""
    _check(oracle, 13, 2065, 2032, 70)
