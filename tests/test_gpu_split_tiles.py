"""The split-x GEMM's tiles with ragged batch, outputs and k stages: every
kernel that a plan can ask for above batch 16, at the shapes of
split_shapes.py (test_plans_cpu.py holds which kernel runs there), against f64
products of the decoded weights.  An output is within 1e-5 of the sum of
magnitudes; over all outputs the error is at most a chain of 24 roundings a
stage, four stages, long: 2^-24 sqrt(96 / 2)."""
import numpy as np
import pytest

import pywelvet
import split_shapes as S
from oracle import DTYPE_NAMES
from test_gpu_dense import elementwise_bound, oracle_weights
from test_gpu_sum_error import error

pytestmark = pytest.mark.gpu
TOTAL = 2.0 ** -24 * np.sqrt(96 / 2)


@pytest.fixture(scope="module", autouse=True)
def device():
    pywelvet.init()


def _weights(rng, kind, out, inn):
    return rng.normal(0, 2.0 if kind == S.FP4 else 0.1, (out, inn)).astype(np.float32)


CASES = [(k, *s[:3]) for s in S.SHAPES for k in s[3]]


@pytest.mark.parametrize("kind,out,inn,batch", CASES,
                         ids=["{}-{}x{}-b{}".format(DTYPE_NAMES[S.DTYPE[k]], i, o, b) for k, o, i, b in CASES])
def test_forward(oracle, kind, out, inn, batch):
    rng = np.random.default_rng(kind * 1000 + batch)
    dtype = S.DTYPE[kind]
    W = _weights(rng, kind, out, inn)
    x = rng.normal(0, 1, (batch, inn)).astype(np.float32)
    bias = rng.normal(0, 0.1, out)
    pre, _ = pywelvet.forward(W, x, act=2, dtype=dtype, bias=bias)
    Wd = oracle_weights(oracle, dtype, W)
    ref = x.astype(np.float64) @ Wd.T + bias
    assert np.all(np.abs(pre - ref) <= elementwise_bound(Wd, x, 1e-5) + 1e-6 * np.abs(bias))
    assert error(pre, ref) <= TOTAL


@pytest.mark.parametrize("kind", S.ONE)
@pytest.mark.parametrize("out,inn,batch", [(1952, 2064, 300), (2016, 2064, 490), (2016, 1296, 200), (1056, 272, 70)])
def test_dx(oracle, kind, out, inn, batch):
    """dX through the transposed codes: K = outputs, half a stage past whole."""
    rng = np.random.default_rng(kind * 77 + batch)
    dtype = S.DTYPE[kind]
    W = _weights(rng, kind, out, inn)
    gy = rng.normal(0, 1, (batch, out)).astype(np.float32)
    with pywelvet.Session(W, batch=batch, act=-1, dtype=dtype) as s:
        dX, _ = s.backward(np.zeros((batch, inn), np.float32), gy, gy)
    Wd = oracle_weights(oracle, dtype, W)
    ref = gy.astype(np.float64) @ Wd
    assert np.all(np.abs(dX - ref) <= elementwise_bound(Wd.T, gy, 1e-5))
    assert error(dX, ref) <= TOTAL


PAIRS = [(k, *s[:3]) for s in S.SHAPES for k in s[4]]


@pytest.mark.parametrize("kind,inter,inn,batch", PAIRS,
                         ids=["{}-{}x{}-b{}".format(DTYPE_NAMES[S.DTYPE[k]], i, o, b) for k, o, i, b in PAIRS])
def test_pair(oracle, kind, inter, inn, batch):
    """Gate and Up in one launch: h = silu(g) u, with |silu'| <= 1.1 the errors of
    g and u weighted by the other factor."""
    rng = np.random.default_rng(kind * 1000 + batch + 1)
    dtype = S.DTYPE[kind]
    G, U = (_weights(rng, kind, inter, inn) for _ in range(2))
    D = np.ones((inn, inter), np.float32)
    x = rng.normal(0, 0.5 / np.sqrt(inn) if kind == S.FP4 else 10 / np.sqrt(inn), (batch, inn)).astype(np.float32)
    h, _ = pywelvet.swiglu_forward(G, U, D, x, dtype=dtype)
    Gd, Ud = oracle_weights(oracle, dtype, G), oracle_weights(oracle, dtype, U)
    xd = x.astype(np.float64)
    g, u = xd @ Gd.T, xd @ Ud.T
    sg = g / (1 + np.exp(-g))
    tol_g, tol_u = (1e-5 * (np.abs(xd) @ np.abs(W).T) for W in (Gd, Ud))
    ref = sg * u
    assert np.all(np.abs(h - ref) <= 1.2 * tol_g * (np.abs(u) + tol_u) + np.abs(sg) * tol_u + 1e-6 * np.abs(ref) + 1e-30)
    # |d h| <= 1.1 |dg| |u| + |sg| |du|: at most 3 times a product's relative error
    assert error(h, ref) <= 3 * TOTAL
