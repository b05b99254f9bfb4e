"""Host-buffer calls whose copies are cut into pieces on several threads and
whose device buffers come from the pool of freed blocks: every byte arrives at
sizes around the pieces' edges, and calls from several threads at once give
what they give one after another."""
import threading

import numpy as np
import pytest

import pywelvet

pytestmark = pytest.mark.gpu
MB = 1 << 18  # floats


@pytest.fixture(scope="module", autouse=True)
def device():
    pywelvet.init()


@pytest.mark.parametrize("n", [1, MB - 1, MB, MB + 1, 2 * MB + 3, 5 * MB + 1023, 8 * MB, 17 * MB + 1, 33 * MB + 5])
def test_copies_are_whole(n):
    """A Float32 store takes its values and gives them back bit for bit."""
    rng = np.random.default_rng(n)
    a, b = (rng.integers(1, 2 ** 30, n, dtype=np.uint32).view(np.float32) for _ in range(2))
    with pywelvet.Session(a.reshape(n, 1), batch=1, dtype=1) as s:
        assert np.array_equal(s.export_f32().ravel().view(np.uint32), a.view(np.uint32))
        s.repack(b)
        raw, _ = s.native()
        assert np.array_equal(raw.view(np.uint32), b.view(np.uint32))


def test_calls_from_several_threads():
    rng = np.random.default_rng(4)
    jobs = [(rng.normal(0, 0.1, (o, i)).astype(np.float32), rng.normal(0, 1, (b, i)).astype(np.float32), d)
            for o, i, b, d in ((700, 640, 5, 1), (1024, 1024, 40, 2), (64, 4096, 9, 26), (900, 333, 3, 9))]
    targets = [np.zeros((x.shape[0], W.shape[0]), np.float32) for W, x, _ in jobs]

    def call(k):
        W, x, d = jobs[k]
        r = pywelvet.normalbp(W, x, targets[k], 1, 0.1, act=0, dtype=d)
        return {n: np.array(v) for n, v in r.items()}

    want = [call(k) for k in range(len(jobs))]
    bad = []

    def work(k):
        for _ in range(6):
            got = call(k)
            bad.extend((k, n) for n in got if not np.array_equal(got[n], want[k][n]))

    team = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not bad, bad[:4]


def test_large_calls_from_several_threads():
    """Three calls at once whose weights (38 MB) go up and whose gradient and
    new weights come down in pieces on several threads each."""
    rng = np.random.default_rng(6)
    jobs = [(rng.normal(0, 0.1, (2304, 4096)).astype(np.float32), rng.normal(0, 1, (2, 4096)).astype(np.float32))
            for _ in range(3)]

    def call(k):
        W, x = jobs[k]
        r = pywelvet.normalbp(W, x, np.zeros((2, 2304), np.float32), 1, 0.1, act=-1, dtype=1)
        return {n: np.array(v) for n, v in r.items()}

    want = [call(k) for k in range(3)]
    for k, (W, _) in enumerate(jobs):  # the Float32 step of the gradient that came down with it, within a rounding each
        assert np.allclose(want[k]["W_after"], W - 0.1 * want[k]["dW"], rtol=3e-7, atol=1e-7)
    bad = []

    def work(k):
        for _ in range(3):
            got = call(k)
            bad.extend((k, n) for n in got if not np.array_equal(got[n], want[k][n]))

    team = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not bad, bad[:4]
