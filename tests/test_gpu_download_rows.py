"""Small results whose rows lie apart on the device (widths that are padded there):
their bytes, and that they take about the time of rows that lie together."""
import time

import numpy as np
import pytest

from seisfem_amd import surrogate

pytestmark = pytest.mark.gpu


def say(msg):
    print("[gpu-case]", msg, flush=True)


def median_ms(f, reps=15):
    f()
    v = []
    for _ in range(reps):
        t = time.perf_counter()
        f()
        v.append(1e3 * (time.perf_counter() - t))
    return float(np.median(v))


@pytest.mark.parametrize("nin,nout", [(13, 97), (1, 500), (31, 1)])
def test_padded_rows(nin, nout):
    say(f"weights and predictions of {nin} inputs and {nout} outputs")
    net = surrogate.MLP(nin, 200, 1, nout, batch=64, seed=3)
    rng = np.random.default_rng(nout)
    for l in range(net.nlayers):
        W, b = (rng.standard_normal(a.shape).astype(np.float32) for a in net.layer(l))
        net.set_layer(l, W, b)
        Wg, bg = net.layer(l)
        assert np.array_equal(Wg, W) and np.array_equal(bg, b)
    X = rng.uniform(0, 1, (70, nin)).astype(np.float32)
    Y, _ = net.predict(X)
    assert np.max(np.abs(Y)) > 0
    for i in (0, 63, 69):
        assert np.array_equal(net.predict(X[i:i + 1])[0][0], Y[i])
    net.close()


def test_padded_rows_take_the_time_of_packed_ones():
    """1024 rows of 13 weights in a pitch of 32, and of 32 weights: 0.04 ms each
    (7 ms for the former when every row was a transfer)."""
    say("time of padded rows")
    ms = {}
    for nin in (13, 32):
        net = surrogate.MLP(nin, 1024, 1, 32, batch=64, seed=3)
        ms[nin] = median_ms(lambda: net.layer(0))
        net.close()
    assert ms[13] < 10 * ms[32] + 0.5, ms
