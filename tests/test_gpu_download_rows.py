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


# below, at and above the sizes where the way of a copy changes (64 KB, 256 KB, 4 MB), shots in
# the caller's order and not, with and without the large pinned buffers of an earlier download
@pytest.mark.parametrize("large_first", [False, True])
@pytest.mark.parametrize("shots,steps,nrec", [(3, 20, 100), (4, 40, 60), (7, 40, 400), (9, 160, 400)])
def test_seismograms_of_all_sizes(shots, steps, nrec, large_first):
    from seisfem_amd import gpu, host
    en, x, y = host.mesh_structured(host.Q4, 20, 20, 0.0, 200.0, 0.0, 200.0)
    vp, rho = np.full(x.size, 3000.0), np.full(x.size, 2000.0)
    prob = host.build_problem(host.Q4, en, x, y, rho, host.elastic_constants(rho, vp, vp / 1.73), vp, 10.0, 5, 5, 1,
                              bbox=(0.0, 200.0, 0.0, 200.0))
    op = gpu.Operator(prob["node_num"], prob["csr"])
    md = gpu.Medium(op, prob["c"], prob["mass_lump"], prob["dirichlet"], prob["mpml"])
    say(f"{shots} shots of {steps} steps at {nrec} receivers, large buffers first: {large_first}")
    net = surrogate.MLP(13, 1100, 1, 1100, batch=32, seed=1)
    if large_first:
        net.layer(1)                                 # 4.8 MB
    src = (150 + 11 * np.arange(shots)).astype(np.int32)
    rec = np.arange(nrec, dtype=np.int32)
    for order in (np.full(shots, steps), steps - (np.arange(shots) * 5) % 9):
        nsteps = order.astype(np.int32)
        run = gpu.Run(op, md, src, steps, rec, 5.0e-4, 25.0, 0.01, nsteps=nsteps, guard_every=40)
        run.advance(steps)
        u, w = run.seismograms()
        run.close()
        assert np.max(np.abs(u)) > 0
        for s in range(shots):
            one = gpu.Run(op, md, src[s:s + 1], steps, rec[s::50], 5.0e-4, 25.0, 0.01, nsteps=nsteps[s:s + 1],
                          guard_every=40)
            one.advance(steps)
            u1, w1 = one.seismograms()
            one.close()
            assert np.array_equal(u[s, :, s::50], u1[0]) and np.array_equal(w[s, :, s::50], w1[0]), s
    for h in (net, md, op):
        h.close()
