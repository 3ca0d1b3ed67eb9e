"""Results of more than 4 MB come back through pinned pieces: the same bytes as
the small ones, which are copied directly."""
import numpy as np
import pytest

from seisfem_amd import gpu, host, surrogate

pytestmark = pytest.mark.gpu


def say(msg):
    print("[gpu-case]", msg, flush=True)


# widths that are a multiple of the padding and widths that are not (rows in a pitch)
@pytest.mark.parametrize("hidden,nout,n", [(1152, 32000, 70), (1101, 16411, 129)])
def test_weights_and_predictions(hidden, nout, n):
    net = surrogate.MLP(13, hidden, 2, nout, batch=64, seed=5)
    rng = np.random.default_rng(hidden)
    say(f"mlp 13-{hidden}-{hidden}-{nout}: weights and {n} predictions")
    for l in range(net.nlayers):
        W, b = net.layer(l)
        W = rng.standard_normal(W.shape).astype(np.float32) / np.float32(np.sqrt(W.shape[1]))
        b = rng.standard_normal(b.shape).astype(np.float32)
        net.set_layer(l, W, b)
        Wg, bg = net.layer(l)
        assert np.array_equal(Wg, W) and np.array_equal(bg, b)
    X = rng.uniform(0, 1, (n, 13)).astype(np.float32)
    Y, _ = net.predict(X)
    assert np.max(np.abs(Y)) > 0
    for i in range(0, n, 16):
        assert np.array_equal(net.predict(X[i:i + 16])[0], Y[i:i + 16])


# traces of several pieces each, and several traces to a piece; shots of different
# lengths (kept longest first inside the run)
@pytest.mark.parametrize("shots,steps,nrec", [(3, 530, 441), (40, 120, 140)])
def test_seismograms(shots, steps, nrec):
    en, x, y = host.mesh_structured(host.Q4, 20, 20, 0.0, 200.0, 0.0, 200.0)
    vp = np.full(x.size, 3000.0)
    rho = np.full(x.size, 2000.0)
    c = host.elastic_constants(rho, vp, vp / 1.73)
    prob = host.build_problem(host.Q4, en, x, y, rho, c, vp, 10.0, 5, 5, 1, bbox=(0.0, 200.0, 0.0, 200.0))
    op = gpu.Operator(prob["node_num"], prob["csr"])
    md = gpu.Medium(op, prob["c"], prob["mass_lump"], prob["dirichlet"], prob["mpml"])
    src = (100 + 5 * np.arange(shots)).astype(np.int32)
    nsteps = (steps - (np.arange(shots) * 37) % 90).astype(np.int32)
    rec = np.arange(nrec, dtype=np.int32)
    say(f"{shots} shots of up to {steps} steps at {nrec} receivers")
    run = gpu.Run(op, md, src, steps, rec, 5.0e-4, 25.0, 0.03, nsteps=nsteps, guard_every=40)
    run.advance(steps)
    u, w = run.seismograms()
    run.close()
    # the shots whose source is a fixed node of the border stay at rest
    assert u.nbytes > 4 << 20 and np.sum(np.max(np.abs(u), axis=(1, 2)) > 0) > shots // 2
    for s in range(0, shots, 13 if shots > 3 else 1):
        one = gpu.Run(op, md, src[s:s + 1], steps, rec[107:114], 5.0e-4, 25.0, 0.03, nsteps=nsteps[s:s + 1], guard_every=40)
        one.advance(steps)
        u1, w1 = one.seismograms()
        one.close()
        assert np.array_equal(u[s, :, 107:114], u1[0]) and np.array_equal(w[s, :, 107:114], w1[0])
