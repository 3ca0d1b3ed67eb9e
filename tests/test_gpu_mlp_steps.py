"""The passes between the products of a training step, and the training steps
that run beside one another, on the GPU.

Gradients: tolerance of tests/test_gpu_mlp.py (the same bf16 operands, FP32
sums in another order: rel-L2 <= 2e-3).
"""
import math

import numpy as np
import pytest

from oracle import mlp_oracle as mo
from seisfem_amd import surrogate

pytestmark = pytest.mark.gpu


def say(msg):
    print("[gpu-case]", msg, flush=True)


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-30))


# batches below, across and beyond the 256 rows of a pass, not multiples of 16 or of 64;
# hidden products in 3, 4 and 16 parts over K; padded and unpadded widths
@pytest.mark.parametrize("batch,hidden,nout", [(24, 160, 96), (264, 136, 97), (520, 200, 64), (64, 1024, 2048)])
def test_gradients_match_oracle(batch, hidden, nout):
    net = surrogate.MLP(13, hidden, 3, nout, batch=batch, seed=7)
    rng = np.random.default_rng(batch)
    X = rng.uniform(0, 1, (batch, 13)).astype(np.float32)
    T = rng.standard_normal((batch, nout)).astype(np.float32)
    Ws, bs = zip(*[net.layer(l) for l in range(net.nlayers)])
    bs = [rng.standard_normal(b.shape).astype(np.float32) * np.float32(0.1) for b in bs]
    for l in range(net.nlayers):
        net.set_layer(l, Ws[l], bs[l])
    say(f"mlp gradients 13-{hidden}x3-{nout} batch {batch}")
    loss_ref, gW, gb = mo.loss_and_grads([w.astype(np.float64) for w in Ws], [b.astype(np.float64) for b in bs], X, T,
                                         round_bf16=True)
    for l in range(net.nlayers):
        loss, g, b = net.gradients(X, T, l)
        assert abs(loss - loss_ref) <= 1e-4 * loss_ref
        assert rel(g, gW[l]) < 2e-3, l
        assert rel(b, gb[l]) < 2e-3, l
    net.close()


def _orders(n, seed, epochs):
    """The sample orders of sfg_mlp_train."""
    mask, out = (1 << 64) - 1, []
    s = (seed * 0x9E3779B97F4A7C15 + 7) & mask
    for _ in range(epochs):
        order = list(range(n))
        for i in range(n - 1, 0, -1):
            s ^= s >> 12
            s = (s ^ (s << 25)) & mask
            s ^= s >> 27
            j = ((s * 2685821657736338717) & mask) % (i + 1)
            order[i], order[j] = order[j], order[i]
        out.append(np.array(order, np.int32))
    return out


# an output layer whose weights stream past the caches (its step runs beside the next
# forward pass) and one whose do not: the same bits as one step at a time
@pytest.mark.parametrize("hidden,nout,batch", [(544, 32000, 40), (544, 4000, 40), (544, 31002, 24)])
def test_training_equals_single_steps(hidden, nout, batch):
    n, epochs, lr = 3 * batch, 2, 1e-3
    rng = np.random.default_rng(nout)
    X = rng.uniform(0, 1, (n, 13)).astype(np.float32)
    T = rng.standard_normal((n, nout)).astype(np.float32)
    say(f"training 13-{hidden}x2-{nout} batch {batch}: {3 * epochs} steps, at once and one by one")
    nets = [surrogate.MLP(13, hidden, 2, nout, batch=batch, seed=3) for _ in range(2)]
    for net in nets:
        net.set_data(X, T)
    nets[0].train(epochs, lr=lr, seed=11)
    k = 0
    for order in _orders(n, 11, epochs):
        for b in range(3):
            prog = min(1.0, k / (3.0 * epochs))
            step_lr = np.float32(float(np.float32(lr)) * 0.5 * (1.0 + math.cos(math.pi * prog)))
            nets[1].train_step(order[b * batch:(b + 1) * batch], float(step_lr))
            k += 1
    for (Wa, ba), (Wb, bb) in zip(nets[0].weights(), nets[1].weights()):
        assert np.array_equal(Wa, Wb) and np.array_equal(ba, bb)
    for net in nets:
        net.close()
