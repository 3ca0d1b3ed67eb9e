"""Large results read back by several threads at once: each gets its own bytes, and
a small result does not wait for another thread's large one."""
import threading
import time

import numpy as np
import pytest

from seisfem_amd import surrogate

pytestmark = pytest.mark.gpu


def say(msg):
    print("[gpu-case]", msg, flush=True)


def together(jobs):
    errors = []

    def guarded(job):
        try:
            job()
        except BaseException as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=guarded, args=(job,)) for job in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_threads_read_their_own_weights():
    """More threads than there are sets of pinned buffers."""
    say("6 threads reading 13 MB of weights each")
    nets, ref = [], []
    for k in range(6):
        net = surrogate.MLP(13, 800, 1, 4001, batch=32, seed=k)
        W = np.random.default_rng(k).standard_normal((4001, 800)).astype(np.float32)
        b = np.random.default_rng(k + 9).standard_normal(4001).astype(np.float32)
        net.set_layer(1, W, b)
        nets.append(net)
        ref.append((W, b))

    def job(k):
        for _ in range(10):
            W, b = nets[k].layer(1)
            assert np.array_equal(W, ref[k][0]) and np.array_equal(b, ref[k][1])

    together([lambda k=k: job(k) for k in range(6)])
    for net in nets:
        net.close()


def test_a_small_result_does_not_wait_for_a_large_one():
    """4.5 MB beside 262 MB: alone 0.4 ms; taking turns it costs what the large one
    costs (9 ms), side by side about a millisecond."""
    large = surrogate.MLP(13, 2048, 1, 32000, batch=32, seed=1)
    small = surrogate.MLP(13, 1024, 1, 1100, batch=32, seed=2)
    say("4.5 MB of weights read beside 262 MB")
    for net in (large, small):
        net.layer(1)
    times = {"large": [], "small": []}
    stop = threading.Event()

    def read(net, name):
        t = time.perf_counter()
        net.layer(1)
        times[name].append(time.perf_counter() - t)

    def read_large():
        for _ in range(12):
            read(large, "large")
        stop.set()

    def read_small():
        while not stop.is_set():
            read(small, "small")

    together([read_large, read_small])
    assert np.median(times["small"]) < 0.7 * np.median(times["large"]), {k: np.median(v) for k, v in times.items()}
    for net in (large, small):
        net.close()
