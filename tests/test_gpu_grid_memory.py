"""Device memory of the grid layout's tables: kept only where a run reads them, and
given back when the memory does not suffice for the layout."""
import ctypes as C

import numpy as np
import pytest

from seisfem_amd import gpu, host

pytestmark = pytest.mark.gpu
MB = 1 << 20


def say(msg):
    print("[gpu-case]", msg, flush=True)


def hip():
    return C.CDLL("libamdhip64.so")


def free_bytes():
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def objects(tc, nx, ny):
    """A mesh whose rows all differ: seven values per row beside the operator's own."""
    bbox = (0.0, 10.0 * nx, 0.0, 10.0 * ny)
    en, x, y = host.mesh_structured(tc, nx, ny, *bbox)
    xm = x
    x = xm + 0.8 * np.sin(0.05 * y) * xm / bbox[1]
    y = y + 0.6 * np.sin(0.07 * xm) * np.sin(np.pi * y / bbox[3])
    rho, vp = 2000.0 + 0.3 * x, np.full(x.size, 3000.0)
    prob = host.build_problem(tc, en, x, y, rho, host.elastic_constants(rho, vp, vp / 1.73), vp, 10.0, 5, 5, 1, bbox=bbox)
    return prob


def open_op(prob):
    op = gpu.Operator(prob["node_num"], prob["csr"])
    return op, gpu.Medium(op, prob["c"], prob["mass_lump"], prob["dirichlet"], prob["mpml"])


def open_run(prob, op, md, shots, **kw):
    n = prob["node_num"]
    src = np.linspace(n // 3, 2 * n // 3, shots).astype(np.int32)
    return gpu.Run(op, md, src, 20, np.arange(0, n, 1 + n // 50, dtype=np.int32), 1.0e-4, 25.0, 0.01, **kw)


def test_tables_of_a_declined_layout_are_not_built():
    """More than 32 shots with seven values per row take lane groups: the operator holds
    no copy of its matrices for a layout that no run has (60 bytes per nonzero)."""
    prob = objects(host.Q4, 300, 300)
    op, md = open_op(prob)
    open_run(prob, op, md, 1, shots_per_lane_group=1).close()
    say("40 shots on a mesh of distinct rows: memory kept by the operator")
    before = free_bytes()
    open_run(prob, op, md, 40).close()
    kept = before - free_bytes()
    assert kept < 12 * MB < 60 * op.nnz // 2, kept
    for h in (md, op):
        h.close()


def test_layout_that_does_not_fit_gives_its_memory_back():
    """With memory for the tables or for the run, but not for both, a default run is
    created in the layout without tables, as one of that layout is."""
    prob = objects(host.Q9, 400, 300)
    op, md = open_op(prob)
    say("default run where the grid layout does not fit")
    # (both layouts' kernels, streams and graphs have been used once)
    for kw in (dict(), dict(shots_per_lane_group=1)):
        run = open_run(prob, op, md, 1, **kw)
        run.advance(20)
        ref = run.seismograms()
        run.close()
    md.close()
    op.close()
    op, md = open_op(prob)
    start = free_bytes()
    run = open_run(prob, op, md, 1, shots_per_lane_group=1)
    need = start - free_bytes()
    run.close()
    open_run(prob, op, md, 1).close()
    tables = start - free_bytes()
    assert need > 150 * MB and tables > need, (need, tables)
    md.close()
    op.close()
    op, md = open_op(prob)
    target, holds = tables + need // 2, []
    try:
        # (memory freed before may be counted as free only after the next allocation)
        for _ in range(4):
            left = free_bytes()
            if left <= target:
                break
            holds.append(C.c_void_p())
            assert hip().hipMalloc(C.byref(holds[-1]), C.c_size_t(left - target)) == 0
        left = free_bytes()
        assert need < left < tables + need, (left, need, tables)
        run = open_run(prob, op, md, 1)
        run.advance(20)
        got = run.seismograms()
        run.close()
        assert left - free_bytes() < 64 * MB
    finally:
        for h in holds:
            assert hip().hipFree(h) == 0
    assert np.max(np.abs(ref[0])) > 0
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])
    for h in (md, op):
        h.close()
