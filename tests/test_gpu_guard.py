"""The energy guard's sums against the fields they are taken of, in every layout
of the state, and batches of more shots than a launch takes blocks in its other
dimensions."""
import numpy as np
import pytest

from seisfem_amd import gpu, host

pytestmark = pytest.mark.gpu


def say(msg):
    print("[gpu-case]", msg, flush=True)


def objects(tc, nx, ny):
    en, x, y = host.mesh_structured(tc, nx, ny, 0.0, 10.0 * nx, 0.0, 10.0 * ny)
    rho, vp = np.full(x.size, 2000.0), np.full(x.size, 3000.0)
    prob = host.build_problem(tc, en, x, y, rho, host.elastic_constants(rho, vp, vp / 1.73), vp, 10.0, 3, 3, 1,
                              bbox=(0.0, 10.0 * nx, 0.0, 10.0 * ny))
    op = gpu.Operator(prob["node_num"], prob["csr"])
    return op, gpu.Medium(op, prob["c"], prob["mass_lump"], prob["dirichlet"], prob["mpml"])


# more nodes than one block sums; lines with and without padding, lane groups of 1, 4, 16 and
# 64 shots, shots that end before the check
@pytest.mark.parametrize("prec", [gpu.FP64, gpu.FP32_KAHAN16])
@pytest.mark.parametrize("nx,ny,shots,launch", [
    (47, 60, 1, {}), (47, 60, 5, {}), (62, 70, 5, {}), (47, 60, 1, dict(shots_per_lane_group=1)),
    (47, 60, 5, dict(shots_per_lane_group=4)), (47, 60, 5, dict(shots_per_lane_group=16)),
    (47, 60, 70, dict(shots_per_lane_group=64))])
def test_energy_is_that_of_the_fields(prec, nx, ny, shots, launch):
    say(f"energy guard Q4 {nx}x{ny}, {shots} shots, precision {prec}, {launch}")
    op, md = objects(host.Q4, nx, ny)
    n, steps = op.node_num, 60
    src = np.linspace(n // 3, 2 * n // 3, shots).astype(np.int32)
    nsteps = (steps - (np.arange(shots) * 7) % 25).astype(np.int32)
    run = gpu.Run(op, md, src, steps, np.zeros(0, np.int32), 5.0e-4, 25.0, 0.02, amplitude=1.0e5, precision=prec,
                  nsteps=nsteps, guard_every=20, **launch)
    run.advance(steps)
    last = run.energy(8)[3]                     # the check after step 60
    for s in range(0, shots, 1 + shots // 7):
        U, W = run.snapshot(s)
        ref = np.array([np.sum(U * U), np.sum(W * W)])
        assert np.all(ref > 0) and np.allclose(last[s], ref, rtol=1e-12, atol=0), (s, last[s], ref)
    for h in (run, md, op):
        h.close()


def test_more_shots_than_blocks_in_a_second_dimension():
    """66000 shots (65536 blocks is the limit there): the default layout against lane groups."""
    op, md = objects(host.Q4, 15, 15)
    n, steps, shots = op.node_num, 6, 66000
    say(f"{shots} shots on {n} nodes")
    src = (40 + np.arange(shots) % 170).astype(np.int32)
    out = []
    for launch in (dict(), dict(shots_per_lane_group=64)):
        run = gpu.Run(op, md, src, steps, np.arange(100, 103, dtype=np.int32), 5.0e-4, 25.0, 0.002, guard_every=3,
                      **launch)
        run.advance(steps)
        out.append(run.seismograms() + run.snapshot(shots - 1) + (run.energy(2),))
        run.close()
    assert np.max(np.abs(out[0][0])) > 0
    for a, b in zip(out[0][:4], out[1][:4]):
        assert np.array_equal(a, b)
    assert np.allclose(out[0][4], out[1][4], rtol=1e-12, atol=0)
    for h in (md, op):
        h.close()
