"""Multi-runs of runs whose launch shape is left to the library: every
combination of shot counts, mesh sizes and meshes whose runs share a block
without the grid layout is taken, and gives each run's own results."""
import numpy as np
import pytest

from seisfem_amd import gpu, host

pytestmark = pytest.mark.gpu


def say(msg):
    print("[gpu-case]", msg, flush=True)


def problem(tc, nx, ny, shuffled=False):
    """A mesh of constant medium; shuffled: its nodes renumbered at random (no lines)."""
    en, x, y = host.mesh_structured(tc, nx, ny, 0.0, 10.0 * nx, 0.0, 10.0 * ny)
    if shuffled:
        new = np.random.default_rng(nx).permutation(x.size)
        xs, ys = np.empty_like(x), np.empty_like(y)
        xs[new], ys[new] = x, y
        en, x, y = new.astype(np.int32)[en - 1] + 1, xs, ys
    rho, vp = np.full(x.size, 2000.0), np.full(x.size, 3000.0)
    return host.build_problem(tc, en, x, y, rho, host.elastic_constants(rho, vp, vp / 1.73), vp, 10.0, 3, 3, 1,
                              bbox=(0.0, 10.0 * nx, 0.0, 10.0 * ny))


def make_runs(specs, prec, steps, **kw):
    """One run per (type, nx, ny, shots, shuffled, launch), and the objects they need."""
    keep, runs = [], []
    for tc, nx, ny, shots, shuffled, launch in specs:
        prob = problem(tc, nx, ny, shuffled)
        n = prob["node_num"]
        rng = np.random.default_rng(nx + shots)
        op = gpu.Operator(n, prob["csr"])
        md = gpu.Medium(op, prob["c"], prob["mass_lump"], prob["dirichlet"], prob["mpml"])
        nsteps = rng.integers(steps // 2, steps + 1, shots).astype(np.int32)
        nsteps[0] = steps
        src = rng.integers(n // 4, 3 * n // 4, shots).astype(np.int32)
        keep += [op, md]
        runs.append(lambda op=op, md=md, src=src, nsteps=nsteps, n=n, launch=launch: gpu.Run(
            op, md, src, steps, np.arange(0, n, 1 + n // 97, dtype=np.int32), 5.0e-4, 25.0, 0.03, precision=prec,
            nsteps=nsteps, guard_every=20, **dict(kw, **launch)))
    return keep, runs


def seismograms(makers, multi, schedule=((0, 1 << 20),)):
    runs = [mk() for mk in makers]
    if multi:
        m = gpu.Multi(runs)
        for blocks, steps in schedule:
            m.set_persistent(blocks)
            m.advance(steps)
    else:
        for r in runs:
            r.advance(1 << 20)
    out = [r.seismograms() + r.snapshot(r.nshots - 1) for r in runs]
    if multi:
        m.close()
    for r in runs:
        r.close()
    return out


def assert_same(got, ref):
    for a, b in zip(got, ref):
        assert np.max(np.abs(b[0])) > 0
        for x, y in zip(a, b):
            assert np.array_equal(x, y)


# an FP32 line of shots beside a survey in lane groups; two FP64 lines on meshes either
# side of 2^18 nodes; an FP64 line on a mesh numbered line by line beside one that is not;
# single shots with and without the grid layout
@pytest.mark.parametrize("prec,specs", [
    (gpu.FP32, [(host.Q4, 20, 25, 8, False, {}), (host.Q4, 22, 19, 64, False, {})]),
    (gpu.FP64, [(host.Q4, 300, 333, 8, False, {}), (host.Q4, 600, 499, 8, False, {})]),
    (gpu.FP64, [(host.Q4, 20, 25, 8, False, {}), (host.Q4, 21, 17, 8, True, {})]),
    (gpu.FP64, [(host.Q4, 20, 25, 1, False, {}), (host.Q9, 9, 8, 1, True, {}),
                (host.Q4, 30, 22, 1, False, dict(shots_per_lane_group=1, kernel_variant=1))])])
def test_default_shapes_share_a_multi_run(prec, specs):
    say(f"multi-run of default shapes, precision {prec}: {[s[:5] for s in specs]}")
    keep, makers = make_runs(specs, prec, 40)
    assert_same(seismograms(makers, True), seismograms(makers, False))
    for h in keep:
        h.close()


@pytest.mark.parametrize("shots", [1, 3, 64])
def test_tuned_launch_shares_a_multi_run_with_sliced_models(shots):
    """A launch the tuner returns names its block: runs of it go into one multi-run
    with single-shot models that take the same block."""
    from seisfem_amd import autotune
    own = autotune.run_kwargs(dict(autotune.candidates(shots)[0], row_order=None, row_order_name="node"))
    assert own["shots_per_lane_group"] == 0 and own["kernel_variant"] == 0
    say(f"the library's own launch of {shots} shots beside sliced models")
    model = dict(block=own["block"], shots_per_lane_group=1, kernel_variant=8, xcd_remap=False)
    keep, makers = make_runs([(host.Q4, 30, 41, shots, False, own), (host.Q4, 20, 23, 1, False, model),
                              (host.Q9, 9, 8, 1, False, model)], gpu.FP32_KAHAN16, 40)
    assert_same(seismograms(makers, True), seismograms(makers, False))
    for h in keep:
        h.close()


# batches too small to fill the GPU alone: default shapes in the grid layout with patches
# of 64 and 128 rows (reach 1 and 2), and beside a lane-group launch
@pytest.mark.parametrize("prec,specs", [
    (gpu.FP64, [(host.Q4, 12, 13, 70, False, {}), (host.T6, 4, 5, 20, False, {}),
                (host.Q4, 11, 11, 45, False, dict(block=256, shots_per_lane_group=32, kernel_variant=5))]),
    (gpu.FP64, [(host.Q4, 12, 13, 70, False, {}), (host.Q9, 5, 6, 19, False, {})]),
    (gpu.FP32_KAHAN16, [(host.Q4, 20, 9, 30, False, {}), (host.Q9, 6, 5, 40, False, {})])])
def test_persistent_schedule_of_default_batches(prec, specs):
    say(f"persistent schedule of default batches, precision {prec}: {[s[:5] for s in specs]}")
    keep, makers = make_runs(specs, prec, 60)
    ref = seismograms(makers, True)
    for schedule in ([(1, 37), (1, 60)], [(2, 60)], [(0, 20), (2, 15), (0, 60)]):
        assert_same(seismograms(makers, True, schedule), ref)
    for h in keep:
        h.close()


def test_persistent_schedule_refuses_what_needs_launches_of_its_own():
    """Few shots in a batch, and single shots beside batches, as without the grid layout."""
    say("persistent schedule: refused combinations")
    for specs in ([(host.Q4, 12, 13, 8, False, {})],
                  [(host.Q4, 12, 13, 70, False, {}), (host.Q4, 12, 13, 1, False, dict(block=256))]):
        keep, makers = make_runs(specs, gpu.FP64, 40)
        runs = [mk() for mk in makers]
        multi = gpu.Multi(runs)
        with pytest.raises(gpu.NativeError) as e:
            multi.set_persistent(1)
        assert e.value.code == -1
        multi.close()
        for h in runs + keep:
            h.close()
