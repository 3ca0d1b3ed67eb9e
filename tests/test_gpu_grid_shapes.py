"""Forms of the grid layout that larger meshes and batches take: 256-row patches,
padded lines, fields staged in two parts, tables of classes in FP64, a medium per
shot, several patch sizes in one multi-run.  Runs are held to the oracle (FP64) and to
64-shot lane groups, bit for bit."""
import numpy as np
import pytest

import oracle
from seisfem_amd import gpu, host

pytestmark = pytest.mark.gpu


def say(msg):
    print("[gpu-case]", msg, flush=True)


def bits_equal(a, b):
    a, b = (np.ascontiguousarray(v, np.float64) for v in (a, b))
    return a.shape == b.shape and np.array_equal(a.view(np.int64), b.view(np.int64))


def problem(tc, nx, ny, kind):
    """A mesh with M-PML layers on three sides.  "classes": the matrices rounded to 30 bits
    below their largest value, so that rows of equal stencils are equal bit for bit;
    "density": M alone changed at every row; "rows": every row has values of its own."""
    edge, pml = 10.0, 5
    en, x, y = host.mesh_structured(tc, nx, ny, 0.0, edge * nx, 0.0, edge * ny)
    n = x.size
    rho = 2000.0 + 0.3 * x + 0.7 * y if kind == "density" else np.full(n, 2000.0)
    vp = np.full(n, 3000.0)
    prob = host.build_problem(tc, en, x, y, rho, host.elastic_constants(rho, vp, vp / 1.73), vp, edge, pml, pml, 1,
                              bbox=(0.0, edge * nx, 0.0, edge * ny))
    csr = []
    for m, (p, j, v) in enumerate(prob["csr"]):
        if kind == "rows":
            v = v * (1.0 + 1.0e-6 * np.sin(np.arange(v.size)))
        elif m > 0 or kind == "classes":
            q = np.max(np.abs(v)) * 2.0 ** -30
            v = np.round(v / q) * q + 0.0        # (no negative zeros)
        csr.append((p, j, v))
    prob["csr"] = csr
    return prob, {host.Q4: 5.0e-4, host.Q9: 2.0e-4, host.T6: 1.5e-4}[tc]


def shots_of(n, shots, steps, seed):
    rng = np.random.default_rng(seed)
    nsteps = rng.integers(steps // 2, steps + 1, shots).astype(np.int32)
    nsteps[rng.integers(0, shots)] = steps
    return rng.integers(n // 4, 3 * n // 4, shots).astype(np.int32), nsteps


# sides that do not divide the patches; (patches x shots) on both sides of the counts up to
# which fields are staged at once (FP64 1024, 256 with reach 2)
CASES = [(host.Q4, 101, 97, "classes", 9), (host.Q4, 101, 97, "rows", 9), (host.Q4, 95, 33, "density", 26),
         (host.Q4, 127, 150, "classes", 30), (host.Q9, 45, 51, "classes", 24), (host.Q9, 31, 41, "density", 18),
         (host.T6, 63, 40, "classes", 7), (host.T6, 63, 40, "rows", 1), (host.Q9, 33, 17, "rows", 6)]


@pytest.mark.parametrize("tc,nx,ny,kind,shots", CASES)
def test_fp64_bit_identical_to_the_oracle(tc, nx, ny, kind, shots):
    prob, dt = problem(tc, nx, ny, kind)
    n, steps = prob["node_num"], 36
    src, nsteps = shots_of(n, shots, steps, nx)
    rec = np.arange(0, n, 1 + n // 400, dtype=np.int32)
    op = gpu.Operator(n, prob["csr"])
    md = gpu.Medium(op, prob["c"], prob["mass_lump"], prob["dirichlet"], prob["mpml"])
    say(f"grid FP64 {host.TYPE_NAMES[tc]} {nx}x{ny} {kind}, {shots} shots")
    run = gpu.Run(op, md, src, steps, rec, dt, 25.0, 0.01, nsteps=nsteps, guard_every=10)
    run.advance(steps)
    u, w = run.seismograms()
    for s in sorted({0, shots // 2, shots - 1, int(np.argmin(nsteps))}):
        k = int(nsteps[s])
        ref = oracle.oracle_masslump(prob, src[s], k + 2, rec, dt, 25.0, 0.01)
        assert ref["status"] == k and np.max(np.abs(ref["seis_u"])) > 0
        assert bits_equal(u[s, :k], ref["seis_u"]) and bits_equal(w[s, :k], ref["seis_w"]), s
        U, W = run.snapshot(s)
        assert bits_equal(U[rec], ref["seis_u"][-1]) and bits_equal(W[rec], ref["seis_w"][-1])
    for h in (run, md, op):
        h.close()


# (patches x shots) on both sides of 2048; the last two with a medium per shot
@pytest.mark.parametrize("prec", [gpu.FP64, gpu.FP32, gpu.FP32_KAHAN16])
@pytest.mark.parametrize("tc,nx,ny,kind,shots,media", [
    (host.Q9, 97, 111, "classes", 37, False), (host.Q4, 63, 80, "classes", 40, False),
    (host.Q4, 150, 163, "density", 23, False), (host.T6, 60, 45, "rows", 19, False),
    (host.Q4, 101, 97, "classes", 18, True), (host.Q9, 62, 51, "density", 47, True)])
def test_forms_equal_lane_groups(prec, tc, nx, ny, kind, shots, media):
    prob, dt = problem(tc, nx, ny, kind)
    n, steps = prob["node_num"], 24
    src, nsteps = shots_of(n, shots, steps, ny)
    rec = np.arange(0, n, 1 + n // 500, dtype=np.int32)
    op = gpu.Operator(n, prob["csr"])
    md = [gpu.Medium(op, [a * (1.0 + 0.002 * s) for a in prob["c"]], prob["mass_lump"] * (1.0 + 0.001 * s),
                     prob["dirichlet"], [a * (1.0 - 0.003 * s) for a in prob["mpml"]])
          for s in range(shots if media else 1)]
    say(f"grid precision {prec} {host.TYPE_NAMES[tc]} {nx}x{ny} {kind}, {shots} shots, media per shot: {media}")
    got = []
    for kw in (dict(), dict(shots_per_lane_group=64, kernel_variant=1)):
        run = gpu.Run(op, md if media else md[0], src, steps, rec, dt, 25.0, 0.004, precision=prec, nsteps=nsteps,
                      guard_every=9, **kw)
        run.advance(13)
        run.advance(steps)
        got.append(run.seismograms() + run.snapshot(shots - 1))
        run.close()
    assert np.max(np.abs(got[0][0])) > 0
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    for h in md + [op]:
        h.close()


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.FP32_KAHAN])
def test_several_patch_sizes_and_batches_in_one_multi_run(prec):
    """64-, 128- and 256-row patches, batches whose shots end at different steps among them."""
    specs = [(host.Q4, 20, 31, "classes", 5), (host.Q9, 15, 18, "rows", 4), (host.Q4, 101, 97, "density", 9),
             (host.T6, 50, 33, "classes", 12), (host.Q9, 45, 51, "classes", 7)]
    say(f"multi-run of {len(specs)} batches with 64 to 256 rows a patch, precision {prec}")
    steps, keep, makers = 26, [], []
    for tc, nx, ny, kind, shots in specs:
        prob, dt = problem(tc, nx, ny, kind)
        n = prob["node_num"]
        src, nsteps = shots_of(n, shots, steps, nx + ny)
        op = gpu.Operator(n, prob["csr"])
        md = gpu.Medium(op, prob["c"], prob["mass_lump"], prob["dirichlet"], prob["mpml"])
        keep += [md, op]
        makers.append(lambda op=op, md=md, src=src, nsteps=nsteps, n=n, dt=dt: gpu.Run(
            op, md, src, steps, np.arange(0, n, 1 + n // 300, dtype=np.int32), dt, 25.0, 0.006, precision=prec,
            nsteps=nsteps, guard_every=8, block=256))
    runs = [mk() for mk in makers]
    multi = gpu.Multi(runs)
    multi.advance(11)
    multi.advance(steps)
    together = [r.seismograms() + r.snapshot(0) for r in runs]
    multi.close()
    for mk, got in zip(makers, together):
        run = mk()
        run.advance(steps)
        ref = run.seismograms() + run.snapshot(0)
        run.close()
        assert np.max(np.abs(ref[0])) > 0
        for a, b in zip(got, ref):
            assert np.array_equal(a, b)
    for h in runs + keep:
        h.close()
