"""Workloads of the GPU time loop and of the surrogate, for timing and for comparing outputs.

Every case goes through the public Python entry points (``seisfem_amd.gpu`` and
``seisfem_amd.surrogate``) with their default launch shapes, as a program that
links the library does; the many-model batch takes the launch shape that
``FEMGenerator`` gives it.  Kinds of case:

  shots     shots of one model stepped by one ``gpu.Run``: back to rest, the step
            loop, seismograms and one snapshot
  media     one model per shot on a shared mesh (``sfg_run_create_media``): the
            form in which the surrogate's training shots are computed
  multi     models of uneven mesh size and length in one ``gpu.Multi``, from
            creation to seismograms (a multi-run steps its models once)
  dt        the CFL estimate ``gpu.estimate_dt``
  train     Adam epochs of the surrogate network over its resident data
  predict   inference of the surrogate network on host arrays

The inputs (meshes, the seven matrices, media, M-PML profiles, stations) are
built here in plain numpy, and ``exact`` steps the same equations in 64 bits in
plain torch.
"""
import functools
import math

import numpy as np
import torch

from seisfem_amd import gpu, surrogate

PRECISION = {"fp64": gpu.FP64, "fp32": gpu.FP32, "kahan": gpu.FP32_KAHAN, "kahan16": gpu.FP32_KAHAN16}
EDGE = 10.0                    # element edge in metres
# time steps inside each element's stability limit at 10 m and 4500 m/s
DT = {"q4": 5.0e-4, "q9": 2.5e-4, "t6": 2.0e-4}
ORDER = {"q4": 1, "q9": 2, "t6": 2}


def listed():
    return [
        # one short shot on a tiny mesh, as in the smoke run: launch latency
        dict(name="shot_q4_16", kind="shots", mesh="q4", nx=16, ny=16, shots=1, steps=60, prec="fp64"),
        # the reference's single-shot setup, homogeneous-size Q4 200 x 200, in FP64
        dict(name="shot_q4_200", kind="shots", mesh="q4", nx=200, ny=200, shots=1, steps=300, prec="fp64"),
        # a Q9 mesh beyond the caches, FP32 with compensated displacements
        dict(name="shot_q9_300_kahan", kind="shots", mesh="q9", nx=300, ny=300, shots=1, steps=200, prec="kahan"),
        # triangles, odd sizes, an explosive (distributed) source, FP64
        dict(name="shot_t6_explosive", kind="shots", mesh="t6", nx=101, ny=203, shots=1, steps=250, prec="fp64",
             explosive=True),
        # a line of shots handed over at once by the drop-in driver, FP64
        dict(name="line_6_q4_fp64", kind="shots", mesh="q4", nx=150, ny=250, shots=6, steps=200, prec="fp64"),
        # the headline: 128 shots of uneven length on Q4 400 x 400, FP32 with bfloat16 Kahan terms
        dict(name="survey_128_q4_kahan16", kind="shots", mesh="q4", nx=400, ny=400, shots=128, steps=120,
             prec="kahan16"),
        # the same survey's accuracy run, batched FP64, fewer shots of it
        dict(name="survey_64_q4_fp64", kind="shots", mesh="q4", nx=300, ny=300, shots=64, steps=80, prec="fp64"),
        # a survey of odd size on Q9 elements
        dict(name="survey_37_q9_kahan", kind="shots", mesh="q9", nx=97, ny=111, shots=37, steps=120, prec="kahan"),
        # training shots of the surrogate: 128 layered models on one mesh
        dict(name="media_128_q4", kind="media", mesh="q4", nx=200, ny=200, shots=128, steps=160, prec="fp32"),
        # independent models of uneven size stepped together
        dict(name="multi_6_q4", kind="multi", mesh="q4", nx=200, ny=150, models=6, steps=400, prec="kahan16"),
        # the surrogate's network: epochs of Adam steps, and inference on a ragged number of models
        dict(name="train_32000", kind="train", hidden=1024, nout=32000, batch=256, n=2000, epochs=24),
        dict(name="predict_1000", kind="predict", hidden=1024, nout=32000, batch=256, n=1000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["shot", "shot", "shots", "shots", "media", "multi", "dt", "train", "predict"])
    if kind == "train":
        hidden = rng.choice([256, 512, 1024])
        return dict(kind=kind, hidden=hidden, nout=rng.choice([500, 4000, 8000, 16000, 32000]),
                    batch=rng.choice([64, 128, 256]), n=_log_int(rng, 300, 2000), epochs=rng.randint(2, 16))
    if kind == "predict":
        return dict(kind=kind, hidden=rng.choice([256, 512, 1024]), nout=rng.choice([500, 8000, 32000]), batch=256,
                    n=_log_int(rng, 1, 1000))
    mesh = rng.choice(["q4", "q4", "q9", "t6"])
    most = {"q4": 400, "q9": 250, "t6": 250}[mesh] if kind in ("shot", "dt") else {"q4": 300, "q9": 130, "t6": 130}[mesh]
    nx, ny = _log_int(rng, 12, most), _log_int(rng, 12, most)
    if kind == "dt":
        return dict(kind=kind, mesh=mesh, nx=nx, ny=ny)
    prec = rng.choice(["fp64", "fp64", "fp32", "kahan", "kahan16"])
    steps = rng.randint(40, 160)
    if kind == "shot":
        return dict(kind="shots", mesh=mesh, nx=nx, ny=ny, shots=1, steps=steps, prec=prec,
                    explosive=rng.random() < 0.3)
    if kind == "multi":
        return dict(kind=kind, mesh=mesh, nx=nx, ny=ny, models=rng.randint(2, 6), steps=steps, prec=prec)
    # no more shot-nodes than the largest survey above
    shots = _log_int(rng, 2, 128)
    return dict(kind=kind, mesh=mesh, nx=nx, ny=ny, shots=shots, steps=steps, prec=prec if kind == "shots" else "fp32")


# ---- meshes and matrices --------------------------------------------------------

def _shape(mesh):
    """Node coordinates of the reference cell and its monomials (powers of r and s).
    A cell is one quadrilateral, or for triangles one half of it."""
    if mesh == "q4":
        return [(0, 0), (1, 0), (0, 1), (1, 1)], [(0, 0), (1, 0), (0, 1), (1, 1)]
    if mesh == "q9":
        g = (0, 0.5, 1)
        return [(r, s) for s in g for r in g], [(a, b) for b in range(3) for a in range(3)]
    return [(0, 0), (1, 0), (0, 1), (0.5, 0), (0.5, 0.5), (0, 0.5)], [(0, 0), (1, 0), (0, 1), (1, 1), (2, 0), (0, 2)]


def _basis(mesh, r, s):
    """Values and derivatives of the shape functions at the points (r, s): [points][nodes]."""
    nodes, mono = _shape(mesh)
    V = np.array([[x ** a * y ** b for a, b in mono] for x, y in nodes], float)
    C = np.linalg.inv(V)                       # monomials -> shape functions
    f = np.stack([r ** a * s ** b for a, b in mono], 1)
    fr = np.stack([a * r ** max(a - 1, 0) * s ** b for a, b in mono], 1)
    fs = np.stack([b * r ** a * s ** max(b - 1, 0) for a, b in mono], 1)
    return f @ C, fr @ C, fs @ C


def _quadrature(mesh):
    g, w = np.polynomial.legendre.leggauss(5)
    g, w = (g + 1) / 2, w / 2
    r, s = (a.reshape(-1) for a in np.meshgrid(g, g, indexing="ij"))
    w = np.outer(w, w).reshape(-1)
    if mesh == "t6":                           # the square folded onto the unit triangle
        return r, s * (1 - r), w * (1 - r)
    return r, s, w


@functools.lru_cache(maxsize=4)
def _mesh(mesh, nx, ny):
    """Coordinates and, on one sorted pattern, the matrices G (density 1), S1..S6 of an
    nx x ny grid of cells: x is height (fastest in the node numbering), y horizontal."""
    p = ORDER[mesh]
    line, lines = p * nx + 1, p * ny + 1
    n = line * lines
    ids = np.arange(n)
    x, y = (ids % line) * (EDGE / p), (ids // line) * (EDGE / p)
    ix, iy = (a.reshape(-1) for a in np.meshgrid(np.arange(nx), np.arange(ny), indexing="ij"))
    corner = iy * p * line + ix * p
    nodes, _ = _shape(mesh)
    off = [[int(round(p * r)) + line * int(round(p * s)) for r, s in nodes]]
    sign = [1.0]
    if mesh == "t6":                           # the other half of each cell: the same triangle turned round
        off.append([int(round(p * (1 - r))) + line * int(round(p * (1 - s))) for r, s in nodes])
        sign.append(-1.0)
    r, s, w = _quadrature(mesh)
    f, fr, fs = _basis(mesh, r, s)
    rows, cols, vals = [], [], [[] for _ in range(7)]
    for o, sg in zip(off, sign):
        dx, dy = fr * (sg / EDGE), fs * (sg / EDGE)
        q = w[:, None, None] * EDGE * EDGE
        pair = lambda a, b: (q * a[:, :, None] * b[:, None, :]).sum(0)  # noqa: E731
        elem = [pair(f, f), pair(dx, dx), pair(dy, dy), pair(dx, dy), pair(dy, dx), pair(f, dx), pair(f, dy)]
        dof = corner[:, None] + np.array(o)[None, :]
        rows.append(np.repeat(dof, len(o), 1).reshape(-1))
        cols.append(np.tile(dof, (1, len(o))).reshape(-1))
        for m in range(7):
            vals[m].append(np.tile(elem[m].reshape(-1), len(corner)))
    key = np.concatenate(rows) * n + np.concatenate(cols)
    order = np.argsort(key, kind="stable")
    key = key[order]
    first = np.flatnonzero(np.concatenate([[True], key[1:] != key[:-1]]))
    row, col = key[first] // n, (key[first] % n).astype(np.int32)
    ptr = np.concatenate([[0], np.cumsum(np.bincount(row, minlength=n))]).astype(np.int32)
    mats = [np.add.reduceat(np.concatenate(v)[order], first) for v in vals]
    return dict(n=n, line=line, lines=lines, x=x, y=y, h=EDGE / p, row=row, col=col, ptr=ptr, mats=mats,
                Lx=nx * EDGE, Ly=ny * EDGE)


def _lumped(M, rho):
    """Diagonal of diag(rho) G scaled to the total mass (HRZ lumping)."""
    diag = np.zeros(M["n"])
    on = M["row"] == M["col"]
    diag[M["row"][on]] = M["mats"][0][on]
    total = np.bincount(M["row"], weights=M["mats"][0], minlength=M["n"])
    return rho * diag * (np.dot(rho, total) / np.dot(rho, diag))


def _damping(M, vpmax):
    """M-PML profiles dx, dy, dxx, dyy, p dxx, p dyy on the bottom and both sides
    (the top, x = xmax, is free)."""
    nl = max(2, min(20, min(M["Lx"], M["Ly"]) // EDGE // 5))
    t, p = nl * EDGE, 0.15
    d0 = 3.0 * vpmax * math.log10(1.0 / 1e-4) / (2.0 * t)
    ax = np.maximum(t - M["x"], 0.0) / t
    lo, hi = np.maximum(t - M["y"], 0.0) / t, np.maximum(M["y"] - (M["Ly"] - t), 0.0) / t
    bx, by = d0 * ax * ax, d0 * (lo * lo + hi * hi)
    dxx, dyy = -2.0 * d0 * ax / t, 2.0 * d0 * (hi - lo) / t
    return [bx + p * by, by + p * bx, dxx, dyy, p * dxx, p * dyy]


def _model(M, rng):
    """A layered isotropic model: density, stiffnesses, lumped mass, profiles."""
    depth = M["Lx"] - M["x"]
    cuts = np.sort(rng.uniform(0.1, 0.9, 3)) * M["Lx"]
    vp = np.sort(rng.uniform(1500.0, 4500.0, 4))[np.searchsorted(cuts, depth, side="right")]
    vs = vp / 1.73
    rho = 310.0 * vp ** 0.25
    c44, c11 = rho * vs * vs, rho * vp * vp
    return dict(rho=rho, c=[c11, c11 - 2 * c44, c11, c44], mass=_lumped(M, rho), mpml=_damping(M, float(vp.max())))


def _clamped(M):
    eps = 0.1 * M["h"]
    return ((M["x"] < eps) | (M["y"] < eps) | (M["y"] > M["Ly"] - eps)).astype(np.int32)


def _node(M, depth, y):
    ix = np.rint((M["Lx"] - depth) / M["h"]).astype(int)
    iy = np.rint(np.asarray(y) / M["h"]).astype(int)
    return (np.clip(iy, 0, M["lines"] - 1) * M["line"] + np.clip(ix, 0, M["line"] - 1)).astype(np.int32)


def _explosion(M, node):
    """An isotropic moment at a node as forces on it and its four grid neighbours."""
    nodes = np.array([node - 1, node + 1, node - M["line"], node + M["line"]], np.int32)
    return nodes, np.array([[-0.5, 0.0], [0.5, 0.0], [0.0, -0.5], [0.0, 0.5]]) / M["h"]


def _job(case, seed):
    """Plain arrays of one shots / media case."""
    rng = np.random.default_rng(seed)
    M = _mesh(case["mesh"], case["nx"], case["ny"])
    S, T = case["shots"], case["steps"]
    job = dict(M=M, S=S, T=T, dt=DT[case["mesh"]], f0=12.0, t0=0.03, flags=_clamped(M),
               models=[_model(M, rng) for _ in range(S if case["kind"] == "media" else 1)])
    job["src"] = np.atleast_1d(_node(M, 2 * EDGE, rng.uniform(0.25, 0.75, S) * M["Ly"]))
    job["rec"] = np.unique(_node(M, 0.0, np.linspace(0.0, M["Ly"], min(201, M["lines"]))))
    # uneven lengths in a survey; a lone shot and a batch of training models run to the end
    job["nsteps"] = np.full(S, T, np.int32)
    if case["kind"] == "shots" and S > 1:
        job["nsteps"] = rng.integers(T // 2, T + 1, S).astype(np.int32)
        job["nsteps"][rng.integers(0, S)] = T
    job["sources"] = [_explosion(M, int(k)) for k in job["src"]] if case.get("explosive") else None
    job["amplitude"] = 1.0 if case["kind"] == "media" else 1.0e7
    return job


def _operator(M, rho):
    scaled = M["mats"][0] if rho is None else M["mats"][0] * rho[M["row"]]
    return gpu.Operator(M["n"], [(M["ptr"], M["col"], v) for v in [scaled] + M["mats"][1:]])


def _medium(op, M, model, flags):
    return gpu.Medium(op, model["c"], model["mass"], flags, model["mpml"])


def _shots_state(case, seed):
    job = _job(case, seed)
    M = job["M"]
    if case["kind"] == "media":
        op = _operator(M, None)
        md = []
        for model in job["models"]:
            md.append(_medium(op, M, model, job["flags"]))
            md[-1].set_row_scale(model["rho"])
        launch = surrogate.FEMGenerator.LAUNCH
    else:
        op = _operator(M, job["models"][0]["rho"])
        md = _medium(op, M, job["models"][0], job["flags"])
        launch = {}
    run = gpu.Run(op, md, job["src"], job["T"], job["rec"], job["dt"], job["f0"], job["t0"],
                  amplitude=job["amplitude"], precision=PRECISION[case["prec"]], nsteps=job["nsteps"],
                  sources=job["sources"], **launch)
    return dict(kind="shots", run=run, steps=job["T"], dtype=_dtype(case), keep=(op, md))


def _dtype(case):
    # seismograms and snapshots come as FP64 arrays; those of an FP32 run hold FP32 values
    return np.float64 if case["prec"] == "fp64" else np.float32


def _multi_jobs(case, seed):
    jobs = []
    rng = np.random.default_rng(seed)
    for k in range(case["models"]):
        # sizes and lengths between half and all of the case's
        size = np.maximum(12, np.rint(np.array([case["nx"], case["ny"]]) * (1.0 - 0.5 * k / case["models"]))).astype(int)
        one = dict(kind="shots", mesh=case["mesh"], nx=int(size[0]), ny=int(size[1]), shots=1, steps=case["steps"])
        job = _job(one, seed * 1000 + k)
        job["nsteps"] = np.array([rng.integers(case["steps"] // 2, case["steps"] + 1) if k else case["steps"]], np.int32)
        jobs.append(job)
    return jobs


# ---- the surrogate's network ----------------------------------------------------

NIN = surrogate.NIN


def _weights(case, seed):
    g = torch.Generator().manual_seed(seed)
    widths = [NIN] + [case["hidden"]] * 3 + [case["nout"]]
    out = []
    for i, o in zip(widths[:-1], widths[1:]):
        a = math.sqrt(6.0 / i) * (0.5 if o == case["nout"] else 1.0)
        out.append((((torch.rand(o, i, generator=g) * 2 - 1) * a).numpy(),
                    ((torch.rand(o, generator=g) * 2 - 1) * 0.05).numpy()))
    return out


def _models_in(case, seed):
    return surrogate.sample_models(case["n"], seed)["X"]


def _traces(case, seed):
    """Normalised band-limited traces: a wavelet arriving at a time set by each model."""
    n, nout = case["n"], case["nout"]
    g = torch.Generator().manual_seed(seed + 1)
    t0 = torch.rand(n, 1, generator=g) * nout
    f = 0.02 + 0.05 * torch.rand(n, 1, generator=g)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    a = ((torch.arange(nout, device=dev) - t0.to(dev)) * f.to(dev)) ** 2
    return ((1 - 2 * a) * torch.exp(-a)).cpu().numpy()


# ---- the measured interface -----------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("shots", "media"):
        return _shots_state(case, seed)
    if kind == "multi":
        jobs = _multi_jobs(case, seed)
        for j in jobs:
            j["op"] = _operator(j["M"], j["models"][0]["rho"])
            j["md"] = _medium(j["op"], j["M"], j["models"][0], j["flags"])
        return dict(kind=kind, jobs=jobs, prec=PRECISION[case["prec"]], steps=case["steps"], dtype=_dtype(case))
    if kind == "dt":
        M = _mesh(case["mesh"], case["nx"], case["ny"])
        model = _model(M, np.random.default_rng(seed))
        op = _operator(M, model["rho"])
        return dict(kind=kind, op=op, md=_medium(op, M, model, _clamped(M)))
    net = surrogate.MLP(NIN, case["hidden"], 3, case["nout"], batch=case["batch"], seed=seed % 1000)
    if kind == "predict":
        net.set_weights(_weights(case, seed))
        return dict(kind=kind, net=net, X=_models_in(case, seed))
    net.set_data(_models_in(case, seed), _traces(case, seed))
    return dict(kind=kind, net=net, epochs=case["epochs"], seed=seed % 1000)


def run(state):
    kind = state["kind"]
    if kind == "shots":
        r = state["run"]
        r.reset()
        r.advance(state["steps"])
        u, w = r.seismograms()
        U, W = r.snapshot(0)
        return [a.astype(state["dtype"], copy=False) for a in (u, w, U, W)]
    if kind == "multi":
        runs = [gpu.Run(j["op"], j["md"], j["src"], state["steps"], j["rec"], j["dt"], j["f0"], j["t0"],
                        amplitude=j["amplitude"], precision=state["prec"], nsteps=j["nsteps"], block=256)
                for j in state["jobs"]]
        multi = gpu.Multi(runs)
        multi.advance(state["steps"])
        out = [[a.astype(state["dtype"], copy=False) for a in r.seismograms()] for r in runs]
        multi.close()
        for r in runs:
            r.close()
        return out
    if kind == "dt":
        return list(gpu.estimate_dt(state["op"], state["md"]))
    if kind == "predict":
        return state["net"].predict(state["X"])[0]
    # a learning-rate schedule over the length of a real training run
    loss, _ = state["net"].train(state["epochs"], lr=1e-3, total_steps=200000, seed=state["seed"])
    return [loss, state["net"].weights()]


def _step_work(M, shots, w, kahan, per_shot_media):
    """Bytes and operations of one time step of `shots` active shots: pattern, the
    seven matrices, coefficients, and the 26 state fields (and Kahan terms) of every
    node and shot read once and written once; 32 products over the pattern."""
    n, nnz = M["n"], len(M["col"])
    coef = 12.0 * n * w * shots if per_shot_media else 11.0 * n * w
    return (4.0 * (n + 1) + nnz * (4.0 + 7.0 * w) + coef + shots * n * (52.0 * w + kahan),
            shots * (64.0 * nnz + 150.0 * n))


def _loop_work(case, M, nsteps, per_shot_media=False):
    w = 8.0 if case["prec"] == "fp64" else 4.0
    kahan = {"kahan": 48.0, "kahan16": 24.0}.get(case["prec"], 0.0)
    b = f = 0.0
    for t in range(case["steps"]):
        act = int((nsteps > t).sum())
        if act:
            sb, sf = _step_work(M, act, w, kahan, per_shot_media)
            b, f = b + sb, f + sf
    return b, f


def work(case):
    kind = case["kind"]
    if kind in ("shots", "media"):
        job = _job(case, 1)
        b, f = _loop_work(case, job["M"], job["nsteps"], kind == "media")
    elif kind == "multi":
        b = f = 0.0
        for j in _multi_jobs(case, 1):
            jb, jf = _loop_work(case, j["M"], j["nsteps"])
            b, f = b + jb, f + jf
    elif kind == "dt":
        # about 200 power iterations of four matrices on two components
        M = _mesh(case["mesh"], case["nx"], case["ny"])
        nnz, n = len(M["col"]), M["n"]
        b, f = 200.0 * (nnz * 36.0 + n * (4.0 + 5 * 8.0 + 32.0)), 200.0 * 16.0 * nnz
    else:
        widths = [NIN] + [case["hidden"]] * 3 + [case["nout"]]
        params = sum(i * o for i, o in zip(widths[:-1], widths[1:]))
        n = case["n"]
        if kind == "predict":
            b, f = 2.0 * params + 4.0 * n * (NIN + case["nout"]), 2.0 * params * n
        else:
            # per step: weights and both moments read and written, their bf16 copy read and written, the batch
            steps = (n // case["batch"]) * case["epochs"]
            b, f = steps * (28.0 * params + 4.0 * case["batch"] * case["nout"]), steps * 6.0 * params * case["batch"]
    return dict(bytes=b, flops=f)


# ---- the same results in 64 bits, in plain torch -----------------------------------

def _table(M, mats, dev):
    """Padded row form of the matrices: columns [k][n] and values [7][k][n]."""
    deg = np.diff(M["ptr"])
    k = np.arange(len(M["col"])) - M["ptr"][M["row"]]
    col = np.tile(np.arange(M["n"]), (int(deg.max()), 1))
    col[k, M["row"]] = M["col"]
    val = np.zeros((7, int(deg.max()), M["n"]))
    for m in range(7):
        val[m][k, M["row"]] = mats[m]
    return torch.from_numpy(col).to(dev), torch.from_numpy(val).to(dev)


def _step_loop(M, job, shots, dev):
    """Split-field M-PML loop of the given shots: seismograms [shots][T][rec] and the final U, W."""
    first = job["models"][0]
    own = len(job["models"]) > 1
    pick = lambda get: torch.from_numpy(np.stack([get(job["models"][s if own else 0]) for s in shots], 1)).to(dev)  # noqa: E731
    mats = [M["mats"][0] if own else M["mats"][0] * first["rho"][M["row"]]] + M["mats"][1:]
    col, val = _table(M, mats, dev)
    scale = pick(lambda m: m["rho"]) if own else 1.0
    c11, c13, c33, c44 = (pick(lambda m, k=k: m["c"][k]) for k in range(4))
    dx, dy, dxx, dyy, dxxp, dyyp = (pick(lambda m, k=k: m["mpml"][k]) for k in range(6))
    mass = pick(lambda m: m["mass"])
    keep = torch.from_numpy(1.0 - job["flags"])[:, None].to(dev) / mass
    n, S, T, dt = M["n"], len(shots), job["T"], job["dt"]
    X = torch.zeros(20, n, S, dtype=torch.float64, device=dev)   # u1..u3 w1..w3, their velocities, Lx1..4 Ly1..4
    acc = torch.zeros(6, n, S, dtype=torch.float64, device=dev)
    force = torch.zeros(2, n, S, dtype=torch.float64, device=dev)
    for i, s in enumerate(shots):
        nodes, wt = job["sources"][s] if job["sources"] else ([job["src"][s]], [[1.0, 0.0]])
        for node, (fu, fw) in zip(nodes, wt):
            force[0, int(node), i] += fu
            force[1, int(node), i] += fw
    if not job["sources"]:   # the force direction: sin and cos of 90 degrees with the loop's 14-digit pi
        a = 90.0 * 3.1415926535898 / 180.0
        force[1] = force[0] * math.cos(a)
        force[0] = force[0] * math.sin(a)
    rec = torch.from_numpy(job["rec"].astype(np.int64)).to(dev)
    lim = torch.from_numpy(job["nsteps"][shots].astype(np.int64)).to(dev)
    seis = torch.zeros(2, S, T, len(rec), dtype=torch.float64, device=dev)
    for t in range(T):
        D = torch.stack([X[0:3].sum(0), X[3:6].sum(0)])
        m, p = torch.zeros_like(X), torch.zeros(6, 2, n, S, dtype=torch.float64, device=dev)
        for k in range(col.shape[0]):
            m.addcmul_(X[:, col[k]], val[0, k][None, :, None])
            d = D[:, col[k]]
            for q in range(6):
                p[q].addcmul_(d, val[q + 1, k][None, :, None])
        m *= scale
        u, v, L = m[0:6], m[6:12], m[12:20]
        (s1u, s1w), (s2u, s2w), (s3u, s3w), (s4u, s4w), (s5u, s5w), (s6u, s6w) = p
        arg = (math.pi * job["f0"] * ((t + 3) * dt - job["t0"])) ** 2
        ps = job["amplitude"] * (1 - 2 * arg) * math.exp(-arg)
        rhs = torch.stack([
            -c11 * s1u - 2 * dx * v[0] - dx * dx * u[0] + L[0] + L[1] + ps * force[0],
            -c13 * s3w - c44 * s4w - (dx + dy) * v[1] - dx * dy * u[1],
            -c44 * s2u - 2 * dy * v[2] - dy * dy * u[2] + L[2] + L[3],
            -c44 * s1w - 2 * dx * v[3] - dx * dx * u[3] + L[4] + L[5] + ps * force[1],
            -c44 * s3u - c13 * s4u - (dx + dy) * v[4] - dx * dy * u[4],
            -c33 * s2w - 2 * dy * v[5] - dy * dy * u[5] + L[6] + L[7]]) * keep
        mem = torch.stack([
            L[0] - dt * (c11 * dxx * s5u + dx * L[0]), L[1] - dt * (c44 * dyyp * s5w + dy * L[1]),
            L[2] - dt * (c13 * dxxp * s6w + dx * L[2]), L[3] - dt * (c44 * dyy * s6u + dy * L[3]),
            L[4] - dt * (c44 * dxx * s5w + dx * L[4]), L[5] - dt * (c13 * dyyp * s5u + dy * L[5]),
            L[6] - dt * (c44 * dxxp * s6u + dx * L[6]), L[7] - dt * (c33 * dyy * s6w + dy * L[7])]) * keep
        new = torch.cat([X[0:6] + dt * X[6:12] + (rhs - 0.5 * acc) * dt * dt,
                         X[6:12] + (1.5 * rhs - 0.5 * acc) * dt, mem])
        on = t < lim
        X = torch.where(on, new, X)
        acc = torch.where(on, rhs, acc)
        seis[0, :, t] = (X[0:3].sum(0)[rec] * on).T
        seis[1, :, t] = (X[3:6].sum(0)[rec] * on).T
    return seis.cpu().numpy(), X[0:3].sum(0).cpu().numpy(), X[3:6].sum(0).cpu().numpy()


def _exact_shots(job, dev):
    M, S = job["M"], job["S"]
    u, w, at = [], [], None
    chunk = max(1, int(3.0e6 // M["n"]))
    for s0 in range(0, S, chunk):
        seis, U, W = _step_loop(M, job, list(range(s0, min(S, s0 + chunk))), dev)
        u.append(seis[0])
        w.append(seis[1])
        at = (U[:, 0].copy(), W[:, 0].copy()) if s0 == 0 else at
    return [np.concatenate(u), np.concatenate(w), at[0], at[1]]


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    kind = case["kind"]
    if kind in ("shots", "media"):
        return _exact_shots(_job(case, seed), dev)
    if kind == "multi":
        return [_exact_shots(j, dev)[:2] for j in _multi_jobs(case, seed)]
    if kind == "predict":
        h = torch.from_numpy(_models_in(case, seed)).double().to(dev)
        ws = _weights(case, seed)
        for l, (W, b) in enumerate(ws):
            h = h @ torch.from_numpy(W).double().to(dev).T + torch.from_numpy(b).double().to(dev)
            if l + 1 < len(ws):
                h = torch.nn.functional.gelu(h, approximate="tanh")
        return h.cpu().numpy()
    # a training run's weights follow the rounding of every step, and the dt estimate
    # is a power iteration stopped at a tolerance: neither has a value of its own
    return None
