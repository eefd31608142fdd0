"""The workloads whose speed is tracked: what programs built on this library have it do.

  listed()             the tracked cases, each a dict of plain values
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  what a program holds before the call: meshes, targets, fields, a batch or network handle
  run(state)           one pass through the public entry points, and its outputs
  work(case)           bytes and operations that one pass cannot do without
  exact(case, seed)    the same outputs in 64 bits from dense linear algebra (torch), where that is affordable

Kinds of case:

  dropin    simple_FEM_1D_transient, the reference's evaluator called as its own programs call it: one field, NR arrays
  noalloc   scft_eval_noalloc: one field in the caller's device memory
  one       Batch.eval of a single instance, host arrays in and out
  columns   Batch.eval of many fields on one mesh, as a finite-difference Jacobian asks for them
  irk       Batch.eval with the two-stage Gauss stepper (the deal.II path), many fields on one mesh
  mix       Batch.eval of an uneven batch: uniform meshes, m log-uniform in 32-4096, or meshes graded toward the wall
  cold      Batch.solve of an uneven batch from w0
  warm      Batch.solve of an uneven batch from fields carried over from the coarser meshes (mesh continuation), with the
            cold fields as the fallback
  predict   the warm-start network's prediction written into a batch's resident field, and the field fetched
  train     one epoch of the warm-start network's training
"""
import math

import numpy as np
import torch

import scft_amd as S
from scft_amd import warmstart as WS

TAU = 0.530252230020752
L_REF = 3.72374357332160

# The solver that the benchmark uses from w0, and what it changes from a predicted or transferred start.
SOLVER = dict(history=16, beta=1.0, tol=1e-6, step_cap=0.0, floor=1e-8, backtrack=1e30, max_halvings=30,
              field_floor=0.5, gs_precond=0.5, gs_field_weight=0.25, gs_shift=3.0, gs_shift_below=0.5,
              max_iter=400, check_every=4, transform=S.MIX_LOG)
PRECOND = {"uniform": 0.5, "graded": 0.6}
WARM = dict(history=8, gs_switch=24, fallback_factor=10.0)


def listed():
    return [
        # the reference's own problem, one evaluation as its solvers call it: latency alone
        dict(name="dropin_m32", kind="dropin", m=32, N=2048, L=L_REF, bc=S.BC_DD, cmat=S.C_ROWSCALED),
        # an evaluation inside a program that keeps its fields on the device; odd size, the deal.II w-mass
        dict(name="noalloc_m203", kind="noalloc", m=203, N=1024, L=3.0, bc=S.BC_DD, cmat=S.C_CONSISTENT),
        # the benchmark's single-instance configuration
        dict(name="one_m1024", kind="one", mesh="uniform", m=1024, N=2048, L=3.72, bc=S.BC_DN),
        # the largest single instance of the production mix: finest wall cells, most steps
        dict(name="one_graded_m4095", kind="one", mesh="graded", m=4095, N=8192, L=8.0, bc=S.BC_DN),
        # the n perturbed fields of a Broyden Jacobian on a mid-size mesh
        dict(name="columns_m256", kind="columns", m=256, N=1024, L=3.72, count=256, bc=S.BC_DN),
        # the deal.II fixture's mesh and stepper, a batch of fields
        dict(name="irk_m32x1024", kind="irk", m=32, N=512, L=L_REF, count=1024, bc=S.BC_DD, cmat=S.C_CONSISTENT),
        # the uniform-mesh benchmark batch, a quarter of it
        dict(name="mix_uniform_1024", kind="mix", mesh="uniform", count=1024, mix=20261202),
        # the production mix, a sixteenth of it
        dict(name="mix_graded_1024", kind="mix", mesh="graded", count=1024, mix=20261205),
        # whole solves: from w0 on uniform meshes; from transferred fields on graded ones
        dict(name="cold_uniform_512", kind="cold", mesh="uniform", count=512, mix=31),
        dict(name="warm_graded_384", kind="warm", mesh="graded", count=384, mix=32),
        # the warm start of a batch, and the training that makes it
        dict(name="predict_2048", kind="predict", mesh="uniform", count=2048, mix=33),
        dict(name="train_8192", kind="train", rows=8192, batch=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dropin", "noalloc", "one", "columns", "irk", "mix", "cold", "warm", "predict", "train"])
    bc, cmat = rng.choice([S.BC_DD, S.BC_DN]), rng.choice([S.C_ROWSCALED, S.C_CONSISTENT])
    L = round(rng.uniform(2.0, 8.0), 3)
    mesh = rng.choice(["uniform", "graded"])
    if kind == "dropin":
        return dict(kind=kind, m=_log_int(rng, 16, 1024), N=rng.choice([512, 1024, 2048, 4096]), L=L, bc=bc, cmat=cmat)
    if kind == "noalloc":
        return dict(kind=kind, m=_log_int(rng, 16, 2048), N=rng.choice([256, 512, 1024, 2048, 4096]), L=L, bc=bc,
                    cmat=cmat)
    if kind == "one":
        return dict(kind=kind, mesh=mesh, m=_log_int(rng, 64, 4095), N=rng.choice([512, 1024, 2048, 4096, 8192]), L=L,
                    bc=bc)
    if kind == "columns":
        m = _log_int(rng, 24, 512)
        return dict(kind=kind, m=m, N=rng.choice([256, 512, 1024, 2048]), L=L, count=m, bc=bc)
    if kind == "irk":
        return dict(kind=kind, m=_log_int(rng, 16, 300), N=rng.choice([128, 256, 512, 1024, 2048]), L=L,
                    count=_log_int(rng, 32, 1024), bc=bc, cmat=cmat)
    if kind == "mix":
        return dict(kind=kind, mesh=mesh, count=_log_int(rng, 32, 768), mix=rng.randrange(1 << 20))
    if kind in ("cold", "warm"):
        return dict(kind=kind, mesh=mesh, count=_log_int(rng, 24, 192), mix=rng.randrange(1 << 20))
    if kind == "predict":
        return dict(kind=kind, mesh="uniform", count=_log_int(rng, 64, 2048), mix=rng.randrange(1 << 20))
    return dict(kind=kind, rows=_log_int(rng, 600, 12000), batch=_log_int(rng, 64, 1024))


# ------------------------------------------------------------------ inputs
def _rng(seed, salt):
    return np.random.default_rng([int(seed), salt])


def _uniform(m, L):
    return np.arange(m + 1) * L / m


def _graded(m, L, ell):
    x = ell * np.expm1(np.log1p(L / ell) / m * np.arange(m + 1))
    x[0], x[-1] = 0.0, L
    return x


def _target(x, bc):
    """The EXP wall profile tanh^2(2 tau x / (tau^2 - x^2)) from each wall."""
    d = np.minimum(x, x[-1] - x) if bc == S.BC_DD else x
    out = np.ones_like(x)
    near = d < TAU
    out[near] = np.tanh(2.0 * TAU * d[near] / (TAU * TAU - d[near] ** 2)) ** 2
    return out


def _field(x, rng):
    """A field on all nodes: the smooth start of the benchmark, its noise, and a long wave of the seed's own."""
    w = 0.1 * np.exp(-x / 0.2) + rng.normal(0.0, 1e-3, len(x))
    w += rng.uniform(0.05, 0.2) * np.cos(rng.uniform(1.0, 3.0) * x + rng.uniform(0.0, 6.0))
    return w


def _w0(x, rng):
    """The benchmark's cold start."""
    w = 0.1 * np.exp(-x / 0.2) + rng.normal(0.0, 1e-3, len(x))
    w[0] = 0.0
    return w


def _unk(a, bc):
    return a[1:-1] if bc == S.BC_DD else a[1:]


def _mix(case):
    """Meshes and step counts of an uneven batch: the case's own, whatever the seed."""
    r, n = _rng(case["mix"], 5), case["count"]
    Ls = r.uniform(2.0, 8.0, n)
    if case["mesh"] == "uniform":
        ms = np.rint(np.exp(r.uniform(np.log(32), np.log(4096), n))).astype(int)
        return [_uniform(int(m), float(L)) for m, L in zip(ms, Ls)], r.choice([512, 1024, 2048, 4096], n).tolist()
    h0, ell = np.exp(r.uniform(np.log(1e-4), np.log(1e-2), n)), r.uniform(0.05, 0.5, n)
    ms = np.clip(np.rint(ell * np.log1p(Ls / ell) / h0), 63, 4095).astype(int)
    return ([_graded(int(m), float(L), float(e)) for m, L, e in zip(ms, Ls, ell)],
            r.choice([512, 1024, 2048, 4096, 8192], n).tolist())


def _mesh_of(case):
    if case.get("mesh") == "graded":
        return _graded(case["m"], case["L"], 0.05 + 0.1 * (case["m"] % 4))
    return _uniform(case["m"], case["L"])


def _fields_of(case, seed):
    """(x, count fields on all nodes, wall values or None) of a case on one mesh."""
    x, bc = _mesh_of(case), case["bc"]
    rng = _rng(seed, 7)
    ws = np.stack([_field(x, rng) for _ in range(case.get("count", 1))])
    if case["kind"] == "columns":  # one field, and its unknowns perturbed one by one
        ws[:] = ws[0]
        cols = np.arange(case["count"]) % (len(x) - 2) + 1
        ws[np.arange(case["count"]), cols] += 1e-4 * np.maximum(np.abs(ws[0][cols]), 1e-2)
    if case["kind"] != "irk":
        ws[:, 0] = 0.0
        if bc == S.BC_DD:
            ws[:, -1] = 0.0
    return x, ws


def _net_params(dims, rng):
    out = []
    for a, b in zip(dims[:-1], dims[1:]):
        lim = math.sqrt(6.0 / (a + b))
        out += [rng.uniform(-lim, lim, a * b), rng.normal(0.0, 0.05, b)]
    return np.concatenate(out).astype(np.float32)


CUTS = (512,)  # one network per range of mesh sizes, as the benchmark splits them


def _predict_inputs(case, seed):
    xs, Ns = _mix(case)
    rng = _rng(seed, 9)
    w0 = [_w0(x, rng) for x in xs]
    nets = [_net_params(WS.DIMS, rng) for _ in range(len(CUTS) + 1)]
    ng, nn = WS.GRID, len(WS.NODE_IDX)
    scale = (np.array([5.0, 7.3, 6.0, -5.5, -5.5], np.float32), np.array([1.7, 0.8, 1.4, 1.5, 1.5], np.float32))
    x_mean = np.concatenate([scale[0], np.zeros(ng, np.float32)])
    x_std = np.concatenate([scale[1], np.ones(ng, np.float32)])
    y_mean = np.concatenate([0.05 * np.cos(np.linspace(0, 9, ng)), np.linspace(2.0, 0.1, nn)]).astype(np.float32)
    y_std = np.concatenate([np.linspace(0.3, 0.05, ng), np.full(nn, 0.4)]).astype(np.float32)
    return xs, Ns, w0, nets, (x_mean, x_std, y_mean, y_std)


def _train_inputs(case, seed):
    rng, n = _rng(seed, 11), case["rows"]
    Ls = rng.uniform(2.0, 8.0, n)
    F = np.empty((n, WS.DIMS[0]))
    F[:, 0] = Ls
    F[:, 1] = np.log(rng.choice([512.0, 1024.0, 2048.0, 4096.0], n))
    F[:, 2] = rng.uniform(np.log(32), np.log(4096), n)
    F[:, 3] = F[:, 4] = np.log(Ls) - F[:, 2]
    t = np.linspace(0.0, 1.0, WS.GRID)
    F[:, 5:] = 0.1 * np.exp(-(t * Ls[:, None]) / 0.2) + rng.normal(0.0, 1e-3, (n, WS.GRID))
    amp, ph = rng.uniform(0.5, 1.5, (n, 1)), Ls[:, None] / 3.0
    Y = np.empty((n, WS.DIMS[-1]))
    Y[:, :WS.GRID] = amp * np.cos(3.0 * t + ph) * np.exp(-2.0 * t) - 0.1 * F[:, 1:2]
    Y[:, WS.GRID:] = 3.0 - 0.4 * F[:, 3:4] * np.linspace(1.0, 0.2, len(WS.NODE_IDX))
    return F.astype(np.float32), Y.astype(np.float32), _net_params(WS.DIMS, rng), 1 + int(seed) % 1000


def _norm_of(F, Y):
    xm, xs, ym, ys = F.mean(axis=0), F.std(axis=0), Y.mean(axis=0), Y.std(axis=0)
    xs[WS.N_SCALARS:] = 1.0
    xs[xs < 1e-6] = 1.0
    ys[ys < 1e-6] = 1.0
    return [v.astype(np.float32) for v in (xm, xs, ym, ys)]


# ----------------------------------------------------------------- prepare
def _options(case, **more):
    return S.anderson_opts(**{**SOLVER, "precond": PRECOND[case["mesh"]], **more})


def _continued(case, xs, Ns, w0, rng):
    """Fields on the meshes `xs` from the batch solved on every other node (mesh continuation)."""
    xc = [np.concatenate([x[:-1:2], x[-1:]]) if (len(x) - 1) % 2 else x[::2] for x in xs]
    wc = [_w0(x, rng) for x in xc]
    b = S.Batch(xc, Ns, [_target(x, S.BC_DN)[1:] for x in xc], bc=S.BC_DN)
    out = b.solve([w[1:] for w in wc], _options(case))
    b.close()
    ys = [np.concatenate([[0.0], w]) for w in out["w"]]
    return S.resample_spline_batch(xc, ys, [x[1:] for x in xs], flat=True)[0]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dropin":
        S.init(N=case["N"], L=case["L"], bc=case["bc"], cmat=case["cmat"])
        x, ws = _fields_of(case, seed)
        w = np.concatenate([[0.0], _unk(ws[0], case["bc"])])
        return dict(kind=kind, w=w, out=np.zeros_like(w))
    if kind == "noalloc":
        x, ws = _fields_of(case, seed)
        dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
        w = dev(_unk(ws[0], case["bc"]))
        return dict(kind=kind, M=len(x), N=case["N"], bc=case["bc"], cmat=case["cmat"], x=dev(x), w=w,
                    pt=dev(_unk(_target(x, case["bc"]), case["bc"])), phi=torch.empty_like(w), r=torch.empty_like(w),
                    rnorm=torch.empty(1, dtype=torch.float64, device="cuda"),
                    status=torch.empty(1, dtype=torch.int32, device="cuda"))
    if kind in ("one", "columns", "irk"):
        x, ws = _fields_of(case, seed)
        bc, n = case["bc"], len(ws)
        b = S.Batch([x] * n, [case["N"]] * n, [_unk(_target(x, bc), bc)] * n, bc=bc,
                    cmat=case.get("cmat", S.C_ROWSCALED), stepper=S.STEP_IRK4 if kind == "irk" else S.STEP_IE)
        if kind == "irk":
            b.set_walls(ws[:, 0], ws[:, -1])
        return dict(kind="eval", b=b, w=b.join([_unk(w, bc) for w in ws]))
    if kind == "train":
        F, Y, p, shuffle = _train_inputs(case, seed)
        net = S.Mlp(WS.DIMS)
        net.set_normalisation(*_norm_of(F, Y))
        return dict(kind=kind, net=net, X=F, Y=Y, p=p, shuffle=shuffle, batch=case["batch"])
    if kind == "predict":
        xs, Ns, w0, params, norm = _predict_inputs(case, seed)
        ws = WS.WarmStart(S, cuts=CUTS)
        for net, p in zip(ws.nets, params):
            net.set_params(p)
            net.set_normalisation(*norm)
        b = S.Batch(xs, Ns, [_target(x, S.BC_DN)[1:] for x in xs], bc=S.BC_DN)
        b.upload([w[1:] for w in w0])
        plan = ws.device_plan(b, WS.Prepared(S, dict(xs=xs, Ns=Ns, w0=w0)))
        return _Predict(b, ws, plan)
    xs, Ns = _mix(case)
    rng = _rng(seed, 7)
    b = S.Batch(xs, Ns, [_target(x, S.BC_DN)[1:] for x in xs], bc=S.BC_DN)
    if kind == "mix":
        ws = [_field(x, rng) for x in xs]
        return dict(kind="eval", b=b, w=b.join([w[1:] for w in ws]))
    w0 = b.join([_w0(x, rng)[1:] for x in xs])
    if kind == "cold":
        return dict(kind="solve", b=b, w=w0, cold=None, opts=_options(case))
    return dict(kind="solve", b=b, w=_continued(case, xs, Ns, w0, rng), cold=w0, opts=_options(case, **WARM))


class _Predict(dict):
    """The handles of a prediction, closed in the order that they need: the plan, the networks, the batch."""

    def __init__(self, b, ws, plan):
        super().__init__(kind="predict", b=b, ws=ws, plan=plan)

    def __del__(self):
        self["plan"].close()
        self["ws"].close()
        self["b"].close()


# --------------------------------------------------------------------- run
def _flat(parts):
    """The one array that a batch's per-instance views are cut from."""
    return parts[0].base


def run(state):
    kind = state["kind"]
    if kind == "dropin":
        rc = S.simple_FEM_1D_transient(state["w"], state["out"])
        return dict(rc=rc, r=state["out"][1:])
    if kind == "noalloc":
        s = state
        rc = S.eval_noalloc(s["M"], s["N"], s["x"].data_ptr(), s["w"].data_ptr(), s["pt"].data_ptr(),
                            s["phi"].data_ptr(), s["r"].data_ptr(), s["rnorm"].data_ptr(), s["status"].data_ptr(),
                            bc=s["bc"], cmat=s["cmat"])
        return dict(rc=rc, phi=s["phi"], r=s["r"], rnorm=s["rnorm"], status=s["status"])
    if kind == "eval":
        out = state["b"].eval(state["w"])
        return dict(phi=_flat(out["phi"]), r=_flat(out["r"]), rnorm=out["rnorm"], status=out["status"].astype(np.int64))
    if kind == "solve":
        out = state["b"].solve(state["w"], state["opts"], w_cold_parts=state["cold"])
        return dict(w=_flat(out["w"]), iters=out["iters"], status=out["status"].astype(np.int64))
    if kind == "predict":
        state["plan"].predict()
        return dict(w=_flat(state["b"].download()["w"]))
    net = state["net"]
    net.set_params(state["p"])
    net.train(state["X"], state["Y"], epochs=1, batch=state["batch"], lr=1e-3, seed=state["shuffle"])
    return dict(params=net.params())


# -------------------------------------------------------------------- work
IE_FLOPS, IRK_FLOPS = 11, 25  # per unknown and step: right-hand side, tridiagonal solve, half a pairing


def work(case):
    kind = case["kind"]
    if kind == "train":
        p = sum(a * b + b for a, b in zip(WS.DIMS[:-1], WS.DIMS[1:]))
        steps = -(-case["rows"] // case["batch"])
        return dict(bytes=4 * (case["rows"] * (WS.DIMS[0] + WS.DIMS[-1]) + 2 * p),
                    flops=6 * case["rows"] * p + 12 * p * steps)
    if kind == "predict":
        xs, _ = _mix(case)
        p = sum(a * b + b for a, b in zip(WS.DIMS[:-1], WS.DIMS[1:]))
        n = sum(len(x) - 1 for x in xs)
        return dict(bytes=16 * n + case["count"] * (4 * WS.DIMS[0] + 8 * WS.GRID) + 8 * p,
                    flops=2 * p * case["count"] + 20 * n)
    if kind in ("mix", "cold", "warm"):
        xs, Ns = _mix(case)
        n, steps = sum(len(x) - 1 for x in xs), sum((len(x) - 1) * N for x, N in zip(xs, Ns))
        evals = {"mix": 1, "cold": 7, "warm": 3}[kind]  # the evaluations that an instance needs, about
        return dict(bytes=40 * n, flops=evals * IE_FLOPS * steps)
    n, c = case["m"] - (1 if case["bc"] == S.BC_DD else 0), case.get("count", 1)
    return dict(bytes=40 * n * c, flops=(IRK_FLOPS if kind == "irk" else IE_FLOPS) * n * c * case["N"])


# ------------------------------------------------------------------- exact
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _steps_matrix(x, w, N, bc, cmat, irk):
    """Dense T with q^{j+1} = T q^j on the unknowns, one per row of w (fields on all nodes), in 64 bits."""
    x, w = torch.tensor(x, dtype=torch.float64), torch.tensor(w, dtype=torch.float64)
    h, M, c = x[1:] - x[:-1], len(x), len(w)
    i = torch.arange(M - 1)
    A, B = torch.zeros(M, M, dtype=torch.float64), torch.zeros(M, M, dtype=torch.float64)
    for T, d, o in ((A, h / 3, h / 6), (B, 1 / h, -1 / h)):
        T[i, i] += d
        T[i + 1, i + 1] += d
        T[i, i + 1] = o
        T[i + 1, i] = o
    if cmat == S.C_ROWSCALED:
        Cm = w[:, :, None] * A
    else:  # the w-mass of the piecewise linear field
        Cm = torch.zeros(c, M, M, dtype=torch.float64)
        wl, wr = w[:, :-1], w[:, 1:]
        Cm[:, i, i] += h * (3 * wl + wr) / 12
        Cm[:, i + 1, i + 1] += h * (wl + 3 * wr) / 12
        Cm[:, i, i + 1] = h * (wl + wr) / 12
        Cm[:, i + 1, i] = h * (wl + wr) / 12
    u = slice(1, M - 1) if bc == S.BC_DD else slice(1, M)
    A, D = A[u, u].contiguous(), (B + Cm)[:, u, u].contiguous()
    dt = 1.0 / N
    if not irk:
        return torch.linalg.solve(A + dt * D, A.expand_as(D).contiguous()).to(_dev())
    n, r3 = A.shape[0], math.sqrt(3.0) / 6
    a = [[0.25, 0.25 - r3], [0.25 + r3, 0.25]]
    G = torch.cat([torch.cat([(A if p == q else 0 * A) + dt * a[p][q] * D for q in (0, 1)], 2) for p in (0, 1)], 1)
    K = torch.linalg.solve(G, torch.cat([-D, -D], 1))
    return (torch.eye(n, dtype=torch.float64) + 0.5 * dt * (K[:, :n] + K[:, n:])).to(_dev())


def _density(T, N):
    """phi(x) = int q(x, s) q(x, 1 - s) ds on the unknowns by the five-level Romberg rule."""
    c, n = T.shape[0], T.shape[1]
    q = torch.empty(N + 1, c, n, dtype=torch.float64, device=T.device)
    q[0] = 1.0
    for j in range(N):
        q[j + 1] = (T[0] @ q[j, 0])[None] if c == 1 else torch.bmm(T, q[j].unsqueeze(2)).squeeze(2)
    s = [2 ** k for k in range(5)]  # strides of the five finest trapezoid rules, extrapolated in h^2
    phi = 0.0
    for k in s:
        lam = math.prod(j * j / (j * j - k * k) for j in s if j != k)
        g = q[::k] * q.flip(0)[::k]
        phi = phi + lam * (k / N) * (g.sum(0) - 0.5 * (g[0] + g[-1]))
    return phi


def _natural_walls(x, w, bc):
    """The field at the walls by the natural spline through the unknowns (the drop-in evaluator's convention)."""
    xs, ys = (x[1:-1], w[1:-1]) if bc == S.BC_DD else (x[1:], w[1:])
    h, n = np.diff(xs), len(xs)
    Mt, rhs = np.eye(n), np.zeros(n)
    for i in range(1, n - 1):
        Mt[i, i - 1:i + 2] = h[i - 1] / 6, (h[i - 1] + h[i]) / 3, h[i] / 6
        rhs[i] = (ys[i + 1] - ys[i]) / h[i] - (ys[i] - ys[i - 1]) / h[i - 1]
    M = np.linalg.solve(Mt, rhs)

    def at(p, k):
        a, b = (xs[k + 1] - p) / h[k], (p - xs[k]) / h[k]
        return a * ys[k] + b * ys[k + 1] + ((a ** 3 - a) * M[k] + (b ** 3 - b) * M[k + 1]) * h[k] ** 2 / 6

    w = w.copy()
    w[0] = at(x[0], 0)
    if bc == S.BC_DD:
        w[-1] = at(x[-1], n - 2)
    return w


def _exact_eval(case, seed):
    x, ws = _fields_of(case, seed)
    bc, cmat = case["bc"], case.get("cmat", S.C_ROWSCALED)
    if case["kind"] == "dropin" and cmat == S.C_CONSISTENT and len(x) > 4:
        ws = np.stack([_natural_walls(x, w, bc) for w in ws])
    phi = _density(_steps_matrix(x, ws, case["N"], bc, cmat, case["kind"] == "irk"), case["N"]).cpu().numpy()
    r = phi - _unk(_target(x, bc), bc)[None]
    return phi.reshape(-1), r.reshape(-1), np.abs(r).max(axis=1)


def _layers(p):
    out, o = [], 0
    for a, b in zip(WS.DIMS[:-1], WS.DIMS[1:]):
        out.append([p[o:o + a * b].reshape(b, a), p[o + a * b:o + a * b + b]])
        o += a * b + b
    return out


def _net(p, X):
    a = X
    layers = _layers(p)
    for k, (W, b) in enumerate(layers):
        a = a @ W.T + b
        if k < len(layers) - 1:
            a = torch.tanh(a)
    return a


def _f64(a):
    return torch.tensor(np.asarray(a), dtype=torch.float64, device=_dev())


def _shuffled(n, seed):
    """The trainer's order of rows in its first epoch: Fisher-Yates from splitmix64(seed)."""
    idx, s, mask = list(range(n)), seed, (1 << 64) - 1
    for i in range(n - 1, 0, -1):
        s = (s + 0x9E3779B97F4A7C15) & mask
        z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        j = (z ^ (z >> 31)) % (i + 1)
        idx[i], idx[j] = idx[j], idx[i]
    return idx


def _exact_train(case, seed):
    F, Y, p, shuffle = _train_inputs(case, seed)
    xm, xs, ym, ys = (_f64(v) for v in _norm_of(F, Y))
    X, T, p = (_f64(F) - xm) / xs, (_f64(Y) - ym) / ys, _f64(p)
    m, v, b1, b2 = torch.zeros_like(p), torch.zeros_like(p), 0.9, 0.999
    order = torch.tensor(_shuffled(len(F), shuffle), device=p.device)
    for t, at in enumerate(range(0, len(F), case["batch"])):
        rows = order[at:at + case["batch"]]
        q = p.clone().requires_grad_()
        (_net(q, X[rows]) - T[rows]).square().mean().backward()
        m, v = b1 * m + (1 - b1) * q.grad, b2 * v + (1 - b2) * q.grad.square()
        p = p - 1e-3 * (m / (1 - b1 ** (t + 1))) / ((v / (1 - b2 ** (t + 1))).sqrt() + 1e-8)
    return dict(params=p.cpu().numpy())


def exact(case, seed):
    kind = case["kind"]
    if kind == "dropin":
        return dict(rc=None, r=_exact_eval(case, seed)[1])
    if kind in ("noalloc", "one", "columns", "irk"):
        phi, r, rnorm = _exact_eval(case, seed)
        return dict(rc=None, phi=phi, r=r, rnorm=rnorm, status=None)
    if kind == "train":
        return _exact_train(case, seed)
    return None  # thousands of uneven marches, or solves to a tolerance
