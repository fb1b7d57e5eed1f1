"""Performance cases of the transient-elasticity path: what a program that uses this package has it do, through
`topopt_in_petsc_transient_amd.capi`, from single operator applications to whole design iterations.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw(rng)` more of the same ranges, `prepare`
makes what a program holds before the call (a context, a density, an MMA object), `run` is one pass, `work` the
bytes and operations a pass cannot do without, and `exact` the outputs in plain numpy / torch FP64 where that is
feasible (operator applications, small gradients, the PDE filter).

Kinds:
  op        one operator application y = N X N u + (1 - N) u on device arrays (X = K, M or the Newmark operator A)
  forward   one design's forward sweep: density, multigrid set-up, initial state, Newmark steps, the last state
  gradient  one design iteration's physics: the forward sweep, then objective and sensitivities by the adjoint
  reduced   the same with the reduced-order (SOMMG) model
  filter    the PDE filter of a density field, with the Heaviside projection, on host arrays
  update    the design update after the physics, on host arrays: filtered gradients, move limits, MMA, the new
            filtered design
The linear solves of whole calls run at rtol 1e-12, as the parity tests do, so that accelerations and gradients (which
amplify a solve's error by the time integrator's 4/dt^2) do not depend on where within a looser tolerance an
iteration stops; the reduced-order model's quasi-static solves, which cannot reach that, at 1e-10, the reference's
own default.
"""
import numpy as np
import torch

from topopt_in_petsc_transient_amd import capi

NU, EMIN, EMAX, RMIN, RMAX = 0.3, 1e-9, 1.0, 1e-3, 1.0
ALPHA, BETA = 1e-2, 1e-4
VOLFRAC = 0.12


def listed():
    return [
        # the smallest call: one Newmark-operator application on the unit-test mesh (launch and host latency)
        {"name": "op_a_fp64_16x8x8", "kind": "op", "ex": 16, "ey": 8, "ez": 8, "which": 2, "prec": 0},
        # an odd, ragged grid: stiffness application
        {"name": "op_k_fp64_97x51x43", "kind": "op", "ex": 97, "ey": 51, "ez": 43, "which": 0, "prec": 0},
        # the operator benchmark's mesh, both precisions
        {"name": "op_a_fp64_128x64x64", "kind": "op", "ex": 128, "ey": 64, "ez": 64, "which": 2, "prec": 0},
        {"name": "op_a_fp32_128x64x64", "kind": "op", "ex": 128, "ey": 64, "ez": 64, "which": 2, "prec": 1},
        # a gradient check on the unit-test mesh: latency-bound sweeps, every state stored
        {"name": "gradient_fp64_16x8x8", "kind": "gradient", "ex": 16, "ey": 8, "ez": 8, "steps": 30, "slots": 0,
         "nlvls": 2, "prec": 0, "objective": 3, "boundaries": 1},
        # the sensitivity-study mesh: MBB supports, dissipation objective, binomial checkpoints
        {"name": "gradient_mixed_32x16x16", "kind": "gradient", "ex": 32, "ey": 16, "ez": 16, "steps": 50, "slots": 8,
         "nlvls": 3, "prec": 1, "objective": 6, "boundaries": 0},
        # the headline benchmark's forward sweep, both precision modes
        {"name": "forward_mixed_128x64x64", "kind": "forward", "ex": 128, "ey": 64, "ez": 64, "steps": 20,
         "nlvls": 4, "prec": 1},
        {"name": "forward_fp64_128x64x64", "kind": "forward", "ex": 128, "ey": 64, "ez": 64, "steps": 20,
         "nlvls": 4, "prec": 0},
        # the headline benchmark's gradient: 20 checkpoint slots, recomputation, adjoint, sensitivities
        {"name": "gradient_mixed_128x64x64", "kind": "gradient", "ex": 128, "ey": 64, "ez": 64, "steps": 100,
         "slots": 20, "nlvls": 4, "prec": 1, "objective": 3, "boundaries": 1},
        # the reduced-order model's gradient on the benchmark mesh
        {"name": "reduced_fp64_128x64x64", "kind": "reduced", "ex": 128, "ey": 64, "ez": 64, "steps": 100,
         "nlvls": 4, "prec": 0, "basis": 5},
        # the design update between two physics solves
        {"name": "update_128x64x64", "kind": "update", "ex": 128, "ey": 64, "ez": 64, "rmin": 0.08},
        # the mesh of the reference's largest job scripts (192 x 96 x 96 elements)
        {"name": "forward_mixed_192x96x96", "kind": "forward", "ex": 192, "ey": 96, "ez": 96, "steps": 10,
         "nlvls": 5, "prec": 1},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _mg_grid(rng, most):
    """A grid with 2:1:1 to 1:1:1 proportions whose extents divide by 2^(nlvls - 1), at most `most` elements,
    and enough levels for a direct coarsest solve."""
    while True:
        nlvls = rng.choice([2, 3, 3, 4, 4, 5])
        f = 1 << (nlvls - 1)
        ey, ez = f * _log_int(rng, 2, 12), f * _log_int(rng, 2, 12)
        ex = f * _log_int(rng, 2, 24)
        coarse = 3 * (ex // f + 1) * (ey // f + 1) * (ez // f + 1)
        if ex * ey * ez <= most and coarse <= 6476 and max(ex, ey, ez) <= 4 * min(ex, ey, ez):
            return ex, ey, ez, nlvls


def draw(rng):
    kind = rng.choice(["op", "op", "forward", "forward", "gradient", "gradient", "reduced", "filter", "update"])
    if kind == "op":
        return {"kind": kind, "ex": _log_int(rng, 9, 192), "ey": _log_int(rng, 7, 96), "ez": _log_int(rng, 5, 96),
                "which": rng.randrange(3), "prec": rng.randrange(2)}
    if kind in ("filter", "update"):
        c = {"kind": kind, "ex": _log_int(rng, 12, 128), "ey": _log_int(rng, 9, 64), "ez": _log_int(rng, 9, 64),
             "rmin": round(rng.uniform(0.03, 0.12), 4)}
        if kind == "filter":
            c["projection"] = rng.randrange(2)
        return c
    ex, ey, ez, nlvls = _mg_grid(rng, 128 * 64 * 64 if kind != "forward" else 160 * 80 * 80)
    c = {"kind": kind, "ex": ex, "ey": ey, "ez": ez, "nlvls": nlvls, "prec": rng.randrange(2)}
    if kind == "forward":
        c["steps"] = rng.randint(4, 30)
    elif kind == "gradient":
        c["steps"] = rng.randint(10, 60)
        c["slots"] = rng.choice([0, 4, 9])
        c["objective"] = rng.randrange(7)
        c["boundaries"] = rng.randrange(2)
    else:
        c["steps"] = rng.randint(20, 100)
        c["basis"] = rng.randint(2, 7)
    return c


# ---------------------------------------------------------------- inputs
def _smooth(f, passes):
    """3-point smoothing along every axis, edges repeated."""
    for _ in range(passes):
        for ax in range(3):
            p = np.concatenate([f.take([0], ax), f, f.take([-1], ax)], ax)
            n = f.shape[ax]
            f = 0.25 * p.take(range(0, n), ax) + 0.5 * f + 0.25 * p.take(range(2, n + 2), ax)
    return f


def _density(case, seed):
    """A design of mean about VOLFRAC with structure a few elements wide, in [0.001, 1]."""
    rng = np.random.default_rng([seed, 1])
    f = _smooth(rng.uniform(0.0, 1.0, (case["ez"], case["ey"], case["ex"])), 3)
    f = (f - f.mean()) / f.std()
    return np.clip(VOLFRAC * (1.0 + 0.5 * f), 0.001, 1.0).ravel()


def _dt(case):
    return 0.005


def _box(case):
    h = 2.0 / 128  # elements of the benchmark's size, whatever the grid
    if case["kind"] in ("gradient",) and case["ex"] <= 16:
        h = 2.0 / 16
    return (0.0, h * case["ex"], 0.0, h * case["ey"], 0.0, h * case["ez"])


def _params(case):
    kind = case["kind"]
    steps = case.get("steps", 1)
    p = capi.default_params(
        nelx=case["ex"], nely=case["ey"], nelz=case["ez"], xc=_box(case), nsteps=steps, t1=_dt(case) * steps,
        pulse_steps=20, precision=case.get("prec", 0), rtol=1e-10 if kind == "reduced" else 1e-12, maxit=500,
        nlvls=case.get("nlvls", 1), cheb_degree=2, checkpoint_slots=case.get("slots", 0), rmin=case.get("rmin", 0.08), filter_rtol=1e-12,
        objective=case.get("objective", 3), boundaries=case.get("boundaries", 1),
        loadloc=2 if case.get("boundaries", 1) == 1 else 0)  # (the MBB beam: its own load preset, z on x = 0, z = max)
    if kind == "reduced":
        p.reduction, p.basis, p.omega0 = 1, case["basis"], 0.01
    return p


def _op_input(case, seed):
    n = (case["ex"] + 1) * (case["ey"] + 1) * (case["ez"] + 1)
    u = np.random.default_rng([seed, 2]).standard_normal(3 * n)
    u.reshape(case["ez"] + 1, case["ey"] + 1, case["ex"] + 1, 3)[:, :, 0, :] = 0.0  # the clamped face
    return u.astype(np.float32) if case["prec"] == 1 else u


def _gradients(case, seed):
    """Objective and constraint gradients as the update meets them: all negative, peaked; 1 / nel."""
    n = case["ex"] * case["ey"] * case["ez"]
    df = -np.exp(np.random.default_rng([seed, 3]).standard_normal(n))
    return df, np.full(n, 1.0 / n)


def prepare(case, seed):
    x = _density(case, seed)
    ctx = capi.Context(_params(case))
    s = {"case": case, "ctx": ctx}
    if case["kind"] in ("filter", "update"):
        s["x"] = x
        if case["kind"] == "update":
            s["df"], s["dg"] = _gradients(case, seed)
            s["gx"] = float(x.mean() - VOLFRAC)
            s["mma"] = capi.MMA(ctx)
        return s
    s["x"] = torch.from_numpy(x).cuda()
    if case["kind"] == "op":
        torch.cuda.synchronize()
        ctx.set_density(s["x"])
        s["u"] = torch.from_numpy(_op_input(case, seed)).cuda()
        s["y"] = torch.empty_like(s["u"])
    elif case["kind"] == "forward":
        s["out"] = [torch.empty(ctx.nd, dtype=torch.float64, device="cuda") for _ in range(3)]
    else:
        s["df"] = torch.empty(ctx.nel, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()  # (the library works on its own stream)
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "op":
        ctx.op_apply(case["which"], s["u"], s["y"], prec=case["prec"])
        return {"y": s["y"]}
    if kind == "filter":
        xt, xp = ctx.filter_project(s["x"], projection=bool(case["projection"]), beta=4.0, eta=0.15)
        return {"xtilde": xt, "xphys": xp}
    if kind == "update":
        x = s["x"]
        xt, xp = ctx.filter_project(x)
        df, dg = ctx.filter_gradients(xt, s["df"], s["dg"])
        lo, hi = s["mma"].outer_movelimit(0.0, 1.0, 0.2, x)
        xn = s["mma"].update(x, df, s["gx"], dg, lo, hi)
        ch, _ = s["mma"].design_change(xn, x)
        xt, xp = ctx.filter_project(xn)
        return {"df": df, "dg": dg, "x": xn, "change": ch, "xphys": xp, "mnd": ctx.mnd(xp)}
    ctx.set_density(s["x"])
    ctx.complete_initial_state()
    ctx.forward()
    if kind == "forward":
        u, v, a = ctx.get_state(case["steps"], out=s["out"])
        return {"u": u, "v": v, "a": a}
    fx, df = ctx.objective_gradient(s["df"])
    return {"fx": fx, "dfdx": df}


# ---------------------------------------------------------------- work
def work(case):
    """Bytes: every input read once and every output written once, per operation the path consists of; operations:
    the element products in the element's symmetry-adapted basis (about 300 per element and operator)."""
    nel = case["ex"] * case["ey"] * case["ez"]
    nd = 3 * (case["ex"] + 1) * (case["ey"] + 1) * (case["ez"] + 1)
    kind = case["kind"]
    if kind == "op":
        es = 4 if case["prec"] == 1 else 8
        return {"bytes": es * (2 * nd + 2 * nel), "flops": 300 * nel}
    if kind in ("filter", "update"):
        # per filter solve the field in and out, and per solve at least one pass over the nodes' vectors
        solves = 1 if kind == "filter" else 4
        return {"bytes": solves * 8 * (2 * nel + 4 * nd // 3) + (8 * 14 * nel if kind == "update" else 0),
                "flops": solves * 60 * nel}
    # a Newmark step: right-hand side from u, v, a; the solve (at least one preconditioned iteration: operator and
    # vector passes); the corrector
    step_b, step_f = 8 * (4 * nd + 2 * nel) + 8 * (8 * nd + 2 * nel) + 8 * 6 * nd, 3 * 300 * nel
    if kind == "forward":
        return {"bytes": case["steps"] * step_b, "flops": case["steps"] * step_f}
    # an adjoint step: operator on the multiplier, the solve, the sensitivities
    adj_b, adj_f = 8 * (3 * nd + 2 * nel) + 8 * (8 * nd + 2 * nel) + 8 * (7 * nd + 5 * nel), 4 * 300 * nel
    if kind == "gradient":
        return {"bytes": case["steps"] * (step_b + adj_b), "flops": case["steps"] * (step_f + adj_f)}
    nb = case["basis"]
    return {"bytes": nb * step_b + case["steps"] * 8 * ((2 * nb + 8) * nd + 5 * nel),
            "flops": nb * step_f + case["steps"] * (300 * nel + 12 * nb * nd)}


# ---------------------------------------------------------------- the same in plain FP64
_C = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]  # element corners


def _element(h):
    """Stiffness (24 x 24, E = 1) and scalar mass (8 x 8, density 1) of the trilinear box element."""
    lam, mu = NU / ((1 + NU) * (1 - 2 * NU)), 1 / (2 * (1 + NU))
    D = np.zeros((6, 6))
    D[:3, :3] = lam
    D[range(3), range(3)] += 2 * mu
    D[range(3, 6), range(3, 6)] = mu
    K, M = np.zeros((24, 24)), np.zeros((8, 8))
    g = 1 / np.sqrt(3.0)
    s = 2 * np.array(_C, float) - 1
    for p in ((a, b, c) for a in (-g, g) for b in (-g, g) for c in (-g, g)):
        f = 1 + s * np.array(p)
        N = 0.125 * f.prod(1)
        d = [0.125 * s[:, i] * f[:, (i + 1) % 3] * f[:, (i + 2) % 3] * 2 / h[i] for i in range(3)]
        B = np.zeros((6, 24))
        for i in range(3):
            B[i, i::3] = d[i]
        B[3, 0::3], B[3, 1::3] = d[1], d[0]
        B[4, 1::3], B[4, 2::3] = d[2], d[1]
        B[5, 0::3], B[5, 2::3] = d[2], d[0]
        w = 0.125 * h[0] * h[1] * h[2]
        K += w * B.T @ D @ B
        M += w * np.outer(N, N)
    return K, M


def _corner_views(case, v):
    ex, ey, ez = case["ex"], case["ey"], case["ez"]
    return [v[c[2]:c[2] + ez, c[1]:c[1] + ey, c[0]:c[0] + ex] for c in _C]


def _interp(x):
    return EMIN + x ** 3 * (EMAX - EMIN), RMIN + x * (RMAX - RMIN)


def _newmark(case):
    dt = _dt(case)
    return [-1.0, 0.0, 2 / dt, 4 / dt, 1.0, 4 / dt ** 2]


def _exact_op(case, seed):
    h = [_box(case)[2 * i + 1] / case[("ex", "ey", "ez")[i]] for i in range(3)]
    K, M = _element(h)
    kf, mf = _interp(_density(case, seed))
    a = _newmark(case)
    cK, cM = {0: (1.0, 0.0), 1: (0.0, 1.0), 2: (1 + a[2] * BETA, a[5] + a[2] * ALPHA)}[case["which"]]
    u = _op_input(case, seed).astype(np.float64)
    v = u.reshape(case["ez"] + 1, case["ey"] + 1, case["ex"] + 1, 3)
    U = np.stack(_corner_views(case, v), -2).reshape(-1, 24)
    Y = cK * kf[:, None] * (U @ K) + cM * mf[:, None] * (U.reshape(-1, 8, 3).transpose(0, 2, 1) @ M).transpose(
        0, 2, 1).reshape(-1, 24)
    Y = Y.reshape(case["ez"], case["ey"], case["ex"], 8, 3)
    y = np.zeros_like(v)
    for c, w in enumerate(_corner_views(case, y)):
        w += Y[..., c, :]
    y[:, :, 0, :] = v[:, :, 0, :]
    return {"y": y.ravel()}


def _exact_gradient(case, seed):
    """Dense matrices, direct solves, and the discrete adjoint of the Newmark recursion (objective 3: the sum over
    the steps of dt/2 u'Ku; the pulse starts at 0, so the initial state is 0)."""
    ex, ey, ez, T = case["ex"], case["ey"], case["ez"], case["steps"]
    h = [_box(case)[2 * i + 1] / (ex, ey, ez)[i] for i in range(3)]
    KE, M8 = _element(h)
    ME = np.kron(M8, np.eye(3))
    x = _density(case, seed)
    kf, mf = _interp(x)
    nx, ny = ex + 1, ey + 1
    nd = 3 * nx * ny * (ez + 1)
    ids = np.arange(nd // 3).reshape(ez + 1, ny, nx)
    en = np.stack([w.ravel() for w in _corner_views(case, ids)], 1)
    dof = (3 * en[:, :, None] + np.arange(3)).reshape(-1, 24)
    idx = (dof[:, :, None] * nd + dof[:, None, :]).ravel()

    def dense(f, E):
        return np.bincount(idx, (f[:, None, None] * E).ravel(), nd * nd).reshape(nd, nd)

    K, M = dense(kf, KE), dense(mf, ME)
    a = _newmark(case)
    dt = _dt(case)
    free = np.ones((ez + 1, ny, nx, 3))
    free[:, :, 0, :] = 0.0
    free = free.ravel()
    F = np.zeros((ez + 1, ny, nx, 3))
    F[0, :, nx - 1, 1] = 1.0
    F[0, 0, nx - 1, 1] = F[0, ny - 1, nx - 1, 1] = 0.5
    F = F.ravel()
    cK, cM = 1 + a[2] * BETA, a[5] + a[2] * ALPHA
    A = (cK * K + cM * M) * np.outer(free, free)
    A[np.arange(nd), np.arange(nd)] += 1 - free
    L = torch.linalg.cholesky(torch.from_numpy(A))
    Kt, Mt = torch.from_numpy(K), torch.from_numpy(M)

    def solve(b):
        return torch.cholesky_solve(torch.from_numpy(b * free)[:, None], L)[:, 0].numpy()

    def mul(B, v):
        return (B @ torch.from_numpy(np.ascontiguousarray(v))).numpy()

    S = [(np.zeros(nd),) * 3]
    for t in range(1, T + 1):
        u, v, w = S[-1]
        load = np.sin(np.pi * t / 20) / ey if t <= 20 else 0.0
        d = a[2] * u - a[0] * v - a[1] * w
        un = solve(load * F + mul(Mt, a[5] * u + a[3] * v + a[4] * w + ALPHA * d) + BETA * mul(Kt, d))
        S.append((un, a[0] * v + a[1] * w + a[2] * (un - u), -a[3] * v - a[4] * w + a[5] * (un - u)))
    fx = sum(0.5 * dt * s[0] @ mul(Kt, s[0]) for s in S)
    dk, dm = np.zeros(kf.size), np.zeros(kf.size)  # d(fx)/d(kfac, mfac)
    gu, gv, ga = (np.zeros(nd) for _ in range(3))

    def quad(E, p, q):
        return ((p[dof] @ E) * q[dof]).sum(1)

    for t in range(T, 0, -1):
        un = S[t][0]
        u, v, w = S[t - 1]
        gu = gu + dt * mul(Kt, un)
        dk += 0.5 * dt * quad(KE, un, un)
        lam = solve(gu + a[2] * gv + a[5] * ga)
        d = a[2] * u - a[0] * v - a[1] * w
        dk += quad(KE, lam, BETA * d - cK * un)
        dm += quad(ME, lam, a[5] * u + a[3] * v + a[4] * w + ALPHA * d - cM * un)
        kl, ml = mul(Kt, lam), mul(Mt, lam)
        dl = ALPHA * ml + BETA * kl
        gu, gv, ga = (a[5] * ml + a[2] * dl - a[2] * gv - a[5] * ga, a[3] * ml - a[0] * dl + a[0] * gv - a[3] * ga,
                      a[4] * ml - a[1] * dl + a[1] * gv - a[4] * ga)
    return {"fx": float(fx), "dfdx": dk * 3 * x ** 2 * (EMAX - EMIN) + dm * (RMAX - RMIN)}


def _exact_filter(case, x, projection):
    """T' K_F^-1 V T x: the Helmholtz matrix is a sum of products of 1-D matrices, so it is solved in their
    generalised eigenvectors."""
    n = (case["ez"], case["ey"], case["ex"])
    box = _box(case)
    h = [box[5] / n[0], box[3] / n[1], box[1] / n[2]]
    R = case["rmin"] / 2 / np.sqrt(3.0)

    def t_node(f):  # each node takes an eighth of its elements
        for ax in range(3):
            z = np.zeros_like(f.take([0], ax))
            f = 0.5 * (np.concatenate([f, z], ax) + np.concatenate([z, f], ax))
        return f

    def t_elem(f):
        for ax in range(3):
            m = f.shape[ax]
            f = 0.5 * (f.take(range(m - 1), ax) + f.take(range(1, m), ax))
        return f

    b = h[0] * h[1] * h[2] * t_node(x.reshape(n))
    lams, vecs = [], []
    for m, hh in zip(n, h):
        K, M = np.zeros((m + 1, m + 1)), np.zeros((m + 1, m + 1))
        for e in range(m):
            K[e:e + 2, e:e + 2] += np.array([[1, -1], [-1, 1]]) / hh
            M[e:e + 2, e:e + 2] += np.array([[2, 1], [1, 2]]) * hh / 6
        w, Q = np.linalg.eigh(M)
        S = Q / np.sqrt(w) @ Q.T
        w, Q = np.linalg.eigh(S @ K @ S)
        lams.append(np.maximum(w, 0.0))
        vecs.append(S @ Q)
    for ax in range(3):
        b = np.moveaxis(np.tensordot(vecs[ax].T, b, (1, ax)), 0, ax)
    b /= 1 + R * R * (lams[0][:, None, None] + lams[1][None, :, None] + lams[2][None, None, :])
    for ax in range(3):
        b = np.moveaxis(np.tensordot(vecs[ax], b, (1, ax)), 0, ax)
    xt = np.clip(t_elem(b).ravel(), 0.0, 1.0)
    xp = xt
    if projection:
        beta, eta = 4.0, 0.15
        xp = (np.tanh(beta * eta) + np.tanh(beta * (xt - eta))) / (np.tanh(beta * eta) + np.tanh(beta * (1 - eta)))
    return {"xtilde": xt, "xphys": xp}


def exact(case, seed):
    if case["kind"] == "op":
        return _exact_op(case, seed)
    if case["kind"] == "filter":
        return _exact_filter(case, _density(case, seed), case["projection"])
    if case["kind"] == "gradient" and case["objective"] == 3 and case["boundaries"] == 1 and case["prec"] == 0 and \
            case["ex"] * case["ey"] * case["ez"] <= 1024:
        return _exact_gradient(case, seed)
    return None  # (larger solves have no direct method within seconds)
