"""The measured cases: what a user of the library has it do, through the
public entry points of glhip.py, from the smallest calls to the largest.

Kinds (the "kind" of a case):
  residual  glh_residual_into on device buffers: system_rhs = -R at a given
            state and its norm, the line search's operation and what a caller
            with a loop of its own asks for;
  step      one Newton step as FemGL::run takes it: assemble the Jacobian and
            the right-hand side, GMRES to 1e-3, damped update;
  solve     a whole Newton solve of one instance to ||R|| <= 1e-10 ||R0||;
  batch     the same of many slab instances at once;
  predict, grad, train
            the coordinate network of the warm start: inference, one loss and
            gradient, a run of training steps.

Meshes are boxes with A = 0 on the two z faces (or diffusive AdGR walls on all
six), adaptive slabs with hanging nodes, and batches of slabs.  The shape, the
material and the options of a case are in its dict; the noise of the state (or
the network's weights and points) comes from the seed.
"""
import importlib.util
import math
import os

import numpy as np
import torch  # before the library: both then share one HIP runtime

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _load(name):
    spec = importlib.util.spec_from_file_location(name, os.path.join(ROOT, "verkko-hem-repo_amd", name + ".py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


G = _load("glhip")
NC = 18
WALLS_Z = (1, 1, 1, 1, 0, 0)     # natural sides, A = 0 on the z faces
WALLS_ADGR = (2, 2, 3, 3, 4, 4)  # diffusive walls on all six faces
NET = dict(n_freq=64, sigma=0.5, width=256, depth=5, n_out=18)  # the warm start's network


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smoke test's mesh: 64 nodes, launches and latency only
        dict(name="residual_q1_3", kind="residual", mesh="box", degree=1, nx=3, ny=3, nz=3, size=6.0, adgr=False,
             p=20.0, t=0.5),
        # first residuals of a phase-diagram sweep of 256 slabs (the sweep's shapes, 2.9e5 nodes)
        dict(name="residual_q1_slabs256", kind="residual", mesh="slabs", count=256, shape_seed=2),
        # the headline cube: 32^3 Q2 cells, 4.94 M dofs
        dict(name="residual_q2_cube32", kind="residual", mesh="box", degree=2, nx=32, ny=32, nz=32, size=40.0,
             adgr=False, p=26.0, t=0.7),
        # an adaptive slab with hanging nodes, matrix-free under the constraints
        dict(name="step_q1_adaptive", kind="step", mesh="adaptive", nx=16, ny=16, nz=4, levels=2, p=22.0, t=0.8,
             matrix_free=True),
        # the assembled Jacobian (the default operator) on a ragged box with diffusive walls
        dict(name="step_q2_assembled", kind="step", mesh="box", degree=2, nx=17, ny=15, nz=9, size=20.0, adgr=True,
             p=26.0, t=0.7, matrix_free=False),
        # the small reference problem: 8^3 Q1 cells, every option at its default
        dict(name="solve_q1_cube8", kind="solve", mesh="box", degree=1, nx=8, ny=8, nz=8, size=20.0, adgr=False,
             p=20.0, t=0.5, matrix_free=False, fp32=False, restart=30),
        # mixed precision: FP32 matrix-free GMRES inside FP64 refinement, ragged box
        dict(name="solve_q2_mixed", kind="solve", mesh="box", degree=2, nx=21, ny=19, nz=14, size=24.0, adgr=False,
             p=26.0, t=0.7, matrix_free=True, fp32=True, restart=100),
        # the headline: a converged plain FP64 solve of the cube
        dict(name="solve_q2_cube32", kind="solve", mesh="box", degree=2, nx=32, ny=32, nz=32, size=40.0, adgr=False,
             p=26.0, t=0.7, matrix_free=True, fp32=False, restart=100),
        # a batch of slabs in FP32 with assembled Jacobians, the sweep's production form
        dict(name="batch_slabs48_fp32", kind="batch", mesh="slabs", count=48, shape_seed=2, matrix_free=False,
             fp32=True),
        # one loss and gradient of a small batch of points
        dict(name="mlp_grad_1000", kind="grad", points=1000),
        # initial guesses for a set of held-out instances
        dict(name="mlp_predict_150k", kind="predict", points=150011),
        # training steps at the warm start's batch
        dict(name="mlp_train_65536", kind="train", batch=65536, steps=20, data=400000),
    ]


def _log(rng, lo, hi):
    """A whole number spread evenly over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _box(rng, degree, lo, hi):
    n = _log(rng, lo, hi)
    ny, nz = max(lo, n - rng.randrange(0, 5)), max(lo, n - rng.randrange(0, 9))
    return dict(mesh="box", degree=degree, nx=n, ny=ny, nz=nz, size=round(max(12.0, 1.25 * degree * n), 2),
                adgr=rng.random() < 0.3, p=round(rng.uniform(10.0, 30.0), 2), t=round(rng.uniform(0.4, 0.75), 3))


def draw(rng):
    kind = rng.choice(["residual", "residual", "step", "solve", "batch", "predict", "grad", "train"])
    if kind == "residual":
        mesh = rng.choice(["box", "box", "slabs", "adaptive"])
        if mesh == "box":
            degree = rng.choice([1, 2])
            return dict(kind=kind, **_box(rng, degree, 2, 48 if degree == 1 else 32))
        if mesh == "slabs":
            return dict(kind=kind, mesh=mesh, count=_log(rng, 2, 256), shape_seed=rng.randrange(1, 1000))
        return dict(kind=kind, mesh=mesh, nx=_log(rng, 3, 24), ny=_log(rng, 3, 24), nz=rng.randrange(2, 7),
                    levels=rng.randrange(1, 3), p=round(rng.uniform(10.0, 30.0), 2), t=0.8)
    if kind == "step":
        if rng.random() < 0.3:
            return dict(kind=kind, mesh="adaptive", nx=_log(rng, 4, 20), ny=_log(rng, 4, 20), nz=rng.randrange(2, 6),
                        levels=rng.randrange(1, 3), p=round(rng.uniform(18.0, 26.0), 2), t=0.8,
                        matrix_free=rng.random() < 0.7)
        mf = rng.random() < 0.6
        degree = rng.choice([1, 2])
        return dict(kind=kind, matrix_free=mf, **_box(rng, degree, 4, (32 if mf else 20) // degree + 8 * (degree - 1)))
    if kind == "solve":
        fp32 = rng.random() < 0.5
        return dict(kind=kind, matrix_free=True, fp32=fp32, restart=100, **_box(rng, 2, 4, 18))
    if kind == "batch":
        return dict(kind=kind, mesh="slabs", count=_log(rng, 4, 48), shape_seed=rng.randrange(1, 1000),
                    matrix_free=rng.random() < 0.5, fp32=rng.random() < 0.6)
    if kind == "predict":
        return dict(kind=kind, points=_log(rng, 100, 300000))
    if kind == "grad":
        return dict(kind=kind, points=_log(rng, 50, 60000))
    return dict(kind=kind, batch=64 * _log(rng, 16, 1024), steps=rng.randrange(5, 21), data=_log(rng, 50000, 400000))


# --------------------------------------------------------------------- inputs
_meshes = {}  # host meshes by shape: a program builds its mesh once, whatever the states it solves for


def _coef(mp, bt=1.0e10):
    return [mp[0], mp[1], mp[2], mp[3], mp[4], mp[5], *G.K_CONST, bt]


def _slabs(case):
    """Meshes and materials of a sweep: slabs of lateral extent 40 and
    thickness D, A = 0 on the two slab faces (the sweep's uneven Q1 meshes)."""
    rng = np.random.default_rng(case["shape_seed"])
    n, h = case["count"], 20.0
    # the solves keep to the region where the B phase is stable in the slab,
    # so that every instance has one state to converge to
    t = rng.uniform(0.3, 0.75, n) if case["kind"] == "batch" else rng.uniform(0.3, 0.95, n)
    d = rng.uniform(16.0, 40.0, n) if case["kind"] == "batch" else rng.uniform(6.0, 40.0, n)
    p = rng.uniform(0.0, 33.9, n)
    nx, nz = rng.integers(8, 17, n), rng.integers(2 if case["kind"] == "residual" else 4, 9, n)
    meshes, coefs, gaps = [], [], []
    for i in range(n):
        meshes.append(G.Mesh(1, (int(nx[i]), int(nx[i]), int(nz[i])), (-h, -h, -d[i] / 2), (h, h, d[i] / 2), WALLS_Z))
        mp = G.matep(p[i], t[i])[1]
        coefs.append(_coef(mp))
        gaps.append(np.full(meshes[-1].n_nodes, mp[9]))
    return dict(mesh=G.Mesh.concat(meshes), coefs=np.array(coefs), gap=np.concatenate(gaps))


def _mesh(case):
    """Host mesh, materials (one row per instance) and bulk gap per node."""
    key = tuple((k, case[k]) for k in sorted(case) if k in ("kind", "mesh", "degree", "nx", "ny", "nz", "size", "adgr",
                                                            "count", "shape_seed", "levels", "p", "t"))
    if key not in _meshes:
        if len(_meshes) >= 24:
            _meshes.clear()
        if case["mesh"] == "slabs":
            _meshes[key] = _slabs(case)
        else:
            mp = G.matep(case["p"], case["t"])[1]
            if case["mesh"] == "box":
                hx = case["size"] / 2
                hy, hz = hx * case["ny"] / case["nx"], max(6.0, hx * case["nz"] / case["nx"])
                m = G.Mesh(case["degree"], (case["nx"], case["ny"], case["nz"]), (-hx, -hy, -hz), (hx, hy, hz),
                           WALLS_ADGR if case["adgr"] else WALLS_Z)
                bt = 3.0 if case["adgr"] else 1.0e10
            else:
                # 2.5 xi0 lateral cells, thickness 12: refined near the slab
                # faces first, then in a part of the slab
                hx, hy, bt = 1.25 * case["nx"], 1.25 * case["ny"], 1.0e10
                f = G.Forest((case["nx"], case["ny"], case["nz"]), (-hx, -hy, -6.0), (hx, hy, 6.0), WALLS_Z)
                for level in range(case["levels"]):
                    m = f.mesh()
                    lo = m.cell_lo()
                    near = np.minimum(lo[:, 2] + 6.0, 6.0 - lo[:, 2]) < (3.1 if level == 0 else 1.6)
                    f = f.refine((near & (lo[:, 0] < (0.5 * hx if level else hx))).astype(np.uint8))
                m = f.mesh()
            _meshes[key] = dict(mesh=m, coefs=np.array([_coef(mp, bt)]), gap=np.full(m.n_nodes, mp[9]))
    return _meshes[key]


def _state(ms, seed):
    """Bulk B phase of each instance's gap with 5% noise, the constraints applied."""
    m, rng = ms["mesh"], np.random.default_rng(seed)
    U = 0.05 * (2.0 * rng.random((m.n_nodes, NC)) - 1.0) * ms["gap"][:, None]
    U[:, [0, 4, 8]] += ms["gap"][:, None]
    if "mask" not in ms:
        ms["mask"] = ((m.arrays()["node_mask"][:, None] >> np.arange(NC, dtype=np.uint32)) & 1).astype(bool)
        ms["lines"] = m.constraints() if m.n_inst == 1 else dict(n_hanging=0)
    U[ms["mask"]] = 0.0
    L = ms["lines"]
    if L["n_hanging"]:
        row = np.repeat(np.arange(m.n_nodes), np.diff(L["hang_ptr"]))
        V = np.zeros_like(U)
        np.add.at(V, row, L["hang_w"][:, None] * U[L["hang_m"]])
        hang = np.diff(L["hang_ptr"]) > 0
        U[hang] = V[hang]
    return np.ascontiguousarray(U.reshape(-1))


def _context(case, ms):
    ctx = G.Context(0)
    co = ms["coefs"]
    ctx.upload_mesh(ms["mesh"])
    if len(co) > 1:
        ctx.set_materials(co)
    else:
        ctx.set_material(co[0, 0], co[0, 1:6], co[0, 6:9], co[0, 9])
    return ctx


def _points(rng, n):
    """Network inputs (x, y, z, T, p, D), scaled to [-1, 1], and smooth order
    parameter profiles of a slab there, in units of the bulk gap."""
    X = rng.uniform(-1.0, 1.0, (n, 6)).astype(np.float32)
    prof = np.tanh(3.0 * (1.0 - np.abs(X[:, 2])) * (1.5 + X[:, 5]))
    Y = np.zeros((n, 18), np.float32)
    Y[:, 0] = Y[:, 4] = prof * (1.0 + 0.05 * X[:, 3])
    Y[:, 8] = prof * prof * (1.0 - 0.1 * X[:, 3])
    Y[:, 9:] = 0.02 * np.sin(3.0 * X[:, [0, 1, 2, 0, 1, 2, 0, 1, 2]] + 2.0 * X[:, [4]])
    return X, Y


def _weights(rng):
    """Flat parameters of NET: per layer W (K x N, row-major), then b."""
    out = []
    K = 2 * NET["n_freq"]
    for layer in range(NET["depth"] + 1):
        N = NET["n_out"] if layer == NET["depth"] else NET["width"]
        out += [rng.normal(0.0, 1.3 / math.sqrt(K), K * N), rng.normal(0.0, 0.1, N)]
        K = N
    return np.concatenate(out).astype(np.float32)


def _net(seed):
    rng = np.random.default_rng(seed)
    net = G.MLP(seed=seed % 1000, **NET)
    net.set_params(_weights(rng))
    return net, rng


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("predict", "grad", "train"):
        net, rng = _net(seed)
        if kind == "train":
            X, Y = _points(rng, case["data"])
            net.set_data(X, Y)
            # the network has been training for a while: Adam's moments are there
            net.train(40, batch=case["batch"], lr=1e-3, seed=seed % 1000, loss_every=0)
            return dict(case=case, net=net, seed=seed % 1000)
        X, Y = _points(rng, case["points"])
        return dict(case=case, net=net, X=X, Y=Y)
    ms = _mesh(case)
    ctx = _context(case, ms)
    U = _state(ms, seed)
    if kind == "residual":
        dev = torch.device("cuda", 0)
        return dict(case=case, ctx=ctx, U=torch.from_numpy(U).to(dev), R=torch.empty(U.size, dtype=torch.float64, device=dev),
                    norm2=torch.empty(ms["mesh"].n_inst, dtype=torch.float64, device=dev))
    ctx.set_solution(U)
    ctx.store_initial()
    if kind != "step":
        ctx.set_matrix_free(case["matrix_free"])
    return dict(case=case, ctx=ctx, gap=ms["gap"])


# --------------------------------------------------------------------- a pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "predict":
        return state["net"].predict(state["X"])
    if kind == "grad":
        loss, grad = state["net"].loss_grad(state["X"], state["Y"])
        return [grad, np.float32(loss)]
    if kind == "train":
        net = state["net"]
        losses = net.train(case["steps"], batch=case["batch"], lr=1e-3, seed=state["seed"], loss_every=case["steps"])
        return [net.params()[0], losses]
    ctx = state["ctx"]
    if kind == "residual":
        ctx.residual_into(state["U"].data_ptr(), state["R"].data_ptr(), state["norm2"].data_ptr())
        return [state["R"], state["norm2"]]
    ctx.restore_initial()
    if kind == "step":
        ctx.assemble(J=True, R=True, matrix_free=case["matrix_free"])
        ctx.solve(rtol=1e-3, maxit=20000, restart=100)
        ctx.newton_step(step=0.83, damped=True)
        return ctx.solution()
    if kind == "batch":
        ctx.newton_solve(rtol=1e-10, max_newton=60, lin_tol=0.1, lin_maxit=3000, restart=100, fp32=case["fp32"])
    else:
        ctx.newton_solve(rtol=1e-10, max_newton=50, lin_tol=0.1, lin_maxit=20000, restart=case["restart"],
                         fp32=case["fp32"])
    U = ctx.solution()
    if case["fp32"]:
        # the fields of the mixed-precision solves go on as FP32 values in
        # units of the gap, the network's training targets
        return (U.reshape(-1, NC) / state["gap"][:, None]).astype(np.float32)
    return U


# ----------------------------------------------------------------------- work
def _sizes(case):
    """(cells, nodes, dofs, values per cell) of a case's mesh."""
    if case["mesh"] == "box":
        k = case["degree"]
        cells = case["nx"] * case["ny"] * case["nz"]
        nodes = (k * case["nx"] + 1) * (k * case["ny"] + 1) * (k * case["nz"] + 1)
        return cells, nodes, nodes * NC, (k + 1) ** 3
    m = _mesh(case)["mesh"]
    return m.n_cells, m.n_nodes, m.n_nodes * NC, m.ns


def _cell_flops(ns):
    """One product J x (or residual) of a cell: three 1D passes for the values
    and gradients and three for the test functions, 1872 at each point."""
    n1 = 2 if ns == 8 else 3
    return 2 * 18 * 18 * n1 * ns + ns * 1872


def work(case):
    kind = case["kind"]
    if kind in ("predict", "grad", "train"):
        K = [2 * NET["n_freq"]] + [NET["width"]] * NET["depth"]
        N = [NET["width"]] * NET["depth"] + [NET["n_out"]]
        macs = sum(k * n for k, n in zip(K, N))
        par = 4 * (macs + sum(N))
        if kind == "predict":
            return dict(bytes=case["points"] * 4 * (6 + 18) + par, flops=2 * macs * case["points"])
        if kind == "grad":
            return dict(bytes=case["points"] * 4 * (6 + 18) + 2 * par, flops=6 * macs * case["points"])
        # weights and both moments read and written each step
        return dict(bytes=case["steps"] * (case["batch"] * 4 * (6 + 18) + 6 * par),
                    flops=case["steps"] * 6 * macs * case["batch"])
    cells, nodes, n, ns = _sizes(case)
    res = dict(bytes=2 * 8 * n + 4 * cells * ns, flops=cells * _cell_flops(ns))
    if kind == "residual":
        return res
    # GMRES steps of a linear solve: about 10 for the first Newton step from
    # the noise, about the nodes along a side later on (to 0.1); Newton steps
    # of a solve
    side = (cells / max(1, case.get("count", 1))) ** (1.0 / 3.0) * (1 if ns == 8 else 2)
    its = 10 if kind == "step" else max(8, int(side))
    steps = 1 if kind == "step" else 13 if kind == "solve" else 10
    v = 4 if case.get("fp32") else 8
    if case["matrix_free"]:
        prod_b, setup_b = cells * ns * NC * v + 2 * v * n, cells * ns * NC * v + 324 * 8 * nodes
    else:
        nnzb = 20 * nodes if ns == 8 else 56 * nodes  # fewer at the walls
        prod_b, setup_b = nnzb * 324 * v, nnzb * 324 * v
    basis_b = its * v * n // 2 + 2 * v * n       # a step reads the basis so far and writes its vector
    prec_b = 171 * v * nodes + 2 * v * n
    per_it = prod_b + basis_b + prec_b
    prod_f = cells * _cell_flops(ns) if case["matrix_free"] else 2 * 27 * nodes * 324
    return dict(bytes=steps * (its * per_it + setup_b + 2 * res["bytes"]),
                flops=steps * (its * (prod_f + 2 * its * n + 2 * 324 * nodes) + 2 * res["flops"]))


# ------------------------------------------------------------ in 64 bits
def _basis(degree):
    """Values and derivatives of the FE_Q(degree) x Gauss(degree + 1) reference
    element: N[q, a], dN[q, a, k], weights w[q], and the mass of each face."""
    n1 = degree + 1
    x, w = np.polynomial.legendre.leggauss(n1)
    x, w = 0.5 * (x + 1.0), 0.5 * w
    s = np.linspace(0.0, 1.0, n1)

    def lag(t):
        L, dL = np.ones((len(t), n1)), np.zeros((len(t), n1))
        for a in range(n1):
            poly = np.poly1d([1.0])
            for b in range(n1):
                if b != a:
                    poly = poly * np.poly1d([1.0, -s[b]]) / (s[a] - s[b])
            L[:, a], dL[:, a] = poly(t), poly.deriv()(t)
        return L, dL

    def outer(fx, fy, fz):  # x fastest in both indices
        return np.einsum("ia,jb,kc->kjicba", fx, fy, fz).reshape(len(fx) * len(fy) * len(fz), n1 ** 3)

    L, D = lag(x)
    N = outer(L, L, L)
    dN = np.stack([outer(D, L, L), outer(L, D, L), outer(L, L, D)], 2)
    W = np.einsum("k,j,i->kji", w, w, w).reshape(-1)
    M = []
    for f in range(6):
        E = lag(np.array([float(f & 1)]))[0]
        B = [L, L, L]
        B[f // 2] = E
        ww = [w, w, w]
        ww[f // 2] = np.ones(1)
        F = outer(*B)
        M.append(F.T @ (F * np.einsum("k,j,i->kji", ww[2], ww[1], ww[0]).reshape(-1)[:, None]))
    return N, dN, W, np.stack(M)


def _energy(U, cells, h, N, dN, W, M, faces, co):
    """Free energy of the field U [nodes, 18]; co: rows of 10 material values
    per cell (broadcast); faces: (cell, local face, id) rows."""
    X = U[cells]                                                    # [e, a, 18]
    val = torch.einsum("qa,eac->eqc", N, X).reshape(len(cells), -1, 2, 3, 3)
    grad = torch.stack([torch.einsum("qa,eac->eqc", dN[:, :, k], X) / h[:, k, None, None] for k in range(3)], -1)
    grad = grad.reshape(len(cells), -1, 2, 3, 3, 3)                 # part, spin, orbital, direction
    u, v = val[:, :, 0], val[:, :, 1]

    def gram(a, b):
        return (a[..., :, None, :] * b[..., None, :, :]).sum(-1)

    uu, vv, uv = gram(u, u), gram(v, v), gram(u, v)
    P, S, Q, A = uu - vv, uu + vv, uv + uv.transpose(-1, -2), uv.transpose(-1, -2) - uv
    dens = [(u * u).sum((-1, -2)), (v * v).sum((-1, -2)), (u * v).sum((-1, -2))]
    D, T, X2 = dens[0] - dens[1], dens[0] + dens[1], dens[2]
    sq = lambda m: (m * m).sum((-1, -2))  # noqa: E731
    c = [co[:, i, None] for i in range(9)]
    f = (c[0] * T + c[1] * (D * D + 4 * X2 * X2) + c[2] * T * T + c[3] * (sq(P) + sq(Q)) + c[4] * (sq(S) + sq(A))
         + c[5] * (sq(S) - sq(A)))
    div = torch.diagonal(grad, dim1=-2, dim2=-1).sum(-1)
    f = f + c[6] * (grad * grad).sum((-1, -2, -3, -4)) + (c[7] + c[8]) * (div * div).sum((-1, -2))
    F = (f * W * (h[:, 0] * h[:, 1] * h[:, 2])[:, None]).sum()
    for lf, ident in sorted(set(map(tuple, faces[:, 1:].tolist()))):
        if ident < 2 or ident > 4:
            continue
        e = faces[(faces[:, 1] == lf) & (faces[:, 2] == ident), 0]
        on = co[e, 9] < 1e10
        keep = torch.tensor([1.0 if (i % 9) % 3 != ident - 2 else 0.0 for i in range(NC)], dtype=U.dtype, device=U.device)
        a, b = [k for k in range(3) if k != lf // 2]
        Y = X[e] * keep
        s = (Y * torch.einsum("ab,ebc->eac", M[lf], Y)).sum((-1, -2))
        F = F + (on * co[e, 6] / co[e, 9] * h[e, a] * h[e, b] * s).sum()
    return F


def _exact_residual(case, seed):
    ms = _mesh(case)
    m, U = ms["mesh"], _state(ms, seed)
    dev = torch.device("cuda", 0) if torch.cuda.is_available() else torch.device("cpu")
    put = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    a = m.arrays()
    node_off, cell_off = m.instances()
    inst = np.repeat(np.arange(m.n_inst), np.diff(cell_off))
    co = put(ms["coefs"][inst])
    N, dN, W, M = (put(x) for x in _basis(m.deg))
    cells, h = put(a["cell_nodes"].reshape(-1, m.ns).astype(np.int64)), put(a["cell_h"].reshape(-1, 3))
    faces = a["faces"].reshape(-1, 3).astype(np.int64)
    field = put(U.reshape(-1, NC)).requires_grad_(True)
    R = torch.zeros_like(field)
    step = 16384
    for c0 in range(0, m.n_cells, step):
        c1 = min(m.n_cells, c0 + step)
        fc = faces[(faces[:, 0] >= c0) & (faces[:, 0] < c1)] - np.array([c0, 0, 0])
        F = _energy(field, cells[c0:c1], h[c0:c1], N, dN, W, M, put(fc), co[c0:c1])
        R += torch.autograd.grad(F, field)[0]
    R = (0.5 * R).detach().cpu().numpy()
    L = ms["lines"]
    if L["n_hanging"]:
        row = np.repeat(np.arange(m.n_nodes), np.diff(L["hang_ptr"]))
        np.add.at(R, L["hang_m"], L["hang_w"][:, None] * R[row])
        R[np.diff(L["hang_ptr"]) > 0] = 0.0
    R[ms["mask"]] = 0.0
    norm2 = np.array([(R[i0:i1] ** 2).sum() for i0, i1 in zip(node_off[:-1], node_off[1:])])
    return [-R.reshape(-1), norm2]


def _forward(case, seed):
    rng = np.random.default_rng(seed)
    par = torch.from_numpy(_weights(rng).astype(np.float64)).requires_grad_(True)
    net = G.MLP(seed=seed % 1000, **NET)
    B = torch.from_numpy(net.params()[1].astype(np.float64))  # the fixed Fourier matrix, an input
    net.close()
    X, Y = (torch.from_numpy(a.astype(np.float64)) for a in _points(rng, case["points"]))
    ang = 2.0 * math.pi * (X @ B)
    H, at, K = torch.cat([torch.sin(ang), torch.cos(ang)], 1), 0, 2 * NET["n_freq"]
    for layer in range(NET["depth"] + 1):
        n = NET["n_out"] if layer == NET["depth"] else NET["width"]
        H = H @ par[at:at + K * n].reshape(K, n) + par[at + K * n:at + K * n + n]
        at, K = at + K * n + n, n
        if layer < NET["depth"]:
            H = torch.nn.functional.silu(H)
    return par, H, Y


def exact(case, seed):
    """In 64 bits, with plain torch: the residual as the derivative of the
    free energy, the network's output and its loss and gradient.  The solves
    have no such value: GMRES stops at a tolerance, and the minima of the free
    energy are manifolds (phase and spin rotations), of which a solve reaches
    the point its own iteration leads to; so has a trained network."""
    kind = case["kind"]
    if kind == "residual":
        return _exact_residual(case, seed)
    if kind == "predict":
        return _forward(case, seed)[1].detach().numpy()
    if kind == "grad":
        par, H, Y = _forward(case, seed)
        loss = ((H - Y) ** 2).mean()
        return [torch.autograd.grad(loss, par)[0].numpy(), float(loss.detach())]
    return None
