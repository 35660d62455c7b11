"""The work that users of the contact-QP solver have it do, as timed cases.

A case names an entry point and its sizes; ``prepare`` makes the bodies and
keeps the handles a program keeps (context, matrix, QPs, FEM body, engine),
``run`` makes the calls such a program makes per frame (or per batch) and
returns every result whole.  The bodies are tetrahedral beams on half-space
planes: the meshes, materials and tolerances are the ones of the repository's
own workloads (525-node and 44,541-node beams, batches of 5k-60k DoF beams
with log-uniform stiffness, 1e-6 KKT tolerance).

``exact`` gives the minimiser in 64 bits by a dense active-set solve with
torch, on a system assembled here with numpy.
"""
import gc
import math

import numpy as np
import torch

import mprgp_amd as M
from mprgp_amd import problems

GRAVITY = (0.0, -9.8, 0.0)
STEP = 0.01
DENSITY = 1000.0
EDGE = 0.05


def listed():
    return [
        # the projector alone, as the simulator's forward() calls it beside the solve; the smallest call
        _case("project_525", "project", 20, 4, 4),
        # one small body's solve per frame, interactive use: latency and launches count
        _case("solve_fp64_525", "solve", 20, 4, 4, products=130),
        # a mid-size body in the mixed FP32/FP64 form
        _case("solve_mixed_7k", "solve", 58, 10, 10, precision="mixed", planes=2, products=130),
        # the benchmark's 133,623-DoF beam, plain FP64: one large body on the whole card
        _case("solve_fp64_133k", "solve", 100, 20, 20, planes=2, products=170),
        # many independent QPs advanced together in the mixed form, more matrix data than the caches hold: the largest
        _case("batch_mixed_64", "batch", 0, 0, 0, count=64, dof_lo=8000, dof_hi=100000, precision="mixed", planes=3, products=200),
        # the same in plain FP64, smaller bodies
        _case("batch_fp64_24", "batch", 0, 0, 0, count=24, dof_lo=3000, dof_hi=20000, planes=3, products=250),
        # a whole time step of a small body, every step with its own power method as the reference runs it
        _case("step_power_2k", "step", 30, 7, 7, products=2400),
        # a whole time step of the 133,623-DoF beam, corotational, the step size 2/|A| kept by the caller
        _case("step_corot_133k", "step", 100, 20, 20, material="corotational", keep_alpha=True, products=300),
        # the one-shot drop-in on host arrays (matrix build, upload, power method, solve, download)
        _case("dropin_20k", "dropin", 50, 11, 10, products=1150),
        # coupled rows: ground rows and self-contact rows of 12 nonzeros
        _case("coupled_537", "coupled", 20, 4, 4, contacts=12, products=2000),
        # the comparator solver on the same kind of body
        _case("ica_10k", "ica", 41, 8, 8, products=800),
        # the serving engine: sessions submitted together and collected as they end
        _case("engine_mixed_24", "engine", 0, 0, 0, count=24, dof_lo=3000, dof_hi=30000, precision="mixed", planes=2, products=200),
    ]


def draw(rng):
    kind = rng.choice(["project", "solve", "solve", "solve", "batch", "batch", "step", "step", "dropin", "coupled",
                       "ica", "engine"])
    prec = rng.choice(["fp64", "mixed"])
    if kind in ("batch", "engine"):
        lo = _log(rng, 2000, 8000)
        hi = _log(rng, 2 * lo, 80000)
        return _case(None, kind, 0, 0, 0, count=rng.randint(2, 40 if kind == "batch" else 20), dof_lo=lo, dof_hi=hi,
                     precision=prec, planes=rng.randint(1, 4), products=200)
    top = {"project": 130000, "solve": 130000, "step": 100000, "dropin": 20000, "coupled": 1600, "ica": 10000}[kind]
    nx, ny, nz = _dims(_log(rng, 600 if kind == "coupled" else 1000, top), rng.uniform(2.5, 8.0))
    if ny > 4 and rng.random() < 0.5:
        nz -= 1
    if kind == "solve":
        return _case(None, kind, nx, ny, nz, precision=prec, planes=rng.randint(1, 3), products=150)
    if kind == "step":
        big = nx * ny * nz > 4000
        return _case(None, kind, nx, ny, nz, material=rng.choice(["linear", "corotational"]), keep_alpha=big,
                     products=300 if big else 2400)
    if kind == "coupled":
        return _case(None, kind, nx, ny, nz, contacts=rng.randint(3, 12), products=2000)
    return _case(None, kind, nx, ny, nz, products={"project": 0, "dropin": 1150, "ica": 800}[kind])


def _case(name, kind, nx, ny, nz, **kw):
    case = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "count": 1, "dof_lo": 0, "dof_hi": 0, "precision": "fp64",
            "planes": 1, "material": "linear", "keep_alpha": False, "contacts": 0, "products": 0}
    case.update(kw)
    if name:
        case["name"] = name
    return case


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dims(dof, aspect=5.0):
    nodes = dof / 3.0
    k = max(2, int(round((nodes / aspect) ** (1.0 / 3.0))) - 1)
    return max(2, int(round(nodes / (k + 1) ** 2)) - 1), k, k


def _bodies(case):
    """Grid sizes of the case's bodies (log-spaced DoF for a batch)."""
    if not case["count"] or not case["dof_hi"]:
        return [(case["nx"], case["ny"], case["nz"])]
    n = case["count"]
    f = (case["dof_hi"] / case["dof_lo"]) ** (1.0 / max(1, n - 1))
    return [_dims(case["dof_lo"] * f ** i) for i in range(n)]


def _counts(nx, ny, nz):
    """Nodes, blocks of A and tets of a grid."""
    nodes = (nx + 1) * (ny + 1) * (nz + 1)
    edges = nx * (ny + 1) * (nz + 1) + (nx + 1) * ny * (nz + 1) + (nx + 1) * (ny + 1) * nz
    faces = nx * ny * (nz + 1) + nx * (ny + 1) * nz + (nx + 1) * ny * nz
    return nodes, nodes + 2 * (edges + faces), 5 * nx * ny * nz


def work(case):
    """Each product with A reads its blocks once (the iteration count is the usual one of the case's kind), the
    assembly reads the tets and writes A once, and the vectors go in and out once."""
    total = flops = 0.0
    for dims in _bodies(case):
        nodes, nb, tets = _counts(*dims)
        value = 4 if case["precision"] == "mixed" else 8
        total += case["products"] * nb * (9 * value + 4) + 8 * 3 * nodes * 4
        flops += case["products"] * nb * 18 + 20 * nodes
        if case["kind"] == "step":
            total += 2 * (nb * 72 + tets * 112)
    return {"bytes": total, "flops": flops}


# ------------------------------------------------------------------ bodies


def _mesh(nx, ny, nz):
    """Grid nodes (x slowest) and 5 tets per cell, mirrored in alternate cells so that face diagonals match."""
    x = np.stack(np.meshgrid(np.arange(nx + 1), np.arange(ny + 1), np.arange(nz + 1), indexing="ij"), -1)
    cell = np.stack(np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij"), -1).reshape(-1, 3)
    cuts = np.array([[0, 1, 2, 4], [1, 2, 3, 7], [1, 4, 5, 7], [2, 4, 6, 7], [1, 2, 4, 7]])
    bits = np.array([[(c >> d) & 1 for d in range(3)] for c in range(8)])
    tets = []
    for odd in (0, 1):
        at = cell[cell.sum(1) % 2 == odd]
        corner = bits.copy()
        corner[:, 0] ^= odd
        p = at[:, None, :] + corner[None, :, :]
        node = (p[..., 0] * (ny + 1) + p[..., 1]) * (nz + 1) + p[..., 2]
        tets.append(node[:, cuts].reshape(-1, 4))
    tets = np.concatenate(tets)
    x = x.reshape(-1, 3) * EDGE
    swap = _volume(x, tets) < 0
    tets[swap, 2], tets[swap, 3] = tets[swap, 3].copy(), tets[swap, 2].copy()
    return x, tets


def _volume(x, t):
    a = x[t[:, 0]]
    return np.einsum("ij,ij->i", np.cross(x[t[:, 1]] - a, x[t[:, 2]] - a), x[t[:, 3]] - a) / 6.0


def _body(case, dims, rng):
    """One placed body: rest positions, tets, material, velocities, planes (normal, offset, band) and its rows."""
    x, tets = _mesh(*dims)
    many = case["kind"] in ("batch", "engine")
    tilt = math.radians(rng.uniform(0.0, 10.0) if many or case["planes"] > 1 else rng.uniform(0.0, 2.0))
    x = x @ np.array([[math.cos(tilt), math.sin(tilt), 0.0], [-math.sin(tilt), math.cos(tilt), 0.0], [0.0, 0.0, 1.0]])
    x[:, 1] += 0.005 - x[:, 1].min()
    young = math.exp(rng.uniform(math.log(3e4), math.log(3e5))) if many else 1e5
    poisson = rng.uniform(0.3, 0.48) if many else 0.45
    v = np.zeros_like(x)
    v[:, 1] = -1.0
    v += rng.normal(0.0, 0.05, v.shape)
    planes = [((0.0, 1.0, 0.0), 0.0, math.inf if case["planes"] == 1 else 0.02)]
    for _ in range(case["planes"] - 1):
        a, b = math.radians(rng.uniform(5.0, 30.0)), rng.uniform(0.0, 2 * math.pi)
        n = np.array([math.sin(a) * math.cos(b), math.cos(a), math.sin(a) * math.sin(b)])
        planes.append((tuple(n), -float(np.quantile(x @ n, rng.uniform(0.005, 0.03))), 0.01))
    node, normal, c, taken = [], [], [], np.zeros(len(x), bool)
    for n, p, band in planes:
        hit = np.nonzero((x @ np.array(n) + p - band <= 0) & ~taken)[0]
        taken[hit] = True
        node.append(hit)
        normal.append(np.tile(np.array(n), (hit.size, 1)))
        c.append(np.full(hit.size, -p))
    return {"x": x, "tets": tets, "young": young, "poisson": poisson, "v": v, "planes": planes,
            "node": np.concatenate(node).astype(np.int32), "normal": np.concatenate(normal), "c": np.concatenate(c)}


def _contacts(body, rng, count):
    """`count` self-contact rows: a vertex against the opposite face of its tet, 12 nonzeros each, on nodes of their own."""
    x, used, rows = body["x"], np.zeros(len(body["x"]), bool), []
    if not count:
        return rows
    for t in rng.permutation(len(body["tets"])):
        i, j, k, l = body["tets"][t]
        if len(rows) == count:
            break
        if used[[i, j, k, l]].any():
            continue
        n = np.cross(x[k] - x[j], x[l] - x[j])
        n /= np.linalg.norm(n)
        n = n if n @ (x[i] - x[j]) >= 0 else -n
        w = rng.dirichlet([3.0, 3.0, 3.0])
        entries = sorted([(i, 1.0), (j, -w[0]), (k, -w[1]), (l, -w[2])])
        rows.append(([3 * a + d for a, _ in entries for d in range(3)], [f * n[d] for _, f in entries for d in range(3)],
                     float(n @ (x[i] - w[0] * x[j] - w[1] * x[k] - w[2] * x[l]))))
        used[[i, j, k, l]] = True
    return rows


def _all_rows(case, body, rng):
    """(pointers, columns, values, offsets) of the plane rows and then the contact rows."""
    m = body["node"].size
    col = (3 * body["node"][:, None] + np.arange(3)).ravel().tolist()
    val, ptr, c = body["normal"].ravel().tolist(), (3 * np.arange(m + 1)).tolist(), body["c"].tolist()
    for cols, vals, rhs in _contacts(body, rng, case["contacts"]):
        col += cols
        val += vals
        c.append(rhs)
        ptr.append(len(col))
    return np.array(ptr, np.int32), np.array(col, np.int32), np.array(val), np.array(c)


# ------------------------------------------------------------ prepare, run


def prepare(case, seed):
    gc.collect()  # contexts of dropped states hold their device memory until collected
    rng = np.random.default_rng(seed)
    kind, mixed = case["kind"], case["precision"] == "mixed"
    ctx = M.Context(0)
    material = M.COROTATIONAL if case["material"] == "corotational" else M.LINEAR
    state = {"kind": kind, "ctx": ctx, "qps": [], "x0": [], "b": []}
    for dims in _bodies(case):
        body = _body(case, dims, rng)
        n = body["x"].shape[0]
        fem = M.Fem(ctx, body["x"], body["tets"], body["young"], body["poisson"], DENSITY)
        qp = fem.matrix.qp()
        x0, v0 = body["x"].ravel().copy(), body["v"].ravel().copy()
        fem.assemble(qp, x0, v0, GRAVITY, STEP, material)
        qp.set_rows(body["node"], body["normal"], body["c"])
        qp.set_x(x0)
        state["qps"].append(qp)
        state["x0"].append(x0)
        state["b"].append(qp.get_rhs())
    if kind == "project":
        state["x"] = x0 + 0.02 * rng.standard_normal(x0.size)
        return state
    if kind == "step":
        state.update(fem=fem, v0=v0, sp=fem.step_params(STEP, GRAVITY, material, body["planes"], 10, 1e-4))
    if kind in ("dropin", "coupled", "ica"):
        ptr, col, val, c = _all_rows(case, body, rng)
        csr = type(problems.rows_to_J(body["node"][:1], body["normal"][:1], n))
        state.update(J=csr((val, col, ptr), shape=(c.size, 3 * n)), c=c)
    if kind == "dropin":
        state["A"] = fem.matrix.to_csr()
        return state
    keep = {}
    if kind != "step" or case["keep_alpha"]:
        _, st = M.solve_batch(ctx, state["qps"], tol=1e-6, max_it=0, power_tol=1e-6)
        keep = [{"alpha_bar": s["alpha_bar"]} for s in st]
    else:
        keep = [{}]
    prec = M.MIXED if mixed else M.FP64
    tol = 1e-9 if kind == "coupled" else 1e-6
    state["p"] = [M.params(tol=tol, max_it=4000 if kind == "batch" else 1000, project_first=1, precision=prec,
                           from_x0=1 if kind == "batch" else 0, **k) for k in keep]
    if kind == "engine":
        state["engine"] = M.Engine(ctx, max_active=64)
    return state


def run(state):
    kind, qps = state["kind"], state["qps"]
    qp = qps[0]
    if kind == "project":
        y = qp.project(state["x"])
        return {"y": y, "feasible": qp.is_feasible(y)}
    if kind == "solve":
        qp.set_rhs(state["b"][0])
        qp.set_x(state["x0"][0])
        qp.solve(state["p"][0])
        return {"x": qp.get_x()}
    if kind == "batch":
        M.solve_batch(state["ctx"], qps, per_qp=state["p"])
        return {"x": [q.get_x() for q in qps]}
    if kind == "step":
        state["fem"].set_state(state["x0"][0], state["v0"])
        state["fem"].advance(qp, state["sp"], state["p"][0])
        x, v = state["fem"].get_state()
        return {"x": x, "v": v}
    if kind == "dropin":
        x = state["x0"][0].copy()
        M.MPRGPDecoupledCon.solve(state["A"], state["b"][0], state["J"], state["c"], x, 1e-6, 1000)
        return {"x": x}
    if kind == "coupled":
        qp.set_x(state["x0"][0])
        M.general_solve(qp, state["J"], state["c"], state["p"][0])
        return {"x": qp.get_x()}
    if kind == "ica":
        qp.set_x(state["x0"][0])
        _, _, lam, _ = M.ica_solve(qp, state["J"], state["c"], tol=1e-6)
        return {"x": qp.get_x(), "lam": lam}
    tickets = []
    for q, x0, p in zip(qps, state["x0"], state["p"]):
        q.reset_x()
        tickets.append(state["engine"].submit(q, p))
    for t in tickets:
        state["engine"].wait(t)
    return {"x": [q.get_x() for q in qps]}


# ------------------------------------------------------------------- exact


def exact(case, seed):
    kind, sizes = case["kind"], [3 * _counts(*d)[0] for d in _bodies(case)]
    if kind != "project" and (max(sizes) > 21000 or sum(n ** 3 for n in sizes) > 3e13):
        return None  # dense factorisations of that size take too long
    if kind == "step" and case["material"] != "linear":
        return None  # stops at a Newton tolerance: no closed form
    rng = np.random.default_rng(seed)
    xs, out = [], {}
    for dims in _bodies(case):
        body = _body(case, dims, rng)
        x0 = body["x"].ravel()
        if kind == "project":
            y = (x0 + 0.02 * rng.standard_normal(x0.size)).reshape(-1, 3)
            gap = body["c"] - np.einsum("ij,ij->i", body["normal"], y[body["node"]])
            y[body["node"]] += body["normal"] * np.maximum(gap, 0.0)[:, None]
            return {"y": y.ravel(), "feasible": None}
        x, lam = _minimise(*_system(body), *_all_rows(case, body, rng))
        if x is None:
            return None
        xs.append(x)
    if kind == "step":
        return {"x": xs[0], "v": (xs[0] - x0) / STEP}
    if kind == "ica":
        return {"x": xs[0], "lam": lam}
    return {"x": xs if kind in ("batch", "engine") else xs[0]}


def _system(body):
    """A = M + h^2 K (dense) and A x at the free motion, for the linear material at rest positions x."""
    x, tets, n = body["x"], body["tets"], len(body["x"])
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    vol = _volume(x, tets)
    e = np.stack([x[tets[:, i]] - x[tets[:, 0]] for i in (1, 2, 3)], 1)
    grad = np.linalg.inv(e).transpose(0, 2, 1)
    grad = np.concatenate([-grad.sum(1, keepdims=True), grad], 1)
    lam = body["young"] * body["poisson"] / ((1 + body["poisson"]) * (1 - 2 * body["poisson"]))
    mu = body["young"] / (2 * (1 + body["poisson"]))
    A = torch.zeros(9 * n * n, dtype=torch.float64, device=dev)
    for i in range(4):
        for j in range(4):
            gi, gj = grad[:, i], grad[:, j]
            k = lam * gi[:, :, None] * gj[:, None, :] + mu * gj[:, :, None] * gi[:, None, :]
            k = (k + mu * np.einsum("ti,ti->t", gi, gj)[:, None, None] * np.eye(3)) * (STEP * STEP * vol)[:, None, None]
            at = (3 * tets[:, i, None, None] + np.arange(3)[None, :, None]) * 3 * n + 3 * tets[:, j, None, None] + np.arange(3)
            A.index_add_(0, torch.from_numpy(at.reshape(-1)).to(dev), torch.from_numpy(k.reshape(-1)).to(dev))
    A = A.view(3 * n, 3 * n)
    mass = np.zeros(n)
    np.add.at(mass, tets, np.repeat(DENSITY * vol[:, None] / 4, 4, 1))
    mass = torch.from_numpy(np.repeat(mass, 3)).to(dev)
    rest = torch.from_numpy(x.ravel()).to(dev)
    free = STEP * body["v"].ravel() + STEP * STEP * np.tile(GRAVITY, n)
    A.diagonal().add_(mass)
    # b = A x + M (h v + h^2 g): the forces vanish at rest, so only the free motion moves the minimiser off x
    return A, rest, mass * torch.from_numpy(free).to(dev)


def _minimise(A, rest, push, ptr, col, val, c):
    """argmin 1/2 d'Ad - d'push subject to J (rest + d) >= c by active sets; (x, multipliers), or None if it cycles."""
    dev, n, m = A.device, A.shape[0], c.size
    chol = torch.linalg.cholesky(A)
    J = torch.zeros(m, n, dtype=torch.float64, device=dev)
    row = torch.from_numpy(np.repeat(np.arange(m), np.diff(ptr))).to(dev)
    J[row, torch.from_numpy(col).long().to(dev)] = torch.from_numpy(val).to(dev)
    Y = torch.cholesky_solve(torch.cat([push[:, None], J.T], 1), chol)
    free, Y = Y[:, 0], Y[:, 1:]
    G, r = J @ Y, torch.from_numpy(c).to(dev) - J @ rest - J @ free
    on = r > 0
    for _ in range(200):
        lam = torch.zeros(m, dtype=torch.float64, device=dev)
        if bool(on.any()):
            s = torch.nonzero(on).ravel()
            lam[s] = torch.linalg.solve(G[s][:, s], r[s])
        w = G @ lam - r
        after = torch.where(on, lam > 0, w < 0)
        if bool((after == on).all()):
            return (rest + free + Y @ lam).cpu().numpy(), lam.cpu().numpy()
        on = after
    return None, None
