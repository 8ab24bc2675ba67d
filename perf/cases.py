"""Workloads of the library as a user's program runs them, through the public entry points.

Five kinds of work, over the sizes from neon's example cubes to several million unknowns:

``newton``   :class:`neon_amd.static_matrix` on a :class:`neon_amd.DeviceMesh`: whole load steps
             of an implicit solve (update, assembly, Dirichlet, Krylov, norms) to 1e-8, FP64 or
             mixed precision; returns the displacement.
``linear``   the same phases called one by one, as a program with its own driver does
             (displacement, constitutive update, assembly, constrained dofs, one linear solve);
             returns the correction, the internal force and the right-hand side.
``tangent``  the assembled tangent and internal force handed to the host (for a host solver).
``adjoint``  the gradient of an objective in every element's parameters.
``csr``      the drop-in ``linear_solver``: a host CSR system solved on the device.

A case's mesh is a box of nx x ny x nz hexahedra with jittered interior nodes and materials drawn
from the seed; ``numbering`` is the grid's own or the one a mesh generator writes (corners, edges,
faces, then the volume's nodes).
"""
import math

import numpy as np

import neon_amd
from neon_amd import problems

MODELS = {
    "neohooke": neon_amd.MODEL_NEOHOOKE,
    "j2": neon_amd.MODEL_J2,
    "nonaffine33": neon_amd.MODEL_MICROSPHERE_NONAFFINE | neon_amd.SPHERE_BO33,
    "j2_damage": neon_amd.MODEL_J2_DAMAGE,
}
FORWARD = [(dz, dy, dx) for dz in (-1, 0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1)]


def _case(name, kind, dims, model="neohooke", precision="fp64", steps=1, stretch=0.02, hole=0.0, numbering="grid",
          consistent=False):
    return {"name": name, "kind": kind, "nx": dims[0], "ny": dims[1], "nz": dims[2], "model": model,
            "precision": precision, "steps": steps, "stretch": stretch, "hole": hole, "numbering": numbering,
            "consistent": consistent}


def _csr_case(name, dims, symmetric):
    return {"name": name, "kind": "csr", "nx": dims[0], "ny": dims[1], "nz": dims[2], "symmetric": symmetric}


def listed():
    return [
        # the smallest call of the drop-in solver: a coarse system inside a host program's own loop
        _csr_case("csr_cg_tiny", (6, 5, 7), True),
        # a large host system through the drop-in conjugate gradient
        _csr_case("csr_cg_large", (61, 67, 71), True),
        # the drop-in BiCGSTAB: an unsymmetric (convective) system of ordinary size
        _csr_case("csr_bicgstab", (31, 29, 37), False),
        # the 10^3 cube of the CPU-runnable configuration, clamped, 1 % in 5 load steps
        _case("newton_cube10", "newton", (10, 10, 10), steps=5, stretch=0.01),
        # an ordinary FP64 block, one load step of 2 %
        _case("newton_block32", "newton", (31, 33, 29)),
        # the mixed-precision flagship at a large size, one load step of 2 %
        _case("newton_mixed96", "newton", (96, 96, 96), precision="mixed"),
        # a microsphere rubber part on a generated mesh (boundary nodes numbered first)
        _case("newton_rubber22", "newton", (22, 19, 24), model="nonaffine33", numbering="generated", consistent=True),
        # one linear solve of a large FP64 block inside a user's own Newton loop
        _case("linear_block80", "linear", (79, 83, 77)),
        # the plate with a hole in its plastic range, consistent tangent
        _case("linear_plate64", "linear", (64, 32, 32), model="j2", stretch=0.003, hole=4.0, consistent=True),
        # viscoplastic damage: the unsymmetric tangent and BiCGSTAB
        _case("linear_damage14", "linear", (14, 13, 15), model="j2_damage", stretch=0.0018),
        # the assembled tangent exported to a host solver
        _case("tangent_block16", "tangent", (16, 17, 15)),
        # the parameter gradient (backward direction) of an ordinary block
        _case("adjoint_block40", "adjoint", (41, 40, 38), consistent=True, stretch=0.05),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dims(rng, n, least=2):
    return tuple(max(least, int(round(n * rng.uniform(0.8, 1.2)))) for _ in range(3))


def draw(rng):
    kind = rng.choice(["newton", "newton", "newton", "linear", "linear", "linear", "csr", "csr", "tangent", "adjoint"])
    if kind == "csr":
        symmetric = rng.random() < 0.6
        c = _csr_case("", _dims(rng, _log_int(rng, 5, 60 if symmetric else 36), 3), symmetric)
    elif kind == "tangent":
        c = _case("", kind, _dims(rng, _log_int(rng, 3, 22)))
    elif kind == "adjoint":
        c = _case("", kind, _dims(rng, _log_int(rng, 8, 44)), consistent=True, stretch=0.05)
    elif kind == "newton":
        if rng.random() < 0.25:
            c = _case("", kind, _dims(rng, _log_int(rng, 3, 24)), model="nonaffine33", consistent=True,
                      numbering=rng.choice(["grid", "generated"]))
        else:
            mixed = rng.random() < 0.5
            c = _case("", kind, _dims(rng, _log_int(rng, 4, 76 if mixed else 56)),
                      precision="mixed" if mixed else "fp64", numbering=rng.choice(["grid", "grid", "generated"]),
                      stretch=round(rng.uniform(0.01, 0.03), 4))
    else:
        model = rng.choice(["neohooke", "neohooke", "j2", "j2_damage"])
        if model == "neohooke":
            c = _case("", kind, _dims(rng, _log_int(rng, 5, 76)), numbering=rng.choice(["grid", "grid", "generated"]))
        elif model == "j2":
            n = _log_int(rng, 6, 32)
            c = _case("", kind, (2 * n, n, max(3, int(n * rng.uniform(0.5, 1.0)))), model="j2", stretch=0.003,
                      hole=n / 8.0, consistent=True)
        else:
            c = _case("", kind, _dims(rng, _log_int(rng, 3, 16)), model="j2_damage", stretch=0.0018)
    del c["name"]
    return c


# ------------------------------------------------------------------------------- inputs
def _generated_numbering(X, conn, ijk, shape):
    """Nodes renumbered as a mesh generator writes them: corners, edges, faces, volume."""
    faces = np.sum((ijk == 0) | (ijk == np.array(shape)), axis=1)
    order = np.argsort(-faces, kind="stable")
    new = np.empty(len(order), np.int32)
    new[order] = np.arange(len(order), dtype=np.int32)
    return X[order], new[conn], ijk[order]


def _mesh(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    h = 1.0 / max(nx, ny, nz)
    X, conn, ijk = problems.box_mesh(nx, ny, nz, L=(nx * h, ny * h, nz * h), jitter=0.1, seed=seed + 1,
                                     hole_radius=case["hole"] * h)
    if case["numbering"] == "generated":
        X, conn, ijk = _generated_numbering(X, conn, ijk, (nx, ny, nz))
    E = len(conn)
    p = np.zeros((E, 4))
    if case["model"] in ("j2", "j2_damage"):
        E_mod = 200.0e3 if case["model"] == "j2" else 134.0e3
        p[:, 0] = E_mod / (3.0 * (1.0 - 2.0 * 0.3))
        p[:, 1] = E_mod / (2.0 * (1.0 + 0.3))
        p[:, 2] = problems.uniform(seed + 2, E, 225.0, 275.0) if case["model"] == "j2" else 85.0
        p[:, 3] = 2000.0 if case["model"] == "j2" else 0.0
    else:
        mu = problems.uniform(seed + 2, E, 0.5, 1.5)
        p[:, 0] = 10.0 * mu
        p[:, 1] = mu
        if case["model"] == "nonaffine33":
            p[:, 0] = 3.0 * mu
            p[:, 2] = problems.uniform(seed + 3, E, 6.0, 12.0)
            p[:, 3] = problems.uniform(seed + 4, E, 1.2, 2.5)
    return X, conn, ijk, p


def _boundaries(case, ijk):
    """Rollers on x = 0, y = 0, z = 0 (the clamped foot for the 1 % cube) and the pulled face."""
    axis = 0 if case["model"] == "j2" else 2
    n = (case["nx"], case["ny"], case["nz"])[axis]
    pull = case["stretch"] * n / max(case["nx"], case["ny"], case["nz"])
    clamped = case["steps"] > 1
    zero = [(2, 0), (2, 1), (2, 2)] if clamped else [(0, 0), (1, 1), (2, 2)]
    bcs = [{"name": f"fixed{a}{c}", "dofs": problems.face_dofs(ijk, a, 0, c), "times": [0.0, 1.0], "values": [0.0, 0.0]}
           for a, c in zero]
    bcs.append({"name": "pulled", "dofs": problems.face_dofs(ijk, axis, n, axis), "times": [0.0, 1.0],
                "values": [0.0, pull]})
    return bcs


def _fixed(bcs):
    return np.unique(np.concatenate([b["dofs"] for b in bcs])).astype(np.int32)


def _deformation(X, case, seed):
    """A stretched state near an equilibrium: the homogeneous part and a small disturbance."""
    s = case["stretch"]
    axis = 0 if case["model"] == "j2" else 2
    h = 1.0 / max(case["nx"], case["ny"], case["nz"])
    u = -0.3 * s * X
    u[:, axis] = s * X[:, axis] * (1.0 + 0.1 * np.sin(3.0 * X[:, (axis + 1) % 3]))
    return u.reshape(-1) + problems.uniform(seed + 5, X.size, -0.05 * s * h, 0.05 * s * h)


def _stencil_system(case, seed):
    """A 27-point diffusion system on the nx x ny x nz grid with random conductances, grounded on
    one face (a host program's conduction matrix); unsymmetric: with a convective part."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    z, y, x = (a.reshape(-1) for a in np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij"))
    val = np.zeros((n, 27))
    col = np.zeros((n, 27), np.int64)
    ok = np.zeros((n, 27), bool)
    row = np.arange(n)
    for k, (dz, dy, dx) in enumerate(FORWARD):
        inside = ((z + dz >= 0) & (z + dz < nz) & (y + dy >= 0) & (y + dy < ny) & (x + dx >= 0) & (x + dx < nx))
        ok[:, k] = inside
        col[:, k] = row + (dz * ny + dy) * nx + dx
    for k in range(14, 27):
        w = problems.uniform(seed + 10 + k, n, 0.5, 1.5) / (1 + sum(abs(d) for d in FORWARD[k]))
        i = row[ok[:, k]]
        j = col[i, k]
        val[i, k] = -w[i]
        val[j, 26 - k] = -w[i]
    val[:, 13] = -val.sum(axis=1) + np.where(z == 0, 2.0, 0.0)
    if not case["symmetric"]:
        for k in range(14, 27):
            i = row[ok[:, k]]
            j = col[i, k]
            c = 0.3 * sum(FORWARD[k]) / 3.0
            val[i, k] += c
            val[j, 26 - k] -= c
    rp = np.concatenate([[0], np.cumsum(ok.sum(axis=1))]).astype(np.int32)
    x_true = np.sin(2.0 * z / nz) + 0.1 * problems.normal(seed + 40, n)
    b = np.where(ok, val * x_true[np.where(ok, col, 0)], 0.0).sum(axis=1)
    return (rp, col[ok].astype(np.int32), val[ok]), b, x_true


def prepare(case, seed):
    seed = 1000 * int(seed)
    ctx = neon_amd.Context(0)
    if case["kind"] == "csr":
        A, b, _ = _stencil_system(case, seed)
        cls = neon_amd.conjugate_gradient_hip if case["symmetric"] else neon_amd.biconjugate_gradient_stabilised_hip
        solver = cls(residual_tolerance=1.0e-12, max_iterations=5000, criterion=neon_amd.STOP_RELATIVE, context=ctx)
        return {"case": case, "A": A, "b": b, "x": np.zeros(len(b)), "solver": solver}
    X, conn, ijk, params = _mesh(case, seed)
    tangent = neon_amd.TANGENT_CONSISTENT if case["consistent"] else neon_amd.TANGENT_REFERENCE
    mesh = neon_amd.DeviceMesh(X, conn, params, model=MODELS[case["model"]], tangent=tangent, context=ctx,
                               damage=problems.DAMAGE_CONSTANTS if case["model"] == "j2_damage" else None)
    bcs = _boundaries(case, ijk)
    state = {"case": case, "mesh": mesh}
    if case["kind"] == "newton":
        sim = problems.simulation(steps=case["steps"], precision=case["precision"], norm_mode=1, newton_iterations=20)
        state["driver"] = neon_amd.static_matrix(mesh, sim, bcs)
        return state
    state["u"] = _deformation(X, case, seed)
    state["fixed"] = _fixed(bcs)
    if case["kind"] == "adjoint":
        # the mismatch at observed top nodes
        top = np.nonzero(ijk[:, 2] == case["nz"])[0]
        dJ = np.zeros(X.size)
        dJ[3 * top] = problems.normal(seed + 6, len(top))
        dJ[3 * top + 1] = problems.normal(seed + 7, len(top))
        state["dJ"] = dJ
    else:
        state["b"] = 1.0e-3 * params[0, 1] * problems.uniform(seed + 6, X.size, 0.5, 1.5) / len(X)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "csr":
        state["solver"].solve(state["A"], state["x"], state["b"])
        return state["x"]
    if kind == "newton":
        return state["driver"].solve()
    mesh = state["mesh"]
    if case["model"] == "j2_damage":
        mesh.save_internal_variables(False)
    mesh.set_displacement(state["u"])
    if kind == "adjoint":
        return mesh.adjoint_gradient(state["dJ"], state["fixed"])
    mesh.update_internal_variables(1.0e-3 if case["model"] == "j2_damage" else 0.0)
    mesh.assemble(neon_amd.PRECISION_FP64)
    if kind == "tangent":
        val, f = mesh.download()
        return {"val": val, "f_int": f}
    b = state["b"].copy()
    mesh.enforce_dirichlet(state["fixed"], b)
    solver = neon_amd.SOLVER_CG if mesh.is_symmetric() else neon_amd.SOLVER_BICGSTAB
    x, _, _ = mesh.solve(b, solver=solver, tol=1.0e-12, max_iterations=20000)
    return {"x": x, "b": b, "f_int": mesh.download(stiffness=False)[1]}


def work(case):
    """Solves: about 21 (27-point systems: 3) Krylov iterations per element along the longest side,
    each reading the stored matrix once (the upper half where it is symmetric) and the
    recurrence's ten vector passes; an assembly writes the tangent and reads the state."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    longest = max(nx, ny, nz)
    if case["kind"] == "csr":
        n, nnz = nx * ny * nz, 27 * nx * ny * nz
        its = 3 * longest
        per = 12 * nnz + 80 * n if case["symmetric"] else 2 * (12 * nnz + 80 * n)
        return {"bytes": 12 * nnz + 16 * n + its * per, "flops": its * (2 * nnz + 12 * n) * (1 if case["symmetric"] else 2)}
    N, E = (nx + 1) * (ny + 1) * (nz + 1), nx * ny * nz
    n, nnz = 3 * N, 9 * 27 * N
    width = 4 if case["precision"] == "mixed" else 8
    assembly = {"bytes": width * nnz + 72 * N + E * (32 + 8 * 8 * 16), "flops": 45536 * E}
    if case["kind"] == "tangent":
        return assembly
    symmetric = case["model"] != "j2_damage"
    its = 21 * longest * (1 if symmetric else 2)
    per = width * (nnz // 2 if symmetric else nnz) + 10 * width * n
    solve = {"bytes": its * per, "flops": its * (2 * nnz + 12 * n)}
    count = 5 * case["steps"] if case["kind"] == "newton" else 1
    return {k: count * (assembly[k] + solve[k]) for k in solve}


# ---------------------------------------------------------------- the same in plain numpy
CORNERS = np.array([(-1, -1, -1), (1, -1, -1), (1, 1, -1), (-1, 1, -1), (-1, -1, 1), (1, -1, 1), (1, 1, 1), (-1, 1, 1)], float)


def _shape_gradients():
    g = np.zeros((8, 8, 3))
    for q, point in enumerate(CORNERS / math.sqrt(3.0)):
        f = 1.0 + CORNERS * point
        for c in range(3):
            g[q, :, c] = CORNERS[:, c] * f[:, (c + 1) % 3] * f[:, (c + 2) % 3] / 8.0
    return g


def _neohooke(X, conn, params, u, consistent):
    """Element tangents (E, 8, 8, 3, 3) and forces (E, 8, 3) of the compressible neo-Hooke model."""
    x = X + u.reshape(-1, 3)
    ke = np.zeros((len(conn), 8, 8, 3, 3))
    fe = np.zeros((len(conn), 8, 3))
    lam, mu = params[:, 0] - 2.0 * params[:, 1] / 3.0, params[:, 1]
    eye = np.eye(3)
    for dN in _shape_gradients():
        J0 = np.einsum("eai,aj->eij", X[conn], dN)
        Jx = np.einsum("eai,aj->eij", x[conn], dN)
        F = Jx @ np.linalg.inv(J0)
        J = np.linalg.det(F)
        lnJ = np.log(J)
        sigma = ((lam * lnJ)[:, None, None] * eye + mu[:, None, None] * (F @ F.transpose(0, 2, 1) - eye)) / J[:, None, None]
        g = np.einsum("aj,ejk->eak", dN, np.linalg.inv(Jx))
        w = np.linalg.det(Jx)
        scale = w / J if consistent else w
        fe += w[:, None, None] * np.einsum("eij,eaj->eai", sigma, g)
        ke += (lam * scale)[:, None, None, None, None] * np.einsum("eai,ebj->eabij", g, g)
        m = (mu - lam * lnJ) * scale
        ke += m[:, None, None, None, None] * np.einsum("ebi,eaj->eabij", g, g)
        diag = m[:, None, None] * np.einsum("eak,ebk->eab", g, g)
        diag += w[:, None, None] * np.einsum("eai,eij,ebj->eab", g, sigma, g)
        ke += diag[:, :, :, None, None] * eye
    return ke, fe


def exact(case, seed):
    seed = 1000 * int(seed)
    if case["kind"] == "csr":
        return _stencil_system(case, seed)[2]
    nodes = (case["nx"] + 1) * (case["ny"] + 1) * (case["nz"] + 1)
    if case["model"] != "neohooke" or case["precision"] != "fp64":
        return None
    if case["kind"] == "tangent" and nodes <= 12000:
        X, conn, _, params = _mesh(case, seed)
        ke, fe = _neohooke(X, conn, params, _deformation(X, case, seed), case["consistent"])
        N = len(X)
        f = np.zeros((N, 3))
        np.add.at(f, conn, fe)
        key = (conn[:, :, None].astype(np.int64) * N + conn[:, None, :]).reshape(-1)
        pair, slot = np.unique(key, return_inverse=True)
        K = np.stack([np.bincount(slot, weights=ke[..., i, j].reshape(-1), minlength=len(pair))
                      for i in range(3) for j in range(3)], axis=1)
        row = pair // N
        ptr = np.searchsorted(row, np.arange(N + 1))
        at, deg = np.arange(len(pair)) - ptr[row], np.diff(ptr)[row]
        val = np.zeros(9 * len(pair))
        for i in range(3):
            for j in range(3):
                val[9 * ptr[row] + i * 3 * deg + 3 * at + j] = K[:, 3 * i + j]
        return {"val": val, "f_int": f.reshape(-1)}
    if case["kind"] == "newton" and nodes <= 1400:
        # the equilibrium itself: full Newton with a dense factorisation, straight to the last step
        X, conn, ijk, params = _mesh(case, seed)
        bcs = _boundaries(case, ijk)
        u = np.zeros(X.size)
        for b in bcs:
            u[b["dofs"]] = b["values"][-1]
        free = np.setdiff1d(np.arange(X.size), _fixed(bcs))
        # start from the linear interpolation along the pulled axis
        top = bcs[-1]["dofs"][0]
        start = u[top] / X[top // 3, 2] * X[:, 2]
        u.reshape(-1, 3)[:, 2] = start
        for b in bcs:
            u[b["dofs"]] = b["values"][-1]
        dof = (3 * conn[:, :, None] + np.arange(3)).reshape(len(conn), 24)
        for _ in range(12):
            ke, fe = _neohooke(X, conn, params, u, True)
            f = np.bincount(dof.reshape(-1), weights=fe.reshape(-1), minlength=X.size)
            K = np.zeros((X.size, X.size))
            k24 = ke.transpose(0, 1, 3, 2, 4).reshape(len(conn), 24, 24)
            np.add.at(K, (dof[:, :, None], dof[:, None, :]), k24)
            d = np.linalg.solve(K[np.ix_(free, free)], -f[free])
            u[free] += d
            if np.linalg.norm(d) <= 1e-13 * np.linalg.norm(u):
                break
        return u
    return None
