"""Performance cases: the assemble / eliminate / solve work a user of the
framework has it do, through its public entry points.

Families (``kind``):

* ``grid``      a structured Q4 / Hex8 cantilever from inputs resident on the
                device: assembly, Dirichlet elimination, multigrid set-up, solve
                to a relative residual of 1e-10, solution to the host.  The
                benchmark's headline step (256 x 64 x 64 elements), and the
                same call at the small and ragged sizes requests have.
* ``distorted`` the same call on a grid whose interior nodes are moved, so that
                every element matrix is its own (a mapped mesh, as the example's
                cylinder).
* ``host``      the drop-in call sequence on a mesh in no particular numbering,
                host arrays in, displacements out: sort-based assembly and a
                Jacobi-type PCG, in the precisions a user picks.
* ``csc``       the reference's own call: ``assemble_system`` from host arrays
                to the 1-based CSC arrays of the matrix.
* ``batch``     many uneven Hex8 problems assembled and solved together.
* ``sweep``     the example's loop: a displacement sweep on the cylinder, one
                displacement after the other (multigrid) or all at once.
* ``serve``     a burst of requests through the multigrid server, every solution
                taken.

Material and loads are the configurations' own: per-element Young's moduli
log-uniform in [0.1, 10] and N(0, 1) nodal loads, or one modulus and end load
per problem in a batch.
"""
from __future__ import annotations

import math
import sys
import time
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "smearfem.jl_amd"))

import smearfem  # noqa: E402

RTOL = 1e-10
E_LO, E_HI = 0.1, 10.0


# ------------------------------------------------------------- the cases --
def listed():
    return [
        # the headline step: 3.2M free dofs, every stage at full size
        {"name": "grid_256x64x64", "kind": "grid", "ndim": 3, "nx": 256, "ny": 64, "nz": 64},
        # the smallest requests (about 1,000 dofs), bound by latency and launches
        {"name": "grid_11x5x5", "kind": "grid", "ndim": 3, "nx": 11, "ny": 5, "nz": 5},
        # a plane problem with odd element counts
        {"name": "grid_301x97", "kind": "grid", "ndim": 2, "nx": 301, "ny": 97, "nz": 0},
        # a mapped mesh: element matrices all different, operators read from memory
        {"name": "distorted_64x24x24", "kind": "distorted", "ndim": 3, "nx": 64, "ny": 24, "nz": 24},
        # the 64 x 16 x 16 cantilever through the default options (FP64, Jacobi)
        {"name": "host_64x16x16_fp64", "kind": "host", "ndim": 3, "nx": 64, "ny": 16, "nz": 16,
         "precision": "fp64", "preconditioner": "jacobi"},
        # a larger one in mixed precision with node-block Jacobi
        {"name": "host_96x24x24_mixed", "kind": "host", "ndim": 3, "nx": 96, "ny": 24, "nz": 24,
         "precision": "mixed", "preconditioner": "block_jacobi"},
        # the reference's assemble_system on a cube, the matrix back on the host
        {"name": "csc_20", "kind": "csc", "ndim": 3, "ne": 20, "ndof": 3},
        # a few uneven problems, default options of a batch
        {"name": "batch_24_mixed", "kind": "batch", "problems": 24, "precision": "mixed",
         "preconditioner": "jacobi", "item_slices": 8, "blocks_per_cu": 0},
        # half of the 512-problem batch with the tuned launch of its fastest form
        {"name": "batch_256_split", "kind": "batch", "problems": 256, "precision": "split",
         "preconditioner": "block_jacobi", "item_slices": 4, "blocks_per_cu": 3},
        # the example's sweep, each displacement from the previous solution
        {"name": "sweep_24", "kind": "sweep", "ne": 24, "count": 6, "together": False},
        # and all its displacements at once (many right-hand sides)
        {"name": "sweep_16_together", "kind": "sweep", "ne": 16, "count": 16, "together": True},
        # a burst of 24 requests of mixed size and dimension
        {"name": "serve_24", "kind": "serve", "requests": 24, "dof_hi": 300000},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _box(rng, ndim, nodes):
    """Element counts of a cantilever with about this many nodes."""
    aspect = rng.uniform(1.0, 4.0)
    s = max(2, round((nodes / aspect) ** (1.0 / ndim)))
    t = max(2, s + rng.randint(-(s // 4), s // 4)) if ndim == 3 else 0
    nx = max(2, round(nodes / (s * max(t, 1))))
    return {"ndim": ndim, "nx": nx, "ny": s, "nz": t}


def draw(rng):
    kind = rng.choice(["grid", "grid", "grid", "distorted", "host", "host", "csc", "batch", "sweep", "serve"])
    if kind == "grid":
        ndim = rng.choice([2, 3])
        dof = _log(rng, 1e3, 3e6 if ndim == 3 else 8e5)
        return dict(_box(rng, ndim, dof / ndim), kind=kind)
    if kind == "distorted":
        ndim = rng.choice([2, 3, 3])
        return dict(_box(rng, ndim, _log(rng, 3e3, 3e5) / ndim), kind=kind)
    if kind == "host":
        ndim = rng.choice([2, 3, 3])
        c = dict(_box(rng, ndim, _log(rng, 1e3, 1.6e5 if ndim == 3 else 3e4) / ndim), kind=kind)
        c["precision"] = rng.choice(["fp64", "mixed", "split", "fp32_matrix"])
        c["preconditioner"] = rng.choice(["jacobi", "block_jacobi"])
        return c
    if kind == "csc":
        ndim = rng.choice([2, 3])
        ne = round(_log(rng, 2, 120 if ndim == 2 else 22))
        return {"kind": kind, "ndim": ndim, "ne": ne, "ndof": rng.choice([1, ndim])}
    if kind == "batch":
        return {"kind": kind, "problems": round(_log(rng, 2, 200)), "precision": rng.choice(["fp64", "mixed", "split"]),
                "preconditioner": rng.choice(["jacobi", "block_jacobi"]), "item_slices": rng.choice([4, 8]),
                "blocks_per_cu": rng.choice([0, 3])}
    if kind == "sweep":
        together = rng.choice([False, False, True])
        return {"kind": kind, "ne": rng.randint(3, 14 if together else 28), "count": rng.randint(2, 6 if not together else 24),
                "together": together}
    return {"kind": "serve", "requests": rng.randint(3, 20), "dof_hi": round(_log(rng, 1e4, 3e5))}


# ---------------------------------------------------------------- inputs --
def _rng(seed, *more):
    return np.random.Generator(np.random.PCG64([int(seed), *more]))


def _dims(case):
    return (case["nx"], case["ny"]) if case["ndim"] == 2 else (case["nx"], case["ny"], case["nz"])


def _young(seed, n):
    return 10.0 ** _rng(seed, 1).uniform(math.log10(E_LO), math.log10(E_HI), n)


def _inputs(case, seed):
    """Mesh arrays, moduli, loads and clamp of a cantilever case."""
    dims = _dims(case)
    nd = len(dims)
    m = smearfem.structured_mesh(dims, lengths=tuple(d / max(dims) for d in dims))
    young = _young(seed, m.n_elem)
    fixed = smearfem.clamp_x0(m)
    f = smearfem.random_face_load(m, nd - 1, 1, fixed, seed)
    nodes, ien = m.NodeList, m.IEN
    if case["kind"] == "distorted":  # interior nodes moved by up to a fifth of an element
        gi = m.node_grid_index()
        inner = np.ones(m.n_nodes, dtype=bool)
        for d in range(nd):
            inner &= (gi[d] > 0) & (gi[d] < dims[d])
        nodes = nodes + np.where(inner, _rng(seed, 2).uniform(-0.2, 0.2, nodes.shape) / max(dims), 0.0)
    if case["kind"] == "host":  # nodes and elements in no particular order
        rng = _rng(seed, 3)
        new = rng.permutation(m.n_nodes)  # new number of each node
        old = np.argsort(new)
        nodes = np.ascontiguousarray(nodes[:, old])
        order = rng.permutation(m.n_elem)
        ien, young = new[ien[order] - 1] + 1, young[order]
        f, fixed = f.reshape(-1, nd)[old].ravel(), fixed.reshape(-1, nd)[old].ravel()
    return {"nd": nd, "dims": dims, "nodes": nodes, "ien": ien, "id": m.ID, "young": young, "fixed": fixed, "f": f}


def _batch_specs(case, seed):
    """Sizes by the case, materials and end loads by the seed."""
    shape, rng = _rng(case["problems"], 7), _rng(seed, 4)
    out = []
    for _ in range(case["problems"]):
        dims = tuple(int(d) for d in shape.integers(4, 33, size=3))
        E, nu = 10.0 ** rng.uniform(-1.0, 1.0), rng.uniform(0.2, 0.4)
        load = tuple(float(v) for v in rng.uniform(-1.0, 1.0, 2)) + (-1.0,)
        out.append(smearfem.cantilever_spec(dims, young=(E, E), nu=nu, end_load=load))
    return out


def _serve_specs(case, seed):
    """Requests of 1,000 to dof_hi dofs, half of them plane."""
    shape, rng = _rng(case["requests"], case["dof_hi"]), _rng(seed, 5)
    out = []
    for _ in range(case["requests"]):
        nd = 3 if shape.uniform() < 0.5 else 2
        cells = 10.0 ** shape.uniform(3.0, math.log10(case["dof_hi"])) / nd
        s = max(2, round((cells / shape.uniform(1.0, 4.0)) ** (1.0 / nd)))
        dims = (max(2, round(cells / s ** (nd - 1))),) + (s,) * (nd - 1)
        load = tuple(float(v) for v in rng.uniform(-1.0, 1.0, nd))
        out.append(smearfem.cantilever_spec(dims, young=(E_LO, E_HI), nu=0.3, seed=int(rng.integers(0, 2 ** 62)),
                                            end_load=load))
    return out


def _deltas(case, seed):
    d0 = _rng(seed, 6).uniform(0.001, 0.01)
    return [float(d0 + 0.01 * k) for k in range(case["count"])]


def prepare(case, seed):
    kind = case["kind"]
    ctx = smearfem.default_context()
    state = {"case": case, "ctx": ctx}
    if kind in ("grid", "distorted"):
        a = _inputs(case, seed)
        mesh = smearfem.Mesh(ctx, a["ien"].shape[0], a["nodes"], a["ien"], a["nd"], "Q1", a["nd"], a["id"],
                             a["young"], 0.3)
        mesh.set_grid(a["dims"])
        bc = smearfem.BoundaryConditions(ctx, a["f"].size, a["f"], a["fixed"])
        state.update(mesh=mesh, bc=bc)
    elif kind == "host":
        state.update(_inputs(case, seed))
    elif kind == "csc":
        nd, ne = case["ndim"], case["ne"]
        m = smearfem.structured_mesh((ne,) * nd)
        ident = m.ID if case["ndof"] == nd else np.arange(1, m.n_nodes + 1, dtype=np.int64)[:, None]
        state.update(nodes=m.NodeList * _rng(seed, 8).uniform(0.5, 2.0, (nd, 1)), ien=m.IEN, id=ident,
                     young=_young(seed, m.n_elem))
    elif kind == "batch":
        state["specs"] = _batch_specs(case, seed)
    elif kind == "sweep":
        state["deltas"] = _deltas(case, seed)
    else:
        state["specs"] = _serve_specs(case, seed)
        state["server"] = smearfem.Server(ctx, precision="fp64", rtol=RTOL, preconditioner="multigrid")
    return state


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind in ("grid", "distorted"):
        K = state["mesh"].assemble()
        S = smearfem.System(K, state["bc"])
        S.set_grid()
        S.solve("fp64", rtol=RTOL, preconditioner="multigrid")
        q = S.solution()
        S.close()
        K.close()
        return q
    if kind == "host":
        K = smearfem.assemble_system(0, state["nodes"], state["ien"], state["nd"], "Q1", state["nd"], state["id"],
                                     state["young"], 0.3, ctx=ctx, device=True, n_elem=state["ien"].shape[0])
        q = smearfem.solve_system(K, state["f"], state["fixed"], precision=case["precision"], rtol=RTOL,
                                  preconditioner=case["preconditioner"])
        K.close()
        return q
    if kind == "csc":
        K = smearfem.assemble_system(case["ne"], state["nodes"], state["ien"], case["ndim"], "Q1", case["ndof"],
                                     state["id"], state["young"], 0.3, ctx=ctx, device=True)
        out = K.csc_arrays()
        K.close()
        return out
    if kind == "batch":
        B = smearfem.Batch.from_specs(state["specs"], ctx)
        B.solve(case["precision"], rtol=RTOL, item_slices=case["item_slices"], blocks_per_cu=case["blocks_per_cu"],
                preconditioner=case["preconditioner"])
        q = np.concatenate(B.solution())
        B.close()
        return q
    if kind == "sweep":
        return smearfem.displacement_sweep(case["ne"], state["deltas"], rtol=RTOL, together=case["together"],
                                           preconditioner="jacobi" if case["together"] else "multigrid", ctx=ctx).q
    server, specs = state["server"], state["specs"]
    ids = [server.submit(sp) for sp in specs]
    server.drain()
    return [server.take(i, sp.n_dof) for i, sp in zip(ids, specs)]


# ------------------------------------------------------- work, tolerance --
def _sizes(case):
    """(nodes, elements, dofs per node, dimension) of each problem of a case."""
    kind = case["kind"]
    if kind in ("grid", "distorted", "host"):
        all_dims = [_dims(case)]
    elif kind == "csc":
        all_dims = [(case["ne"],) * case["ndim"]]
    elif kind == "sweep":
        all_dims = [(case["ne"],) * 3]
    else:
        all_dims = [sp.dims for sp in (_batch_specs if kind == "batch" else _serve_specs)(case, 0)]
    return [(math.prod(d + 1 for d in dims), math.prod(dims), case.get("ndof", len(dims)), len(dims)) for dims in all_dims]


def work(case):
    """Inputs read once, outputs written once; one multiply and add per
    entry of the matrix (one application of the operator per solution)."""
    kind = case["kind"]
    nbytes = flops = 0.0
    for nodes, elems, ndof, nd in _sizes(case):
        nnz = _nnz_nodes(nodes, elems, nd) * ndof * ndof
        if kind in ("batch", "serve"):  # generated from a spec
            nbytes += 8.0 * nodes * ndof
            flops += 2.0 * nnz
        elif kind == "sweep":
            nbytes += 8.0 * nodes * ndof * case["count"]
            flops += 2.0 * nnz * case["count"]
        else:
            mesh = 8.0 * nodes * nd + (4.0 if kind in ("grid", "distorted") else 8.0) * elems * 2 ** nd + 8.0 * elems
            if kind == "csc":
                nbytes += mesh + 16.0 * nnz
                flops += 2.0 * elems * 2 ** nd * (2 ** nd * ndof) ** 2
            else:
                nbytes += mesh + (8.0 + 1.0 + 8.0) * nodes * ndof
                flops += 2.0 * nnz
    return {"bytes": nbytes, "flops": flops}


def _nnz_nodes(nodes, elems, nd):
    """About the number of coupled node pairs of a grid."""
    side_n, side_e = nodes ** (1.0 / nd), elems ** (1.0 / nd)
    return (side_n + 2.0 * side_e) ** nd


def tolerance(case):
    if case["kind"] == "csc":  # FP64 sums of up to 8 element matrices in another order
        return {"rel": 1e-13, "max": 1e-11}
    # solutions to a relative residual of 1e-10: what two solvers that stop
    # there differ by (the displacement error bar of the benchmark)
    return {"rel": 1e-8, "max": 1e-6}


# -------------------------------------------------- the same in 64 bits --
_CORNER = {2: np.array([[-1, -1], [1, -1], [1, 1], [-1, 1]], dtype=np.float64),
           3: np.array([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1],
                        [-1, -1, 1], [1, -1, 1], [1, 1, 1], [-1, 1, 1]], dtype=np.float64)}


def _element_matrices(X, nu, scalar=False):
    """Element stiffness matrices for unit modulus.  X: [elements, corners,
    dimension] coordinates; 2-point Gauss rule per direction; plane stress in
    2D; ``scalar``: the Laplace operator."""
    nd = X.shape[2]
    C = torch.tensor(_CORNER[nd], device=X.device)
    nen = C.shape[0]
    if nd == 3:
        c = 1.0 / ((1.0 + nu) * (1.0 - 2.0 * nu))
        lam, mu = nu * c, 0.5 / (1.0 + nu)
    else:
        lam, mu = nu / (1.0 - nu * nu), 0.5 / (1.0 + nu)
    width = nen if scalar else nen * nd
    Ke = torch.zeros(X.shape[0], width, width, dtype=torch.float64, device=X.device)
    eye = torch.eye(nd, dtype=torch.float64, device=X.device)
    for g in _CORNER[nd] / math.sqrt(3.0):
        gp = torch.tensor(g, device=X.device)
        one = 0.5 * (1.0 + C * gp)  # [corner, direction]
        dN = torch.stack([0.5 * C[:, d] * torch.prod(torch.cat([one[:, :d], one[:, d + 1:]], 1), 1)
                          for d in range(nd)], 1)
        J = X.transpose(1, 2).contiguous() @ dN  # dx_i / dxi_j
        G = dN @ torch.linalg.inv(J)
        w = torch.linalg.det(J).abs()[:, None, None]
        gg = G @ G.transpose(1, 2).contiguous()
        if scalar:
            Ke += w * gg
            continue
        # (a, i), (b, j): lam G_ai G_bj + mu G_aj G_bi + mu delta_ij G_a . G_b
        ai_bj = G.reshape(-1, width, 1) * G.reshape(-1, 1, width)
        aj_bi = ai_bj.reshape(-1, nen, nd, nen, nd).transpose(2, 4).reshape(-1, width, width)
        same = (gg[:, :, None, :, None] * eye[None, None, :, None, :]).reshape(-1, width, width)
        Ke += w * (lam * ai_bj + mu * aj_bi + mu * same)
    return Ke


def _grid_conn(dims):
    """[elements, corners] 0-based node numbers of a grid (x fastest)."""
    nd = len(dims)
    ax = [np.arange(d) for d in dims] + [np.arange(1)] * (3 - nd)
    k, j, i = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    at = lambda a, b, c: ((i + a) + (dims[0] + 1) * ((j + b) + (dims[1] + 1) * (k + c))).ravel()  # noqa: E731
    quad = [(0, 0), (1, 0), (1, 1), (0, 1)]
    return np.stack([at(a, b, c) for c in range(2 if nd == 3 else 1) for a, b in quad], 1)


def _grid_nodes(dims, lengths):
    ax = [np.linspace(0.0, L, d + 1) for L, d in zip(lengths, dims)]
    return np.stack([g.ravel() for g in np.meshgrid(*ax[::-1], indexing="ij")][::-1])


def _solve64(problems, limit_s=18.0):
    """Displacements of problems {conn, Ke (one or per element), scale, fixed,
    f, q_d, extra (conn, matrices)} by Jacobi-preconditioned CG in 64 bits, one
    recurrence per problem, all in step; None where it takes too long."""
    dev, began = "cuda", time.perf_counter()
    P, L = len(problems), max(p["f"].size for p in problems)
    terms = []
    free = torch.zeros(P, L, dtype=torch.bool, device=dev)
    b, qd = (torch.zeros(P, L, dtype=torch.float64, device=dev) for _ in range(2))
    for k, p in enumerate(problems):
        n = p["f"].size
        free[k, :n] = torch.from_numpy(np.asarray(p["fixed"]) == 0).to(dev)
        b[k, :n] = torch.from_numpy(p["f"]).to(dev)
        qd[k, :n] = torch.from_numpy(p.get("q_d", np.zeros(n))).to(dev)
        for conn, Ke, scale in [(p["conn"], p["Ke"], p["scale"])] + p.get("extra", []):
            nd = Ke.shape[-1] // conn.shape[1]
            dofs = torch.from_numpy(conn).to(dev)[:, :, None] * nd + torch.arange(nd, device=dev)
            terms.append((dofs.reshape(conn.shape[0], -1) + k * L, Ke, None if scale is None else
                          torch.from_numpy(np.asarray(scale, dtype=np.float64)).to(dev)[:, None]))

    def apply(u):
        flat, out = u.reshape(-1), torch.zeros(P * L, dtype=torch.float64, device=dev)
        for dofs, Ke, scale in terms:
            v = flat[dofs]
            y = v @ Ke if Ke.dim() == 2 else (Ke * v[:, None, :]).sum(2)
            out.index_add_(0, dofs.reshape(-1), (y if scale is None else y * scale).reshape(-1))
        return out.reshape(P, L)

    diag = torch.zeros(P * L, dtype=torch.float64, device=dev)
    for dofs, Ke, scale in terms:
        d = torch.diagonal(Ke, dim1=-2, dim2=-1).expand(dofs.shape)
        diag.index_add_(0, dofs.reshape(-1), (d if scale is None else d * scale).reshape(-1))
    inv = torch.where(free, 1.0 / diag.reshape(P, L).clamp_min(1e-300), 0.0)
    r = torch.where(free, b - apply(torch.where(free, 0.0, qd)), 0.0)
    bb = (r * r).sum(1, keepdim=True)
    x, z = torch.zeros_like(r), inv * r
    p, rz = z.clone(), (r * z).sum(1, keepdim=True)
    for it in range(200000):
        if it % 50 == 0:
            if bool(((r * r).sum(1, keepdim=True) <= 1e-26 * bb).all()):
                break
            if time.perf_counter() - began > limit_s:
                return None
        q = torch.where(free, apply(p), 0.0)
        alpha = rz / (p * q).sum(1, keepdim=True).clamp_min(1e-300)
        x += alpha * p
        r -= alpha * q
        z = inv * r
        new = (r * z).sum(1, keepdim=True)
        p = z + (new / rz.clamp_min(1e-300)) * p
        rz = new
    x = (x + torch.where(free, 0.0, qd)).cpu().numpy()
    return [x[k, :p["f"].size] for k, p in enumerate(problems)]


def _gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def _spec_young(seed, n):
    """Log-uniform moduli of a spec: SplitMix64 of (seed, stream 1, element)."""
    u = np.uint64
    with np.errstate(over="ignore"):
        c = u(0x9E3779B97F4A7C15)
        z = (u(seed) ^ u(0xD1B54A32D192ED03) ^ (np.arange(n, dtype=np.uint64) * c)) + c
        z = (z ^ (z >> u(30))) * u(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> u(27))) * u(0x94D049BB133111EB)
        z = z ^ (z >> u(31))
    return E_LO * (E_HI / E_LO) ** (((z >> u(12)).astype(np.float64) + 0.5) * 2.0 ** -52)


def _spec_problem(sp):
    dims, nd = sp.dims, sp.ndim
    lengths = sp.box[1::2]
    conn, nodes = _grid_conn(dims), _grid_nodes(dims, lengths)
    idx = np.stack(np.unravel_index(np.arange(nodes.shape[1]), [d + 1 for d in dims[::-1]]))[::-1]
    share = np.where(idx[0] == dims[0], 1.0, 0.0)
    for d in range(1, nd):
        share = share * np.where((idx[d] == 0) | (idx[d] == dims[d]), 0.5, 1.0) * lengths[d] / dims[d]
    ke = _element_matrices(_gpu(nodes[:, conn[:1]].transpose(1, 2, 0)), sp.nu)[0]
    young = np.full(conn.shape[0], sp.young[0]) if sp.young[0] == sp.young[1] else _spec_young(sp.seed, conn.shape[0])
    return {"conn": conn, "Ke": ke, "scale": young, "fixed": np.repeat(idx[0] == 0, nd),
            "f": (share[:, None] * np.array(sp.traction[:nd])[None, :]).ravel()}


def _sweep_problems(case, seed):
    ne = case["ne"]
    nodes, conn = _grid_nodes((ne,) * 3, (1.0,) * 3), _grid_conn((ne,) * 3)
    bottom, top = nodes[2] == 0.0, nodes[2] == 1.0
    xy = nodes[:2] - 0.5  # the square section mapped to a disc: |x'| = max(|x|, |y|)
    far = np.abs(xy).max(0)
    nodes[:2] = xy * np.where(far > 1e-12, far / np.maximum(np.hypot(xy[0], xy[1]), 1e-300), 0.0)
    faces = np.concatenate([c for c in (conn[bottom[conn[:, 0]]][:, :4], conn[top[conn[:, 4]]][:, 4:])])
    X = _gpu(nodes[:, faces].transpose(1, 2, 0))
    C = torch.tensor(_CORNER[2], device="cuda")
    mass = torch.zeros(X.shape[0], 4, 4, dtype=torch.float64, device="cuda")
    for g in _CORNER[2] / math.sqrt(3.0):
        one = 0.5 * (1.0 + C * torch.tensor(g, device="cuda"))
        N = one[:, 0] * one[:, 1]
        t1 = (X * (0.5 * C[:, 0] * one[:, 1])[None, :, None]).sum(1)
        t2 = (X * (0.5 * C[:, 1] * one[:, 0])[None, :, None]).sum(1)
        mass += torch.linalg.cross(t1, t2).norm(dim=1)[:, None, None] * (N[:, None] * N[None, :])
    eye = torch.eye(3, dtype=torch.float64, device="cuda")
    penalty = (100.0 * mass[:, :, None, :, None] * eye[None, None, :, None, :]).reshape(-1, 12, 12)
    Ke = 40.0 * _element_matrices(_gpu(nodes[:, conn].transpose(1, 2, 0)), 0.4)
    fixed = np.zeros(nodes.shape[1] * 3, dtype=bool)
    fixed[2::3] = bottom | top
    out = []
    for d in _deltas(case, seed):
        qd = np.zeros(fixed.size)
        qd[2::3][top] = -d
        out.append({"conn": conn, "Ke": Ke, "scale": None, "fixed": fixed, "f": np.zeros(fixed.size), "q_d": qd,
                    "extra": [(faces, penalty, None)]})
    return out


def _csc64(case, seed):
    nd, ne, ndof = case["ndim"], case["ne"], case["ndof"]
    nodes = _grid_nodes((ne,) * nd, (1.0,) * nd) * _rng(seed, 8).uniform(0.5, 2.0, (nd, 1))
    conn = _grid_conn((ne,) * nd)
    ke = _element_matrices(_gpu(nodes[:, conn].transpose(1, 2, 0)), 0.3, scalar=ndof == 1)
    if ndof > 1:
        ke = ke * _gpu(_young(seed, conn.shape[0]))[:, None, None]
    dofs = (conn[:, :, None] * ndof + np.arange(ndof)).reshape(conn.shape[0], -1)
    n = nodes.shape[1] * ndof
    key = (dofs[:, None, :] * n + dofs[:, :, None]).ravel()  # column, then row
    at = np.unique(key, return_inverse=True)[1].ravel()
    return [None, None, np.bincount(at, weights=ke.cpu().numpy().ravel())]


def exact(case, seed):
    kind = case["kind"]
    if kind == "csc":
        return _csc64(case, seed)
    if kind == "batch":
        if case["problems"] > 64:  # memory for the padded vectors grows with the batch
            return None
        q = _solve64([_spec_problem(sp) for sp in _batch_specs(case, seed)])
        return None if q is None else np.concatenate(q)
    if kind == "serve":
        specs = _serve_specs(case, seed)
        out, spent = [None] * len(specs), time.perf_counter()
        for k, sp in enumerate(specs):
            q = _solve64([_spec_problem(sp)], 18.0 - (time.perf_counter() - spent))
            if q is None:
                break
            out[k] = q[0]
        return out
    if kind == "sweep":
        # linear in the displacement: one solve, scaled
        problems, deltas = _sweep_problems(case, seed), _deltas(case, seed)
        q = _solve64(problems[:1])
        return None if q is None else [q[0] * (d / deltas[0]) for d in deltas]
    a = _inputs(case, seed)
    conn = a["ien"] - 1
    if kind == "distorted":
        ke = _element_matrices(_gpu(a["nodes"][:, conn].transpose(1, 2, 0)), 0.3)
    else:
        ke = _element_matrices(_gpu(a["nodes"][:, conn[:1]].transpose(1, 2, 0)), 0.3)[0]
    q = _solve64([{"conn": conn, "Ke": ke, "scale": a["young"], "fixed": a["fixed"], "f": a["f"]}])
    return None if q is None else q[0]
