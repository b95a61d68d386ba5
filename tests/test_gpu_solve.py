"""GPU Dirichlet elimination + solve against direct solves of the oracle's K.

Bar (every precision mode): displacement within 1e-8 relative
(||u - u_ref||_2 / ||u_ref||_2) of a direct FP64 solve of the reference's
K_ff u = C'(f - K q_d).  Small cases are solved to relative residual 1e-12;
the 64x16x16 cantilever to 1e-10 (its FP64 attainable residual is about
3e-11: scipy's direct solve itself reaches 2.7e-11).  Solutions are bitwise
reproducible run to run.
"""
import json
from pathlib import Path

import numpy as np
import pytest
import scipy.sparse.linalg as spla

import oracle as O
import smearfem
from smearfem.mesh import clamp_x0, element_young_loguniform, face_load, random_face_load, structured_mesh
from smearfem.solve import BoundaryConditions, System, solve_system

pytestmark = pytest.mark.gpu
GOLD = Path(__file__).resolve().parent / "golden"
ERR = 1e-8


def relerr(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def device_K(ctx, m, young=1.0, nu=0.3, coords=None):
    return smearfem.assemble_system(0, m.NodeList if coords is None else coords, m.IEN, m.ndim, "Q1", m.ndim, m.ID,
                                    young, nu, ctx=ctx, device=True, n_elem=m.n_elem)


def oracle_direct(m, fixed, f, q_d=None, young=1.0, nu=0.3, coords=None):
    K = O.assemble_system(0, m.NodeList if coords is None else coords, m.IEN, m.ndim, "Q1", m.ndim, m.ID, young,
                          nu, n_elem=m.n_elem)
    Kff, rhs = O.eliminate(K, fixed, f, q_d)
    u = O.dense_solve(Kff, rhs) if Kff.shape[0] <= 4000 else spla.spsolve(Kff.tocsc(), rhs)
    return O.recombine(fixed, q_d, u), K


@pytest.mark.parametrize("precision,fmt,pc", [("fp64", "csr", "jacobi"), ("fp64", "bsr", "jacobi"),
                                              ("mixed", "bsr", "jacobi"), ("mixed", "csr", "jacobi"),
                                              ("fp32_matrix", "bsr", "jacobi"), ("fp32_matrix", "csr", "jacobi"),
                                              ("split", "bsr", "jacobi"), ("fp64", "bsr", "block_jacobi"),
                                              ("mixed", "bsr", "block_jacobi"), ("split", "bsr", "block_jacobi")])
def test_cfg1_q4_plane_strain_cantilever(ctx, precision, fmt, pc):
    # unit square 32x32, E=1, nu=0.3 plane strain via (E/(1-nu^2), nu/(1-nu)),
    # left edge clamped, unit traction (+x) on the right edge
    print(f"[case] cfg1 {precision} {fmt} {pc}", flush=True)
    m = structured_mesh((32, 32))
    E, nu = 1.0 / (1 - 0.09), 0.3 / 0.7
    fixed = clamp_x0(m)
    f = face_load(m, 0, 1, 0, 1.0)
    K = device_K(ctx, m, E, nu)
    q, R, st = solve_system(K, f, fixed, precision=precision, fmt=fmt, rtol=1e-12, reactions=True,
                            return_stats=True, preconditioner=pc)
    K.close()
    q_ref, Kref = oracle_direct(m, fixed, f, young=E, nu=nu)
    assert st["converged"] and st["rel_residual"] <= 1e-12
    assert relerr(q, q_ref) <= ERR
    assert np.abs(q[fixed == 1]).max() == 0.0
    # equilibrium: reactions balance the applied load
    assert np.abs(R[fixed == 1].reshape(-1, 2).sum(0) + f.reshape(-1, 2).sum(0)).max() < 1e-9
    assert np.abs(R[fixed == 0]).max() == 0.0


@pytest.mark.parametrize("precision,pc", [("fp64", "jacobi"), ("mixed", "jacobi"), ("fp32_matrix", "jacobi"),
                                          ("split", "jacobi"), ("fp64", "block_jacobi"), ("mixed", "block_jacobi"),
                                          ("split", "block_jacobi")])
def test_hex8_cantilever_per_element_young(ctx, precision, pc):
    print(f"[case] hex8 12x4x4 {precision} {pc}", flush=True)
    m = structured_mesh((12, 4, 4), lengths=(3.0, 1.0, 1.0))
    young = element_young_loguniform(m.n_elem, 0.1, 10.0, seed=7)
    fixed = clamp_x0(m)
    f = random_face_load(m, 2, 1, fixed, seed=3)
    K = device_K(ctx, m, young)
    q, st = solve_system(K, f, fixed, precision=precision, rtol=1e-12, return_stats=True, preconditioner=pc)
    K.close()
    q_ref, _ = oracle_direct(m, fixed, f, young=young)
    assert st["converged"]
    assert relerr(q, q_ref) <= ERR


def test_cfg2_against_direct_fixture(ctx):
    gold = json.loads((GOLD / "cfg2_direct.json").read_text())
    m = structured_mesh(gold["dims"], lengths=gold["lengths"])
    fixed = clamp_x0(m)
    f = face_load(m, 0, 1, 2, -1.0)
    K = device_K(ctx, m)
    assert K.nnz == gold["nnz_K"]
    bc = BoundaryConditions(ctx, K.shape[0], f, fixed)
    S = System(K, bc)
    bc.close()
    assert S.n_free == gold["n_free"] and S.nnz == gold["nnz_Kff"]
    for precision, fmt, pc in (("fp64", "csr", "jacobi"), ("fp64", "bsr", "jacobi"), ("mixed", "bsr", "jacobi"),
                               ("fp32_matrix", "bsr", "jacobi"), ("split", "bsr", "jacobi"),
                               ("split", "bsr", "block_jacobi"), ("mixed", "bsr", "block_jacobi")):
        print(f"[case] cfg2 {precision} {fmt} {pc}", flush=True)
        st = S.solve(precision, fmt, rtol=1e-10, preconditioner=pc)
        q, R = S.solution(reactions=True)
        u = q[fixed == 0]
        assert abs(np.linalg.norm(u) - gold["norm_u"]) <= ERR * gold["norm_u"]
        su = np.array(gold["sample_u"])
        assert np.abs(u[gold["sample_idx"]] - su).max() <= ERR * np.abs(su).max()
        gi = m.node_grid_index()
        tip = np.repeat(gi[0] == 64, 3)
        assert abs(q[tip][2::3].mean() - gold["tip_mean_uz"]) <= ERR * abs(gold["tip_mean_uz"])
        assert np.allclose(R[fixed == 1].reshape(-1, 3).sum(0), gold["reaction_sum"], atol=1e-9)
        print(f"  iterations={st['iterations']} updates={st['fp64_updates']} ms={st['solve_ms']:.1f}", flush=True)
    S.close()
    K.close()


def test_patch_test_prescribed_linear_field(ctx):
    m = structured_mesh((6, 4, 5), lengths=(2.0, 1.0, 1.5))
    rng = np.random.default_rng(5)
    gi = m.node_grid_index()
    interior = (gi[0] > 0) & (gi[0] < 6) & (gi[1] > 0) & (gi[1] < 4) & (gi[2] > 0) & (gi[2] < 5)
    coords = m.NodeList.copy()
    coords[:, interior] += 0.05 * rng.standard_normal((3, interior.sum()))
    A = rng.standard_normal((3, 3)) * 0.1
    u_lin = (A @ coords).T.reshape(-1)
    fixed = np.repeat(~interior, 3).astype(np.uint8)
    K = device_K(ctx, m, coords=coords)
    for precision in ("fp64", "mixed", "fp32_matrix", "split"):
        q = solve_system(K, None, fixed, u_lin, precision=precision, rtol=1e-13)
        assert np.abs(q - u_lin).max() <= 1e-10 * np.abs(u_lin).max()
    K.close()


def test_partial_dof_clamp_every_path(ctx):
    # setboundaryCond-style constraints: only the z dof of the bottom and top
    # nodes prescribed (examples/vector3D.jl:159-168) plus one pinned corner
    m = structured_mesh((4, 4, 4))
    gi = m.node_grid_index()
    fixed = np.zeros(m.n_dof, dtype=np.uint8)
    q_d = np.zeros(m.n_dof)
    bottom, top = gi[2] == 0, gi[2] == 4
    fixed[2::3] = bottom | top
    q_d[2::3] = np.where(top, -0.05, 0.0)
    fixed[0:3] = 1  # pin node 1 to remove rigid motion in x, y
    fixed[3 * 4 + 1] = 1  # and node 5's y (rotation about z)
    K = device_K(ctx, m, 40.0, 0.4)
    bc = BoundaryConditions(ctx, K.shape[0], None, fixed, q_d)
    S = System(K, bc)
    bc.close()
    # nodes with some dofs fixed: padded node blocks (unit diagonal on the
    # fixed dofs) carry every block path; the scalar rows remain available
    assert S.block == 3
    q_ref, _ = oracle_direct(m, fixed, None, q_d, young=40.0, nu=0.4)
    for prec, fmt, pc, rtol in (("fp64", "csr", "jacobi", 1e-12), ("fp64", "bsr", "jacobi", 1e-12),
                                ("fp64", "bsr", "block_jacobi", 1e-12), ("split", "bsr", "block_jacobi", 1e-12),
                                ("mixed", "bsr", "block_jacobi", 1e-11), ("mixed", "csr", "jacobi", 1e-11)):
        st = S.solve(prec, fmt, rtol=rtol, preconditioner=pc)
        assert st["format"] == fmt and st["stop_reason"] == 1
        q = S.solution()
        assert relerr(q, q_ref) <= ERR, (prec, fmt, pc)
        assert np.all(q[fixed == 1] == q_d[fixed == 1])
    # a warm start from a solution converged to the same tolerance needs no iteration
    S.solve("fp64", "bsr", rtol=1e-12)
    st = S.solve("fp64", "bsr", rtol=1e-12, x0_zero=False)
    assert st["iterations"] <= 1
    S.close()
    K.close()


def test_solve_bitwise_reproducible(ctx):
    m = structured_mesh((16, 6, 6), lengths=(3.0, 1.0, 1.0))
    fixed = clamp_x0(m)
    f = random_face_load(m, 2, 1, fixed, seed=1)
    K = device_K(ctx, m, element_young_loguniform(m.n_elem, 0.1, 10.0, seed=2))
    for precision, pc in (("fp64", "jacobi"), ("mixed", "jacobi"), ("fp32_matrix", "jacobi"), ("split", "jacobi"),
                          ("split", "block_jacobi"), ("mixed", "block_jacobi")):
        a, sa = solve_system(K, f, fixed, precision=precision, rtol=1e-10, return_stats=True, preconditioner=pc)
        b, sb = solve_system(K, f, fixed, precision=precision, rtol=1e-10, return_stats=True, preconditioner=pc)
        assert np.array_equal(a, b) and sa["iterations"] == sb["iterations"]
    K.close()


def test_zero_load_and_iteration_cap(ctx):
    m = structured_mesh((6, 3, 3))
    fixed = clamp_x0(m)
    K = device_K(ctx, m)
    q, st = solve_system(K, None, fixed, return_stats=True)
    assert st["converged"] and st["iterations"] == 0 and not q.any()
    f = face_load(m, 0, 1, 2, -1.0)
    with pytest.raises(smearfem.NotConvergedError):
        solve_system(K, f, fixed, rtol=1e-14, max_iter=3)
    K.close()


def test_unattainable_tolerance_stops_on_stagnation(ctx):
    # 1e-15 is below what FP64 arithmetic can reach for a bending cantilever:
    # the solver must stop by itself (stagnation), not run to max_iter
    m = structured_mesh((16, 4, 4), lengths=(4.0, 1.0, 1.0))
    fixed = clamp_x0(m)
    f = face_load(m, 0, 1, 2, -1.0)
    K = device_K(ctx, m)
    bc = BoundaryConditions(ctx, K.shape[0], f, fixed)
    S = System(K, bc)
    bc.close()
    for precision in ("fp64", "mixed"):
        st = S.solve(precision, rtol=1e-15, max_iter=100000, raise_on_fail=False)
        assert st["status"] == smearfem.NotConvergedError.code
        assert st["stop_reason"] == 3 and st["iterations"] < 20000
        assert st["rel_residual"] < 1e-9  # still the best FP64-accurate answer
        # it stopped at the rounding floor eps*|| |rhs| + |K||x| || / ||rhs||
        assert 0 < st["floor_residual"] < 1e-10 and st["rel_residual"] <= 20 * st["floor_residual"]
    S.close()
    K.close()


@pytest.mark.parametrize("split", ["1", "4"])
@pytest.mark.parametrize("dims", [(1, 1, 1), (4, 3, 3), (7, 3, 1), (5, 4, 8), (9, 7), (1, 1), (33, 3)])
def test_operator_pass_forms(dims, split, monkeypatch):
    # the sliced operator pass with a wavefront per slice and with a block per
    # slice: row counts around the 64 of a slice (4, 64, 64, 225, 72, 2, 132
    # block rows), rows narrower than the columns loaded early, every
    # precision, and the iteration cap met exactly
    print(f"[case] operator pass {dims} split={split}", flush=True)
    monkeypatch.setenv("SFEM_SELL_SPLIT", split)
    ctx = smearfem.Context(0)
    m = structured_mesh(dims)
    young = element_young_loguniform(m.n_elem, 0.1, 10.0, seed=11)
    fixed = clamp_x0(m)
    f = random_face_load(m, m.ndim - 1, 1, fixed, seed=12)
    perm = np.random.default_rng(13).permutation(m.n_nodes)  # node k is numbered perm[k]
    inv = np.argsort(perm)
    f, fixed = f.reshape(-1, m.ndim)[inv].ravel(), fixed.reshape(-1, m.ndim)[inv].ravel()
    nodes, ien = m.NodeList[:, inv], perm[m.IEN - 1] + 1
    K = smearfem.assemble_system(0, nodes, ien, m.ndim, "Q1", m.ndim, m.ID, young, 0.3, ctx=ctx, device=True,
                                 n_elem=m.n_elem)
    Kr = O.assemble_system(0, nodes, ien, m.ndim, "Q1", m.ndim, m.ID, young, 0.3, n_elem=m.n_elem)
    Kff, rhs = O.eliminate(Kr, fixed, f)
    q_ref = O.recombine(fixed, None, O.dense_solve(Kff, rhs))
    bc = BoundaryConditions(ctx, K.shape[0], f, fixed)
    S = System(K, bc)
    for precision, pc in (("fp64", "jacobi"), ("fp64", "block_jacobi"), ("mixed", "jacobi"),
                          ("mixed", "block_jacobi"), ("split", "block_jacobi"), ("fp32_matrix", "jacobi")):
        st = S.solve(precision, "bsr", rtol=1e-12, preconditioner=pc)
        assert st["stop_reason"] == 1 and relerr(S.solution(), q_ref) <= ERR, (precision, pc)
    full = S.solve("fp64", "bsr", rtol=1e-12)
    if full["iterations"] > 3:
        st = S.solve("fp64", "bsr", rtol=1e-12, max_iter=3, raise_on_fail=False)
        assert st["iterations"] == 3 and st["stop_reason"] == 4
    S.close()
    bc.close()
    K.close()
    ctx.close()


@pytest.mark.parametrize("split,fmt", [("1", "bsr"), ("4", "bsr"), ("1", "csr")])
def test_operator_pass_timing(split, fmt, monkeypatch):
    # time_kernels: every iteration's operator pass is timed, FP64 residuals
    # are not, whatever the polling interval; the bytes are those of one pass:
    # the matrix, p and q, and z and the new p where the pass forms p
    print(f"[case] pass timing split={split} {fmt}", flush=True)
    monkeypatch.setenv("SFEM_SELL_SPLIT", split)
    ctx = smearfem.Context(0)
    m = structured_mesh((24, 8, 8))
    young = element_young_loguniform(m.n_elem, 0.1, 10.0, seed=17)
    fixed = clamp_x0(m)
    K = device_K(ctx, m, young)
    bc = BoundaryConditions(ctx, K.shape[0], random_face_load(m, 2, 1, fixed, seed=18), fixed)
    S = System(K, bc)
    n, nnz, slices = S.n_free, S.nnz, -(-(S.n_free // 3) // 64)
    vecs = 4 if split == "4" or fmt == "csr" else 2  # CSR forms p in its gathers up to 30,000 dofs
    modes = [("fp64", 8, 8), ("mixed", 4, 4)] + ([("split", 6, 8)] if fmt == "bsr" else [])
    for precision, vb, xb in modes:
        plain = S.solve(precision, fmt, rtol=1e-10)
        for every in (1, 7, 64, 200):
            st = S.solve(precision, fmt, rtol=1e-10, check_every=every, time_kernels=True)
            assert st["iterations"] == plain["iterations"] and st["fp64_updates"] == plain["fp64_updates"] > 2
            assert st["spmv_timed"] == st["iterations"] and 0.0 < st["spmv_ms"] < st["solve_ms"]
        if fmt == "bsr":
            op = nnz // 9 * (9 * vb + 4) + 12 * slices + 8
        else:
            op = nnz * (vb + 4) + 4 * (n + 1)
        assert st["spmv_bytes"] == op + vecs * n * xb
    for h in (S, bc, K, ctx):
        h.close()


@pytest.mark.parametrize("dims", [(121, 122), (122, 122), (122, 123), (25, 19, 19)])
def test_csr_pass_forms(ctx, dims):
    # the scalar CSR operator pass on both sides of the 30,000 dofs up to which
    # it forms p in its gathers (29,766, 30,012, 30,256 and 30,000 dofs)
    print(f"[case] csr pass {dims}", flush=True)
    m = structured_mesh(dims)
    fixed = clamp_x0(m)
    f = random_face_load(m, m.ndim - 1, 1, fixed, seed=21)
    q_ref, Kr = oracle_direct(m, fixed, f)
    K = device_K(ctx, m)
    bc = BoundaryConditions(ctx, K.shape[0], f, fixed)
    S = System(K, bc)
    for precision in ("fp64", "mixed", "fp32_matrix"):
        st = S.solve(precision, "csr", rtol=1e-11, time_kernels=True)
        assert st["stop_reason"] in (1, 3) and relerr(S.solution(), q_ref) <= ERR, precision
        vecs = 4 if S.n_free <= 30000 else 2
        vb, xb = {"fp64": (8, 8), "mixed": (4, 4), "fp32_matrix": (4, 8)}[precision]
        assert st["spmv_bytes"] == S.nnz * (vb + 4) + 4 * (S.n_free + 1) + vecs * S.n_free * xb
    for h in (S, bc, K):
        h.close()


@pytest.mark.parametrize("dims", [(320, 255), (320, 256)])
def test_operator_pass_line(ctx, dims):
    # 1,280 slices, the last size whose slices a block's wavefronts share, and
    # 1,285: both against a direct solve, in a shuffled numbering, and the
    # bytes of the pass tell the form (z read and p written, or not)
    print(f"[case] operator pass line {dims}", flush=True)
    m = structured_mesh(dims, lengths=tuple(d / max(dims) for d in dims))
    fixed = clamp_x0(m)
    f = random_face_load(m, 1, 1, fixed, seed=22)
    perm = np.random.default_rng(23).permutation(m.n_nodes)
    inv = np.argsort(perm)
    f, fixed = f.reshape(-1, 2)[inv].ravel(), fixed.reshape(-1, 2)[inv].ravel()
    mesh = (0, m.NodeList[:, inv], perm[m.IEN - 1] + 1, 2, "Q1", 2, m.ID, 1.0, 0.3)
    K = smearfem.assemble_system(*mesh, ctx=ctx, device=True, n_elem=m.n_elem)
    Kff, rhs = O.eliminate(O.assemble_system(*mesh, n_elem=m.n_elem), fixed, f)
    q_ref = O.recombine(fixed, None, spla.spsolve(Kff.tocsc(), rhs))
    bc = BoundaryConditions(ctx, K.shape[0], f, fixed)
    S = System(K, bc)
    slices = -(-S.n_free // 128)
    for precision, vb, xb in (("fp64", 8, 8), ("mixed", 4, 4), ("fp32_matrix", 4, 8), ("split", 6, 8)):
        st = S.solve(precision, "bsr", rtol=1e-12, raise_on_fail=False, preconditioner="block_jacobi")
        assert st["stop_reason"] in (1, 3) and relerr(S.solution(), q_ref) <= ERR, precision
        vecs = 4 if slices <= 1280 else 2
        assert st["spmv_bytes"] == S.nnz // 4 * (4 * vb + 4) + 12 * slices + 8 + vecs * S.n_free * xb
    for h in (S, bc, K):
        h.close()
