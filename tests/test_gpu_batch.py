"""GPU parity of the batched solve (many uneven P1 problems in one launch) through the C ABI.

Bars: per problem the CSR pattern, the operator-combination values and the load vector bit-exact
against the oracle (the batch runs the single-problem per-item code); the FP32-inner/FP64-refined
solution with true relative residual <= 1.5e-8 and within 1e-6 of the oracle's FP64 solution
solved to 1e-13; graph replays bit-identical to the eager launch; a problem with an exact-zero
node reports the reference's error without disturbing the others."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle as O
from drops_amd import batch as BT
from drops_amd import dhip as D
from drops_amd.mesh import KuhnMesh, sphere

pytestmark = pytest.mark.gpu

COEF = (1.0, 1.0, 1.0)


def lc_of(m):
    return (1.0, 1.0, m.h)


def small_set(nprob=24, seed=3):
    probs = BT.make_problems(nprob, seed, nmin=8, nmax=20)
    phi, off = BT.level_sets(probs)
    meshes = [p[0] for p in probs]
    return meshes, phi, off


def make_batch(ctx, meshes, phi, off, **kw):
    # each problem solves mass + LB + h * stabilisation with its own mesh size
    return ctx.batch(meshes, phi, off, coef=COEF, rhs_kind=D.RHS_3XY_MINUS_X3, **kw)


def test_batch_matches_oracle(ctx):
    print("[gpu batch] 24 problems, eager", flush=True)
    meshes, phi, off = small_set()
    b = make_batch(ctx, meshes, phi, off)
    b.solve(tol=1e-8)
    st = b.stats()
    assert np.all(st["status"] == D.OK), st["status"]
    assert np.all(st["resid"] <= 1e-8)
    assert len(set(st["ndof"].tolist())) > 5   # uneven sizes
    for p, m in enumerate(meshes):
        g = b.problem(p)
        sz = int(np.prod(m.halfgrid_shape))
        mm = KuhnMesh(m.orig, m.e, m.n)
        check_problem_lc(mm, phi[off[p]:off[p] + sz].reshape(m.halfgrid_shape), g, lc_of(m))
    b.close()


def check_problem_lc(m, phi, g, lc, tol=1e-8):
    om = O.make_mesh(m.orig, m.e, m.n)
    dof, nd = O.number_p1if(om, phi)
    r = O.assemble_p1(om, phi, dof, nd, coef=COEF, rhs_kind=O.RHS_3XY_MINUS_X3)
    comb = (1.0 * (lc[0] * r["mass"] + lc[1] * r["lb"])) + lc[2] * r["stab"]
    assert np.array_equal(g["rowptr"].astype(np.int64), r["rowptr"])
    assert np.array_equal(g["colind"], r["colind"])
    assert np.array_equal(g["comb"], comb)
    assert np.array_equal(g["rhs"], r["rhs"])
    A = sp.csr_matrix((comb, r["colind"], r["rowptr"]), shape=(nd, nd))
    b = r["rhs"]
    assert np.linalg.norm(b - A @ g["x"]) <= 1.5 * tol * np.linalg.norm(b)
    xo, it, res, ok = O.pcg_jacobi(r["rowptr"], r["colind"], comb, b, tol=1e-13, max_iter=100000)
    assert np.linalg.norm(g["x"] - xo) <= 1e-6 * np.linalg.norm(xo)


def test_batch_graph_replay_and_tiles(ctx):
    print("[gpu batch] graph replay, tile sizes", flush=True)
    meshes, phi, off = small_set(16, seed=5)
    b = make_batch(ctx, meshes, phi, off)
    b.solve(tol=1e-8)
    ref = [b.problem(p) for p in range(len(meshes))]
    ref_st = b.stats()
    for _ in range(3):
        b.solve(tol=1e-8, graph=True)
        st = b.stats()
        assert np.array_equal(st["iters"], ref_st["iters"])
        for p in range(len(meshes)):
            g = b.problem(p)
            assert np.array_equal(g["x"], ref[p]["x"])
    # other workgroup sizes: identical assembly, solutions to the same tolerance
    for threads in (128, 512):
        ctx.tune("batch_threads", threads)
        try:
            b.solve(tol=1e-8)
            st = b.stats()
            assert np.all(st["status"] == D.OK) and np.all(st["resid"] <= 1e-8)
            for p in range(len(meshes)):
                g = b.problem(p)
                assert np.array_equal(g["comb"], ref[p]["comb"])
                assert np.linalg.norm(g["x"] - ref[p]["x"]) <= 1e-6 * np.linalg.norm(ref[p]["x"])
        finally:
            ctx.tune("batch_threads", 256)
    # classification and local matrices by a grid-wide pre-pass instead of inside each problem's
    # workgroup: the same assembled systems, iteration counts and solutions bit for bit
    ctx.tune("batch_prepass", 1)
    try:
        for graph in (False, True):
            b.solve(tol=1e-8, graph=graph)
            st = b.stats()
            assert np.array_equal(st["iters"], ref_st["iters"]) and np.array_equal(st["ncut"], ref_st["ncut"])
            for p in range(len(meshes)):
                g = b.problem(p)
                for k in ("rowptr", "colind", "comb", "rhs", "x"):
                    assert np.array_equal(g[k], ref[p][k]), (p, k)
    finally:
        ctx.tune("batch_prepass", 0)
    # assembly launch and a separate PCG launch: with the same workgroup size bit for bit, with
    # 1024 threads per problem to the same tolerance
    ctx.tune("batch_split", 1)
    try:
        for sthreads in (256, 1024):
            ctx.tune("batch_solve_threads", sthreads)
            for graph in (False, True):
                b.solve(tol=1e-8, graph=graph)
                st = b.stats()
                assert np.all(st["status"] == D.OK) and np.all(st["resid"] <= 1e-8)
                for p in range(len(meshes)):
                    g = b.problem(p)
                    assert np.array_equal(g["comb"], ref[p]["comb"]) and np.array_equal(g["rhs"], ref[p]["rhs"])
                    if sthreads == 256:
                        assert np.array_equal(g["x"], ref[p]["x"]), p
                    else:
                        assert np.linalg.norm(g["x"] - ref[p]["x"]) <= 1e-6 * np.linalg.norm(ref[p]["x"])
    finally:
        ctx.tune("batch_split", 0)
        ctx.tune("batch_solve_threads", 1024)
    b.close()


def test_batch_inner_solves_run_to_the_end(ctx):
    """To 1e-6 every problem takes two inner solves of 1e-4, which end at 1e-8 (twice that for what the FP32
    recurrence's residual and the FP64 one differ by; 5e-8 for 42,796 rows, measured 3.3e-8)."""
    print("[gpu batch] inner solves", flush=True)
    meshes, phi, off = small_set(12, seed=9)
    big = KuhnMesh.box(-2.0, 2.0, 80, shift=tuple(5e-5 * np.array([1.0, 2.0, 3.0])))   # the form in memory
    pb = big.sample_p2(sphere(radius=1.9)).ravel()
    b = make_batch(ctx, meshes + [big], np.concatenate([phi, pb]), np.concatenate([off, [phi.size]]))
    b.solve(tol=1e-6)
    st = b.stats()
    assert np.all(st["status"] == D.OK) and np.all(st["outer"] == 2) and np.all(st["resid"][:-1] <= 2e-8), st["resid"]
    assert st["resid"][-1] <= 5e-8, st["resid"]
    b.close()


def test_batch_without_cut_tets(ctx):
    """Problems whose level set cuts nothing, among others and alone: converged with no unknowns, row pointers (0).
    The batch before leaves its memory behind."""
    print("[gpu batch] nothing cut", flush=True)
    meshes, phi, off = small_set(8, seed=13)
    empty = [KuhnMesh.box(-2.0, 2.0, n) for n in (6, 5, 9)]
    ep = [m.sample_p2(sphere(radius=9.0)).ravel() for m in empty]
    eo = np.concatenate([[0], np.cumsum([p.size for p in ep])[:-1]]).astype(np.int64)
    b = make_batch(ctx, meshes + empty, np.concatenate([phi] + ep), np.concatenate([off, eo + phi.size]))
    b.solve(tol=1e-8)
    assert np.all(b.stats()["status"] == D.OK) and np.all(b.stats()["ndof"][:8] > 0)
    assert all(b.problem(p)["rowptr"].tolist() == [0] for p in range(8, 11))
    b.close()
    b = make_batch(ctx, empty, np.concatenate(ep), eo)
    for graph in (False, True, True):
        b.solve(tol=1e-8, graph=graph)
        st = b.stats()
        assert np.all(st["status"] == D.OK)
        for k in ("ncut", "ndof", "nnz", "iters"):
            assert np.all(st[k] == 0)
        for p in range(3):
            assert b.problem(p)["rowptr"].tolist() == [0]
    b.close()


def test_batch_zero_node_problem_isolated(ctx):
    print("[gpu batch] exact-zero node in one problem", flush=True)
    meshes, phi, off = small_set(4, seed=7)
    bad = KuhnMesh.box(-2.0, 2.0, 8)   # the unit sphere passes through grid vertices (1, 0, 0), ...
    pb = bad.sample_p2(sphere()).ravel()
    meshes = meshes + [bad]
    off = np.concatenate([off, [phi.size]])
    phi = np.concatenate([phi, pb])
    b = make_batch(ctx, meshes, phi, off)
    b.solve(tol=1e-8)
    st = b.stats()
    assert st["status"][-1] == D.E_ZERO_NODE
    assert np.all(st["status"][:-1] == D.OK)
    with pytest.raises(D.DhipError):
        b.problem(len(meshes) - 1)
    b.close()


# rows per problem from 1 to 27 per thread of the solver's 512, beyond its register classes and beyond its LDS:
# (cells across, radius) of spheres, about 1.86 (radius n)^2 rows
CLASS_SIZES = [(16, 1.0), (22, 1.0), (27, 1.0), (31, 1.0), (35, 1.0), (39, 1.0), (43, 1.0), (46, 1.0), (49, 1.0),
               (53, 1.0), (58, 1.0), (63, 1.0), (67, 1.0), (71, 1.0), (80, 1.0), (64, 1.5), (80, 1.9)]


def test_batch_size_classes(ctx):
    """One problem of every size class of the batched PCG, alone and together: the system of
    dhip_assemble_p1 bit for bit, a true residual within the tolerance (1.5: the FP64 residual is summed in
    another order here), replays bit-identical."""
    print("[gpu batch] size classes", flush=True)
    meshes = [KuhnMesh.box(-2.0, 2.0, n, shift=tuple(4e-3 / n * np.array([1.0, 2.0, 3.0]))) for n, _ in CLASS_SIZES]
    phis = [m.sample_p2(sphere(radius=r)) for m, (_, r) in zip(meshes, CLASS_SIZES)]
    off = np.concatenate([[0], np.cumsum([p.size for p in phis])[:-1]]).astype(np.int64)
    b = make_batch(ctx, meshes, np.concatenate([p.ravel() for p in phis]), off)
    b.solve(tol=1e-8)
    st = b.stats()
    assert np.all(st["status"] == D.OK)
    assert 12 * st["nnz"].max() > 5 << 20   # read back below in more than one piece of pinned memory
    slots = -(-st["ndof"] // 512)
    assert {1, 2, 3, 4, 5, 6, 7, 8, 9} <= set(slots.tolist()) and slots.max() > 76 and 28 < np.sort(slots)[-2] <= 76
    first = []
    for p, m in enumerate(meshes):
        g = b.problem(p)
        first.append(g["x"])
        ctx.mesh(m)
        ctx.levelset(phis[p])
        ctx.assemble_p1(coef=COEF, rhs_kind=D.RHS_3XY_MINUS_X3, lc=lc_of(m))
        ref = ctx.csr()
        for k in ("rowptr", "colind", "comb", "rhs"):
            assert np.array_equal(g[k], ref[k]), (p, k)
        A = sp.csr_matrix((g["comb"], g["colind"], g["rowptr"]))
        assert np.linalg.norm(g["rhs"] - A @ g["x"]) <= 1.5e-8 * np.linalg.norm(g["rhs"]), (p, slots[p])
    for graph in (False, True, True):
        b.solve(tol=1e-8, graph=graph)
        for p in range(len(meshes)):
            assert np.array_equal(b.problem(p)["x"], first[p]), p
    b.close()
