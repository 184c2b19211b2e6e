"""GPU parity of the batched solve (many uneven P1 problems in one launch) through the C ABI.

Bars: per problem the CSR pattern, the operator-combination values and the load vector bit-exact
against the oracle (the batch runs the single-problem per-item code); the FP32-inner/FP64-refined
solution with true relative residual <= 1.5e-8 and within 1e-6 of the oracle's FP64 solution
solved to 1e-13; graph replays bit-identical to the eager launch; a problem with an exact-zero
node reports the reference's error without disturbing the others."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg  # noqa: F401

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
    print("[gpu batch] graph replay, tuning keys", flush=True)
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
    # the launches have one geometry: the keys of other ones are accepted and change nothing, values out of
    # their ranges are refused
    for key, value, bad in (("batch_threads", 128, 100), ("batch_prepass", 1, 2), ("batch_split", 1, -1),
                            ("batch_solve_threads", 256, 128), ("batch_blocks_per_cu", 1, 9)):
        ctx.tune(key, value)
        with pytest.raises(D.DhipError):
            ctx.tune(key, bad)
    b.solve(tol=1e-8)
    for p in range(len(meshes)):
        assert np.array_equal(b.problem(p)["x"], ref[p]["x"])
    b.close()


def test_batch_inner_solves_halve_what_is_left(ctx):
    """The last inner solve runs to half of what is left to the tolerance: two solves to 1e-8, every problem at 5e-9
    by the FP32 recurrence's residual (1.2 times that for what the FP64 one differs by), and the solutions as near to the
    exact ones."""
    print("[gpu batch] inner solves", flush=True)
    meshes, phi, off = small_set(24, seed=9)
    b = make_batch(ctx, meshes, phi, off)
    b.solve(tol=1e-8)
    st = b.stats()
    assert np.all(st["status"] == D.OK) and np.all(st["outer"] == 2) and np.all(st["resid"] <= 6e-9), st["resid"]
    for p in range(len(meshes)):
        g = b.problem(p)
        x = sp.linalg.spsolve(sp.csc_matrix((g["comb"], g["colind"], g["rowptr"])), g["rhs"])
        assert np.linalg.norm(g["x"] - x) <= 1.2e-8 * np.linalg.norm(x), p
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


# cells across, radius and shift (in cells over 1, 1.7, 2.3) of spheres with exactly 512 k and 512 k + 1 rows: the last
# of one size class of the batched PCG and the first of the next
CLASS_EDGES = {
    1: ((10, 1.67341, 0.557), (10, 1.66762, 0.365)), 2: ((14, 1.67358, 0.289), (14, 1.67212, 0.372)),
    3: ((17, 1.69165, 0.597), (17, 1.68816, 0.629)), 4: ((20, 1.65799, 0.602), (20, 1.65644, 0.377)),
    5: ((22, 1.68232, 0.281), (22, 1.68174, 0.39)), 6: ((24, 1.69104, 0.707), (24, 1.69096, 0.654)),
    7: ((26, 1.68612, 0.479), (26, 1.69112, 0.248)), 8: ((28, 1.67421, 0.09), (28, 1.68274, 0.354)),
    9: ((30, 1.65832, 0.683), (30, 1.65293, 0.289)), 11: ((33, 1.66738, 0.714), (33, 1.66788, 0.754)),
    13: ((36, 1.66251, 0.138), (36, 1.66099, 0.623)), 15: ((38, 1.69258, 0.758), (38, 1.69242, 0.857)),
    17: ((41, 1.66852, 0.086), (41, 1.66742, 0.324)), 19: ((43, 1.68174, 0.543), (43, 1.68142, 0.516)),
    28: ((52, 1.68864, 0.536), (52, 1.68804, 0.732)), 76: ((86, 1.68252, 0.535), (86, 1.68201, 0.251))}


def test_batch_size_classes(ctx):
    """The last and the first row count of every size class of the batched PCG, alone and together: the system
    of dhip_assemble_p1 bit for bit, a true residual within the tolerance (1.01: it is summed in another order
    here), replays bit-identical."""
    print("[gpu batch] size classes", flush=True)
    rows = [512 * k + i for k in CLASS_EDGES for i in (0, 1)]
    shape = [e for k in CLASS_EDGES for e in CLASS_EDGES[k]]
    meshes = [KuhnMesh.box(-2.0, 2.0, n, shift=tuple(f / n * np.array([1.0, 1.7, 2.3]))) for n, _, f in shape]
    phis = [m.sample_p2(sphere(radius=r)) for m, (_, r, _) in zip(meshes, shape)]
    off = np.concatenate([[0], np.cumsum([p.size for p in phis])[:-1]]).astype(np.int64)
    b = make_batch(ctx, meshes, np.concatenate([p.ravel() for p in phis]), off)
    b.solve(tol=1e-8)
    st = b.stats()
    assert np.all(st["status"] == D.OK)
    assert 12 * st["nnz"].max() > 4 << 20   # read back below in more than one piece of pinned memory
    assert st["ndof"].tolist() == rows
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
        assert np.linalg.norm(g["rhs"] - A @ g["x"]) <= 1.01e-8 * np.linalg.norm(g["rhs"]), (p, rows[p])
    for graph in (False, True, True):
        b.solve(tol=1e-8, graph=graph)
        for p in range(len(meshes)):
            assert np.array_equal(b.problem(p)["x"], first[p]), p
    b.close()
