"""The mixed-precision PCG over tagged records: every rows-per-thread class and the forms it hands over (eight
rows a thread, a slice beyond the LDS, the fenced exchange), tiny and ragged systems, and solves after solves in
one context, whose records must not be taken for this one's.  Each solution's true FP64 residual meets the
tolerance (x 1.01: it is summed in another order here)."""
import numpy as np
import pytest
import scipy.sparse as sp

import cases
from drops_amd import dhip as D

pytestmark = pytest.mark.gpu


def assembled(ctx, n, lc=None):
    m, phi = cases.c1_sphere(n)
    ctx.mesh(m)
    ctx.levelset(phi)
    ctx.assemble_p1(rhs_kind=D.RHS_3XY_MINUS_X3, lc=lc or (1.0, 1.0, m.h))
    g = ctx.csr()
    return sp.csr_matrix((g["comb"], g["colind"], g["rowptr"])), g["rhs"]


def check(ctx, M, b, tol, **kw):
    M = M.tocsr()
    M.sort_indices()
    A = ctx.csr_create(M.indptr, M.indices, M.data)
    x, it, res, ok = ctx.pcg(A, b, tol=tol, precision=D.FP32_IR, **kw)
    A.close()
    assert ok and res <= tol and np.linalg.norm(b - M @ x) <= 1.01 * tol * np.linalg.norm(b)
    return x, it


@pytest.mark.parametrize("rows", [0, 100, 512, 700, 1500, 2048, 3000])
def test_rows_per_block(ctx, rows):
    print(f"[gpu mixed pcg] {rows} rows per block", flush=True)
    M, b = assembled(ctx, 48)
    ctx.tune("pcg_rows_per_block", rows)
    try:
        x, it = check(ctx, M, b, 1e-8)
        assert np.array_equal(check(ctx, M, b, 1e-8)[0], x)
        ctx.tune("coherent_exchange", 0)
        y, it0 = check(ctx, M, b, 1e-8)
    finally:
        ctx.tune("pcg_rows_per_block", 0)
        ctx.tune("coherent_exchange", 2)
    assert np.linalg.norm(x - y) <= 1e-6 * np.linalg.norm(y) and it <= 1.2 * it0 + 20


@pytest.mark.parametrize("exchange", [0, 2])
def test_inner_solves_run_to_the_end(ctx, exchange):
    """An inner solve runs to 1e-4 whatever the caller's tolerance leaves to do: to 1e-6 two of them, which end at
    1e-8 and not below 1e-6 (twice that for what the FP32 recurrence's residual and the FP64 one differ by)."""
    print(f"[gpu mixed pcg] inner solves, exchange {exchange}", flush=True)
    ctx.tune("coherent_exchange", exchange)
    try:
        for n in (16, 48):
            M, b = assembled(ctx, n)
            x, _, res, ok = ctx.pcg(ctx.csr_create(M.indptr, M.indices, M.data), b, tol=1e-6, precision=D.FP32_IR)
            assert ok and res <= 2e-8
            assert np.linalg.norm(b - M @ x) <= 2.02e-8 * np.linalg.norm(b)
    finally:
        ctx.tune("coherent_exchange", 2)


def test_sizes_and_tolerances(ctx):
    print("[gpu mixed pcg] sizes", flush=True)
    rng = np.random.default_rng(2)
    for n in (1, 2, 63, 257, 513, 2999):
        M = sp.diags([np.full(n, 4.0), np.full(n - 1, -1.0), np.full(n - 1, -1.0)], [0, 1, -1], format="csr")
        M = M + sp.diags(rng.uniform(0.1, 1.0, n))
        b = rng.normal(size=n)
        for tol in (1e-3, 1e-6, 1e-12):
            check(ctx, M, b, tol)
        check(ctx, M, b, 1e-8, x0=rng.normal(size=n))
    for n, tol in ((16, 1e-10), (33, 1e-6), (64, 1e-12)):
        M, b = assembled(ctx, n)
        check(ctx, M, b, tol)
    # rows longer than a block's LDS holds: the memory form
    M = sp.random(6000, 6000, density=0.02, random_state=3, format="csr")
    M = M + M.T + sp.diags(np.full(6000, 200.0))
    check(ctx, M, rng.normal(size=6000), 1e-8)


def ill_conditioned(rng):
    """A dense symmetric positive definite matrix with a condition number up to 1e8, half of them scaled by
    rows and columns over six decades, and a right-hand side."""
    n, k = int(rng.choice([8, 16, 40])), 10.0 ** rng.uniform(4, 8)
    Q, _ = np.linalg.qr(rng.normal(size=(n, n)))
    ev = np.exp(rng.uniform(0.0, np.log(k), n))
    A = (Q * ev) @ Q.T
    if rng.random() < 0.5:
        s = 10.0 ** rng.uniform(-3, 3, n)
        A = s[:, None] * A * s[None, :]
    A = (A + A.T) / 2
    return sp.csr_matrix(A), rng.normal(size=n) if rng.random() < 0.5 else A @ rng.normal(size=n)


@pytest.mark.parametrize("seed", [11, 12])
def test_condition_beyond_fp32(ctx, seed):
    """Where the single-reduction recurrences lose the step length in FP32 the solve goes on in the two-reduction
    form: what converges there (the fenced exchange runs it from the start) converges, to the same tolerance and
    within twice the iterations and two passes of 400.  Dense matrices, and operators without stabilisation."""
    print(f"[gpu mixed pcg] condition numbers beyond FP32, seed {seed}", flush=True)
    rng = np.random.default_rng(seed)
    systems = [ill_conditioned(rng) for _ in range(80)]
    systems += [assembled(ctx, 32, lc) for lc in ((1.0, 1.0, 0.0), (1.0, 0.0, 0.0), (1e-3, 1.0, 0.0))]
    worse = converged = 0
    for M, b in systems:
        A = ctx.csr_create(M.indptr, M.indices, M.data)
        got = {}
        for exchange in (0, 2):
            ctx.tune("coherent_exchange", exchange)
            try:
                got[exchange] = ctx.pcg(A, b, tol=1e-8, max_iter=8000, precision=D.FP32_IR, raise_on_fail=False)
            finally:
                ctx.tune("coherent_exchange", 2)
        A.close()
        (x, it, _, ok), (_, it0, _, ok0) = got[2], got[0]
        assert np.all(np.isfinite(x)) or not ok0
        if ok:
            assert np.linalg.norm(b - M @ x) <= 1.01e-8 * np.linalg.norm(b)
        converged += ok0
        worse += bool(ok0 and (not ok or it > 2 * it0 + 800))
    assert converged >= 50 and worse == 0, (converged, worse)
