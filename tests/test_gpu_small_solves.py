"""The one-work-group solvers at the edges of their shapes against a direct FP64
solve of the same rows: every number of nodes a thread (2, 4, 8, 19 and 26 of CG; 2, 4
and 10 of BiCGStab; `_npt` says which a grid takes), columns that end inside a
segment, edges without Dirichlet nodes, 1-D grids, the axial rows, the electrodes'
rows, and sizes past the largest, which go to the launches per iteration; the CG
iterates themselves; and what a failed solve leaves.

Bound: with relative residual rtol in the 2-norm the error is at most
cond(L) rtol |f| / |phi| <= cond(L) rtol (|L| |phi| >= |f|); cond is taken
from the dense matrix, or estimated in the 1-norm from a sparse factorisation."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl

pytestmark = pytest.mark.gpu

RTOL = 1e-12


CG = ((2, 1024), (4, 1024), (8, 1024), (19, 512), (26, 512))
BI = ((2, 1024), (4, 1024), (10, 512))


def _npt(nx, ny, shapes):
    """Nodes a thread: the first shape (nodes, threads) that gives every column segment
    a thread of its own; 0 for the launches per iteration."""
    return next((n for n, t in shapes if nx * -(-ny // n) <= t), 0)


def _lu(A):
    """Factorisation and 1-norm condition estimate."""
    lu = spl.splu(A.tocsc())
    inv = spl.LinearOperator(A.shape, matvec=lu.solve, rmatvec=lambda b: lu.solve(b, trans="T"))
    return lu, spl.onenormest(A) * spl.onenormest(inv)


def _rows(nx, ny, axial, az=1.0):
    """The five-point rows (a missing neighbour has no link), and the weights of f."""
    w = np.ones(nx)
    if axial:
        w = np.arange(nx, dtype=float)
        w[0], w[-1] = 0.5, nx - 1.5
    k = np.arange(nx * ny).reshape(ny, nx)
    cx = np.arange(nx - 1) + 0.5 if axial else np.ones(nx - 1)
    cy = w * az if axial else w
    links = [(k[:, :-1], k[:, 1:], np.broadcast_to(cx, (ny, nx - 1))),
             (k[:-1], k[1:], np.broadcast_to(cy, (ny - 1, nx)))]
    a, b, c = (np.concatenate([x[q].ravel() for x in links]) for q in range(3))
    n = nx * ny
    off = sp.coo_matrix((c, (a, b)), shape=(n, n))
    off = off + off.T
    return (sp.diags(np.asarray(off.sum(1)).ravel()) - off).tocsr(), np.tile(w, ny)


def _dense(nx, ny, tags, axial):
    A, w = _rows(nx, ny, axial)
    return A.toarray(), w


@pytest.mark.parametrize("nx,ny,axial", [
    (40, 1, False), (600, 1, False), (3, 3, False), (33, 17, False), (17, 33, False), (64, 32, False), (50, 45, False), (61, 60, False), (100, 25, True),
    (20, 61, True), (33, 130, True), (37, 77, False),
])
@pytest.mark.parametrize("walls", ["all", "left"])
def test_cg_one_work_group(gpu_ready, nx, ny, axial, walls):
    from iskra_amd import Context, _lib as L
    tags = np.zeros((ny, nx), np.int8)
    if axial:
        tags[:, -1] = 1
        if walls == "all":
            tags[0, :] = tags[-1, :] = 2
    else:
        tags[:, 0] = 1
        if walls == "all":
            tags[:, -1] = 2
            if ny > 1:
                tags[0, :] = tags[-1, :] = 2
    rng = np.random.default_rng(nx * ny)
    rho = rng.normal(size=nx * ny)
    ctx = Context()
    try:
        if axial:
            ctx.grid_axial((nx, ny), (1.0, 1.0))
        elif ny > 1:
            ctx.grid(2, (nx, ny), (1.0, 1.0))
        else:
            ctx.grid(1, (nx,), (1.0,))
        ctx.poisson(L.POISSON_PCG, 1.0, tags.ravel(), rtol=RTOL, max_iter=20000)
        for t, v in ((1, 3.0), (2, -1.0)):
            ctx.tag_value(t, v)
        ctx.set_field(L.F_RHO, rho)
        it, rr = ctx.solve(L.WARM_ZERO)
        assert 0 < it and rr <= RTOL
        phi = ctx.field(L.F_PHI)
    finally:
        ctx.close()
    A, w = _dense(nx, ny, tags, axial)
    t = tags.ravel()
    free = t == 0
    ref = np.where(t == 1, 3.0, np.where(t == 2, -1.0, 0.0))
    F = A[np.ix_(free, free)]
    ref[free] = np.linalg.solve(F, (rho * w)[free] - A[np.ix_(free, ~free)] @ ref[~free])
    err = np.linalg.norm((phi - ref)[free]) / np.linalg.norm(ref[free])
    assert err <= 2 * np.linalg.cond(F) * RTOL + 1e-14 * np.linalg.cond(F), err


@pytest.mark.parametrize("nx,ny,axial,npt", [
    (40, 61, False, 4), (61, 100, False, 8), (100, 90, False, 19), (60, 150, True, 19),
    (97, 129, True, 26), (98, 130, False, 26), (19, 600, False, 26), (103, 131, False, 0),
    (103, 131, True, 0), (257, 57, True, 0),
])
def test_cg_larger(gpu_ready, nx, ny, axial, npt):
    from iskra_amd import Context, _lib as L
    assert _npt(nx, ny, CG) == npt
    tags = np.zeros((ny, nx), np.int8)
    tags[:, -1] = 1
    tags[0, :] = 2
    if not axial:
        tags[ny // 3:ny // 2, nx // 2] = 1  # nodes inside the grid
    rho = np.random.default_rng(nx + ny).normal(size=nx * ny)
    ctx = Context()
    try:
        if axial:
            ctx.grid_axial((nx, ny), (1.0, 0.8))
        else:
            ctx.grid(2, (nx, ny), (1.0, 1.0))
        ctx.poisson(L.POISSON_PCG, 1.0, tags.ravel(), rtol=RTOL, max_iter=20000)
        for t, v in ((1, 3.0), (2, -1.0)):
            ctx.tag_value(t, v)
        ctx.set_field(L.F_RHO, rho)
        it, rr = ctx.solve(L.WARM_ZERO)
        assert 0 < it and rr <= RTOL
        phi = ctx.field(L.F_PHI)
    finally:
        ctx.close()
    A, w = _rows(nx, ny, axial, 1.0 / 0.8 ** 2)
    t = tags.ravel()
    free = t == 0
    ref = np.where(t == 1, 3.0, np.where(t == 2, -1.0, 0.0))
    assert np.array_equal(phi[~free], ref[~free])
    lu, cond = _lu(A[free][:, free])
    ref[free] = lu.solve((rho * w)[free] - A[free][:, ~free] @ ref[~free])
    err = np.linalg.norm((phi - ref)[free]) / np.linalg.norm(ref[free])
    assert err <= 2 * cond * RTOL + 1e-14 * cond and err <= 1e-5, (err, cond)


@pytest.mark.parametrize("nx,ny,axial", [(9, 14, False), (40, 1, False), (33, 40, True),
                                         (97, 129, True)])
def test_cg_iterates(gpu_ready, nx, ny, axial):
    """The iterates themselves, restated: z is the FP32 rounding of the FP64 r /
    diag, p is FP32, everything else FP64.  After a few iterations the sums' order
    leaves about 1e-14; z from FP32 operands would leave 1e-8."""
    from iskra_amd import Context, IskraError, _lib as L
    its = 6
    tags = np.zeros((ny, nx), np.int8)
    tags[:, -1] = 1
    rng = np.random.default_rng(nx * ny + 1)
    rho = rng.normal(size=nx * ny)
    ctx = Context()
    try:
        if axial:
            ctx.grid_axial((nx, ny), (1.0, 0.7))
        elif ny > 1:
            ctx.grid(2, (nx, ny), (1.0, 1.0))
        else:
            ctx.grid(1, (nx,), (1.0,))
        ctx.poisson(L.POISSON_PCG, 1.0, tags.ravel(), rtol=RTOL, max_iter=its)
        ctx.tag_value(1, 3.0)
        ctx.set_field(L.F_RHO, rho)
        with pytest.raises(IskraError) as ex:
            ctx.solve(L.WARM_ZERO)
        assert ex.value.code == L.E_CONVERGE
        phi = ctx.field(L.F_PHI)
    finally:
        ctx.close()
    A, w = _rows(nx, ny, axial, 1.0 / 0.7 ** 2)
    free = tags.ravel() == 0
    diag = A.diagonal()
    x = np.where(free, 0.0, 3.0)
    r = np.where(free, rho * w - A @ x, 0.0)
    z = (r / diag).astype(np.float32)
    p, beta = np.zeros(nx * ny, np.float32), np.float32(0)
    for _ in range(its):
        rz = r @ z.astype(np.float64)
        p = (np.float64(beta) * p + z).astype(np.float32)
        Ap = np.where(free, A @ p.astype(np.float64), 0.0)
        alpha = rz / (p.astype(np.float64) @ Ap)
        x = x + alpha * p
        r = r - alpha * Ap
        z = (r / diag).astype(np.float32)
        beta = np.float32(r @ z.astype(np.float64) / rz)
    assert np.abs(phi - x).max() <= 1e-11 * np.abs(x).max(), np.abs(phi - x).max()


@pytest.mark.parametrize("n,nx", [(11, 11), (21, 29), (45, 45), (49, 63), (65, 65), (75, 75)])
def test_bicgstab_electrodes(gpu_ready, n, nx):
    """Floating rows on the left wall and a fixed node: the device's potential is
    that of the reference's rows (as restated by the oracle) at every number of
    nodes a thread and by launches above 5000 nodes."""
    from iskra_amd import Context, _lib as L
    from oracle import surfaces as S
    assert _npt(nx, n, BI) == {11: 2, 21: 2, 45: 4, 49: 4, 65: 10, 75: 0}[n]
    dh = 0.1
    b = np.zeros((nx, n), np.int8)
    b[0, 1:n - 1] = 1
    b[nx - 1, n // 3:2 * n // 3] = 2
    b[nx - 2, 0] = b[nx - 2, n - 1] = 3
    flat = lambda m: np.ascontiguousarray(m.T).ravel()  # noqa: E731
    ctx = Context()
    try:
        ctx.grid(2, (nx, n), (dh, dh))
        ctx.poisson(L.POISSON_PCG, 8.854e-12, None, rtol=RTOL, max_iter=20000)
        ctx.electrode(flat(b == 1), fixed=False, sigma=1e-9)
        ctx.electrode(flat(b == 2), fixed=False, sigma=-2e-10)
        ctx.electrode(flat(b == 3), fixed=True, phi=2.0)
        rho = np.random.default_rng(n).normal(0.0, 1e-9, nx * n)
        ctx.set_field(L.F_RHO, rho)
        it, rr = ctx.solve(L.WARM_ZERO)
        phi = ctx.field(L.F_PHI)
        assert rr <= RTOL
        # from the solution the solve has nothing left to do
        it2, rr2 = ctx.solve(L.WARM_PREV)
        assert it2 <= 2 and rr2 <= RTOL
        assert np.abs(ctx.field(L.F_PHI) - phi).max() <= 1e-6 * np.abs(phi).max()
    finally:
        ctx.close()
    A, rhs, rdof, _ = S.electrode_system(nx, n, dh, dh, fixed=[(b == 3, 2.0)],
                                         floating=[(b == 1, 1e-9), (b == 2, -2e-10)])
    if nx * n > 1000:
        nn = nx * n
        rhs = rhs.copy()
        rhs[:nn][rdof] = -rho[rdof] / 8.854e-12
        lu, cond = _lu(sp.csr_matrix(A[:nn, :nn] * dh ** 2))
        ref = lu.solve((rhs[:nn] - A[:nn, nn:] @ rhs[nn:]) * dh ** 2)
        assert np.abs(phi - ref).max() <= 2 * cond * RTOL * np.abs(ref).max(), cond
        assert np.abs(phi - ref).max() <= 1e-6 * np.abs(ref).max()
        return
    ref = S.electrode_potential(A, rhs, rdof, rho, 8.854e-12)
    # cond of these rows is below 1e4 (a Laplacian of < 1000 nodes)
    assert np.abs(phi - ref).max() <= 1e4 * 2 * RTOL * np.abs(ref).max()


@pytest.mark.parametrize("electrodes", [False, True])
def test_failed_solve_leaves_E(gpu_ready, electrodes):
    """A step whose solve does not converge raises, and E stays what it was."""
    from iskra_amd import Context, IskraError, _lib as L
    nx, ny = 33, 21
    tags = np.zeros((ny, nx), np.int8)
    tags[:, 0] = 1
    ctx = Context()
    try:
        ctx.grid(2, (nx, ny), (0.1, 0.1))
        sid = ctx.species(-1.0, 1.0, 1.0, 16, track_ids=False)
        ctx.upload(sid, np.full((4, 2), 1.0), np.zeros((4, 3)))
        E = []
        for max_iter in (5000, 2):
            ctx.poisson(L.POISSON_PCG, 1.0, None if electrodes else tags.ravel(), rtol=1e-10,
                        max_iter=max_iter)
            if electrodes:
                ctx.electrode(tags.ravel() == 1, fixed=True, phi=3.0)
                b = np.zeros((ny, nx), bool)
                b[5:15, -1] = True
                ctx.electrode(b.ravel(), fixed=False, sigma=0.5)
            else:
                ctx.tag_value(1, 3.0)
            if max_iter > 2:
                ctx.deposit()
                ctx.solve(L.WARM_ZERO)
                ctx.efield()
            else:
                ctx.set_field(L.F_PHI, np.zeros(nx * ny))
                with pytest.raises(IskraError) as ex:
                    ctx.step(1e-3)
                assert ex.value.code == L.E_CONVERGE
            E.append((ctx.field(L.F_EX), ctx.field(L.F_EY)))
        assert np.abs(E[0][0]).max() > 0
        assert np.array_equal(E[0][0], E[1][0]) and np.array_equal(E[0][1], E[1][1])
    finally:
        ctx.close()
