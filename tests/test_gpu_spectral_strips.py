"""The spectral solve in strips (grids of up to 64 x 128 interior nodes) at the edges
of its strips and blocks, and the sizes just beyond, which take four products."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (1, 128), (64, 1), (64, 128), (63, 14), (17, 15), (48, 28), (16, 16), (33, 127),
         (64, 129), (65, 64)]


def _reference(rho, ring, mx, my):
    """FP64 five-point solve, dx = eps0 = 1, ring: node array of wall values."""
    tx = sp.diags([-1.0, 2.0, -1.0], [-1, 0, 1], shape=(mx, mx))
    ty = sp.diags([-1.0, 2.0, -1.0], [-1, 0, 1], shape=(my, my))
    A = sp.kron(sp.eye(my), tx) + sp.kron(ty, sp.eye(mx))
    f = rho[1:-1, 1:-1].copy()
    f[:, 0] += ring[1:-1, 0]
    f[:, -1] += ring[1:-1, -1]
    f[0] += ring[0, 1:-1]
    f[-1] += ring[-1, 1:-1]
    out = ring.copy()
    out[1:-1, 1:-1] = spl.spsolve(A.tocsc(), f.ravel()).reshape(my, mx)
    return out


def _context(mx, my, rtol):
    from iskra_amd import Context, _lib as L
    ctx = Context(0)
    ctx.grid(2, (mx + 2, my + 2), (1.0, 1.0))
    tags = np.zeros((my + 2, mx + 2), np.int8)
    tags[0], tags[-1], tags[1:-1, 0], tags[1:-1, -1] = 1, 2, 3, 4
    ctx.poisson(L.POISSON_SPECTRAL, 1.0, tags, rtol=rtol)
    ring = np.zeros(tags.shape)
    for t, v in ((1, 0.5), (2, -1.25), (3, 2.0), (4, 0.125)):
        ctx.tag_value(t, v)
        ring[tags == t] = v
    return ctx, ring


@pytest.mark.parametrize("mx,my", SIZES)
def test_solve_and_field(gpu_ready, mx, my):
    """phi to round-off times the operator's condition, (n / 2)^2 at the most; in
    the time loop phi is that of the solve from the same density, and E its central
    differences, rounded once."""
    from iskra_amd import _lib as L
    ctx, ring = _context(mx, my, 1e-9)
    rng = np.random.default_rng(1000 * mx + my)
    rho = rng.standard_normal((my + 2, mx + 2))
    ctx.set_field(L.F_RHO, rho)
    it, rr = ctx.solve()
    assert it == 1 and rr <= 1e-12
    phi = ctx.field(L.F_PHI).reshape(ring.shape)
    ref = _reference(rho, ring, mx, my)
    cond = (max(mx, my) + 2) ** 2 / 4.0
    assert np.abs(phi - ref).max() <= 2.0 ** -52 * 8 * cond * np.abs(ref).max()
    assert np.array_equal(phi[[0, -1]], ring[[0, -1]])
    assert np.array_equal(phi[:, [0, -1]], ring[:, [0, -1]])
    s = ctx.species(-1.0, 1.0, 1.0, 2000, track_ids=False)
    ctx.boundary(s, [L.BND_DISCARD, L.BND_DISCARD])
    ctx.sample_maxwellian(s, 1500, [mx + 1.0, my + 1.0], [1e-3] * 3, seed=3, stream=0)
    ctx.step(1e-3, 3)
    phi = ctx.field(L.F_PHI).reshape(ring.shape)
    E = [np.asarray(ctx.field(f), np.float32).reshape(ring.shape) for f in (L.F_EX, L.F_EY)]
    ex = np.empty_like(phi)
    ey = np.empty_like(phi)
    ex[:, 1:-1] = (phi[:, :-2] - phi[:, 2:]) / 2.0
    ex[:, 0], ex[:, -1] = phi[:, 0] - phi[:, 1], phi[:, -2] - phi[:, -1]
    ey[1:-1] = (phi[:-2] - phi[2:]) / 2.0
    ey[0], ey[-1] = phi[0] - phi[1], phi[-2] - phi[-1]
    assert np.array_equal(E[0], ex.astype(np.float32))
    assert np.array_equal(E[1], ey.astype(np.float32))
    ctx.solve()
    assert np.array_equal(phi, ctx.field(L.F_PHI).reshape(ring.shape))
    ctx.close()


@pytest.mark.parametrize("mx,my", [(17, 15), (64, 128), (64, 129)])
def test_a_pass_short_of_rtol_is_corrected(gpu_ready, mx, my):
    """rtol below a pass's round-off: corrections follow, and where they do not
    reach it either the solve says so."""
    from iskra_amd import _lib as L
    ctx, ring = _context(mx, my, 1e-19)
    rho = np.random.default_rng(mx).standard_normal(ring.shape)
    ctx.set_field(L.F_RHO, rho)
    with pytest.raises(L.IskraError) as ex:
        ctx.solve()
    assert ex.value.code == L.E_CONVERGE
    ref = _reference(rho, ring, mx, my)
    cond = (max(mx, my) + 2) ** 2 / 4.0
    phi = ctx.field(L.F_PHI).reshape(ring.shape)
    assert np.abs(phi - ref).max() <= 2.0 ** -52 * 8 * cond * np.abs(ref).max()
    ctx.close()
