"""Ionisation products of one MCC call: every product sits at its parent's
place, ids follow the parents' ids (electrons next + rank, the R ions of a
product next + rank R + r), headers count them, for no product, a handful,
and more than one work-group's sort holds, stored in another order than the
ids'."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ME = 9.1093837015e-31
MI = 40 * 1.66053906660e-27


@pytest.mark.parametrize("n,prob,ratio", [(40, 0.0, 1), (1, 0.3, 1), (700, 0.05, 2),
                                          (20000, 0.3, 1), (16385, 0.32, 3), (200000, 0.32, 2)])
def test_products(gpu_ready, n, prob, ratio):
    from iskra_amd import Context, _lib as L
    cells = 300
    rng = np.random.default_rng(n)
    ctx = Context()
    try:
        ctx.grid(1, (cells + 1,), (1e-4,))
        ctx.rng(7)
        e = ctx.species(-1.6e-19, ME, 6.0, 2 * n + 10, track_ids=True)
        i = ctx.species(1.6e-19, MI, 6.0 / ratio, ratio * n + 10, track_ids=True)
        cell = rng.integers(0, cells, n).astype(np.int32)
        ox = (np.arange(n) / (n + 1.0)).astype(np.float32)  # tells the parents apart
        v = rng.normal(0.0, 3e6, (3, n)).astype(np.float32)
        ids = rng.permutation(3 * n)[:n].astype(np.uint32)
        ctx.set_state(e, cell, ox, None, v[0], v[1], v[2], ids)
        sig = 1e-19
        # max_P = 1 - exp(-n sigma g_max dt), g_max at the table's last energy
        g = np.sqrt(2 * 1000.0 * 1.60217646e-19 / ME)
        dt = 1e-11
        dens = -np.log1p(-prob) / (sig * g * dt)
        m = ctx.mcc(e, [L.COLL_IONIZATION], [0.0], [([0.0, 1000.0], [sig, sig])], ion=i,
                    target_m=MI)
        ctx.set_field(L.F_TARGET, np.full(cells + 1, dens), index=m)
        before = ctx.get_state(e)
        ev = ctx.mcc_run(m, dt)
        se, si = ctx.get_state(e), ctx.get_state(i)
    finally:
        ctx.close()
    p = int(ev[0])
    assert (p == 0) == (prob == 0.0) or n == 1
    # threshold 0: every collision ionises
    assert len(se["cell"]) == n + p and len(si["cell"]) == ratio * p
    if n == 200000:
        assert p > 8192
    parent = dict(zip(zip(before["cell"], before["ox"]), before["id"]))
    pe = np.array([parent[k] for k in zip(se["cell"][n:], se["ox"][n:])], dtype=np.int64)
    assert len(set(pe)) == p
    rank = np.empty(p, np.int64)
    rank[np.argsort(pe)] = np.arange(p)
    nxt = int(ids.max()) + 1
    assert np.array_equal(se["id"][n:], nxt + rank)
    # particle order of the products, and the ions behind them
    pos = {k: q for q, k in enumerate(before["id"])}
    assert np.all(np.diff([pos[k] for k in pe]) > 0)
    pi = np.array([parent[k] for k in zip(si["cell"], si["ox"])], dtype=np.int64)
    assert np.array_equal(pi, np.repeat(pe, ratio))
    assert np.array_equal(si["id"], np.repeat(rank * ratio, ratio) + np.tile(np.arange(ratio), p))
