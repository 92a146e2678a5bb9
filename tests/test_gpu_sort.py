"""The counting sort's order against numpy's stable argsort of the same keys
(exact: the stable order by a key is unique), at the edges of its strips and
rounds, with discarded particles, and over each scan variant: one bin group
scanned by one work-group, several groups, strips whose columns fit a thread's
registers and more, an exact sort in one pass and in two."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,cells,tile,n", [
    (1, 64, 64, 1), (1, 64, 64, 63), (1, 500, 32, 257), (1, 1024, 16, 70001),
    (2, (24, 40), 8, 0), (2, (24, 40), 8, 255), (2, (24, 40), 8, 256), (2, (65, 31), 8, 8193),
    (2, (64, 64), 8, 40000),        # 4096 cells in one exact pass
    (2, (200, 130), 8, 30011),      # 27,200 cells: by cell, then by tile
    (2, (64, 64), 2, 5000),         # 1024 tiles of 4 cells
    (1, 500, 32, 700001), (2, (24, 40), 8, 1023 * 1024 + 1),  # strips counted by four waves
    (2, (720, 720), 8, 300007),     # 8100 tiles: 8 bins a thread of the bin scan
])
@pytest.mark.parametrize("ids", [True, False])
def test_sort_order(gpu_ready, dim, cells, tile, n, ids):
    from iskra_amd import Context
    nc = (cells,) if dim == 1 else cells
    rng = np.random.default_rng(n + tile)
    i = rng.integers(0, nc[0], n).astype(np.int32)
    j = rng.integers(0, nc[1], n).astype(np.int32) if dim == 2 else np.zeros(n, np.int32)
    cell = i | (j << 16)
    cell[rng.random(n) < 0.1] = -1
    f = rng.random((5, n), dtype=np.float32)
    ident = rng.permutation(n).astype(np.uint32)
    ctx = Context()
    try:
        ctx.grid(dim, [c + 1 for c in nc], [1.0] * dim)
        ctx.tuning(tile=tile, margin=2 if tile > 2 else 1)
        s = ctx.species(1.0, 1.0, 1.0, n + 5, track_ids=ids)
        ctx.set_state(s, cell, f[0], f[1], f[2], f[3], f[4], ident)
        log2 = tile.bit_length() - 1
        ntx = -(-nc[0] // tile)
        key = (i >> log2) + ntx * (j >> log2)

        def check(key):
            live = np.flatnonzero(cell >= 0)
            order = live[np.argsort(key[live], kind="stable")]
            st = ctx.get_state(s)
            assert np.array_equal(st["cell"], cell[order])
            for k, a in (("ox", f[0]), ("vx", f[2]), ("vy", f[3]), ("vz", f[4])):
                assert np.array_equal(st[k], a[order]), k
            if dim == 2:
                assert np.array_equal(st["oy"], f[1][order])
            if ids:
                assert np.array_equal(st["id"], ident[order])

        check(key)
        ctx.sort(s, exact_cell=True)
        inner = (i & (tile - 1)) + ((j & (tile - 1)) << log2 if dim == 2 else 0)
        check(key.astype(np.int64) * tile ** dim + inner)
    finally:
        ctx.close()


def test_sort_more_strips_than_registers(gpu_ready):
    """Above 2048 strips of 8192 particles the column scans read the table twice."""
    from iskra_amd import Context
    n, cells, tile = 2049 * 8192 + 77, 500, 32
    rng = np.random.default_rng(1)
    i = rng.integers(0, cells, n, dtype=np.int32)
    cell = np.where(rng.random(n, dtype=np.float32) < 0.1, np.int32(-1), i)
    zero = np.zeros(n, np.float32)
    ctx = Context()
    try:
        ctx.grid(1, [cells + 1], [1.0])
        ctx.tuning(tile=tile)
        s = ctx.species(1.0, 1.0, 1.0, n + 5, track_ids=True)
        ctx.set_state(s, cell, zero, None, zero, zero, zero, np.arange(n, dtype=np.uint32))
        st = ctx.get_state(s)
    finally:
        ctx.close()
    live = np.flatnonzero(cell >= 0)
    order = live[np.argsort((i[live] // tile).astype(np.int16), kind="stable")]
    assert np.array_equal(st["id"], order) and np.array_equal(st["cell"], cell[order])
