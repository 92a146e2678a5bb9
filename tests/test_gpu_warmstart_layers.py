"""The network's kernels at the edges of their tiles: channel counts that fill
no block of 32 or 64, planes smaller than a tile, one image and several."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NETS = [(1, 16, 16, 1), (2, 16, 16, 3), (2, 48, 32, 1), (3, 32, 32, 2), (2, 80, 16, 1),
        (3, 16, 64, 1)]


@pytest.mark.parametrize("L,base,S,batch", NETS)
def test_output_and_gradients(gpu_ready, L, base, S, batch):
    """Activations and masked gradients are rounded to bf16 at the same points on
    both sides, in FP64 between them on the oracle's.  A sum that differs in the
    last bit flips a rounding now and then, a change of at most 2^-8 of that
    value: relative to the norm less than 2^-8 a layer even if all flipped, so
    (4 L + 1) 2^-8 over the layers on the way; about 3e-2 at L = 2, the bound
    taken for all."""
    import oracle as O
    from iskra_amd import Context, _lib, warmstart as W
    rng = np.random.default_rng(100 * base + S)
    p = np.concatenate([rng.standard_normal(n) * np.sqrt(2.0 / (9 * cin))
                        for _, n, cin, _ in W.layer_slices(L, base)]).astype(np.float32)
    x = rng.standard_normal((batch, S, S)).astype(np.float32)
    t = rng.standard_normal((batch, S, S)).astype(np.float32)
    ctx = Context(0)
    net = _lib.WarmStart(ctx, levels=L, base=base, side=S, max_batch=batch)
    net.set_params(p)
    out = net.forward(x)
    loss, g = net.backward(x, t)
    loss2, g2 = net.backward(x, t)
    assert loss == loss2 and np.array_equal(g, g2)
    oref, lref, gref = O.ws_run(L, base, p.astype(np.float64), x.astype(np.float64),
                                t.astype(np.float64), round_bf16=True)

    def err(a, b):
        return np.linalg.norm(a - b) / np.linalg.norm(b)

    assert err(out.ravel(), np.asarray(oref).ravel()) < 3e-2
    assert loss == pytest.approx(lref, rel=1e-3)
    for k, (off, n, cin, cout) in enumerate(W.layer_slices(L, base)):
        e = err(g[off:off + n], gref[off:off + n])
        print("layer", k, cin, cout, e)
        assert e < 3e-2, (k, cin, cout, e)
    net.close()
    ctx.close()
