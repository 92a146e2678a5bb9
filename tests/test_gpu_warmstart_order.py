"""The order in which the network's kernels add up products is part of their
results (a different one ends a training run in another network), so it follows
from a layer's shape and batch alone, whatever tile computes it:

 convolutions and input gradients, k = tap * Cin + ci in blocks of 32: blocks of 32
   channels with their 9 taps in order, or all blocks by k (`_chunk_major`);
 weight gradients: blocks of 32 consecutive pixels; chunks of 64-pixel segments
   are summed by themselves and then in order (`_chunks`).

Every sum here has at most one nonzero product a block, +-2^40 and small powers
of two: a partial sum of 2^40 swallows the small ones before it (and RN(2^40 + s) =
2^40), so the result tells the order exactly, and it is compared exactly."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BIG = 2.0 ** 40


def _chunk_major(npix, side, cin, cout):
    px, most = 64, -1
    for ct, bp in ((64, 256), (32, 256), (16, 256), (64, 64), (32, 64), (16, 64)):
        if cout % ct or npix % bp:
            continue
        nb = npix // bp * (cout // ct)
        if nb > most:
            px, most = bp, nb
        if nb >= 256:
            break
    return px == 256 and cin % 32 == 0 and side % 16 == 0


def _block_rank(npix, side, cin, cout):
    """rank[tap, ci] of the block that holds k = (tap, ci) in the chain."""
    tap, ci = np.meshgrid(np.arange(9), np.arange(cin), indexing="ij")
    if _chunk_major(npix, side, cin, cout):
        return (ci // 32) * 9 + tap
    return (tap * cin + ci) // 32


def _draw(rng, rank):
    """Weights [9, cin] with one nonzero a block: a pair of +-BIG and powers of
    two in up to 6 other blocks; and what the chain adds up to."""
    w = np.zeros(rank.shape, np.float32)
    blocks = rng.permutation(rank.max() + 1)[:8]
    vals = [BIG, -BIG] + [2.0 ** k for k in range(len(blocks) - 2)]
    at = {}
    for b, v in zip(blocks, vals):
        k = rng.choice(np.flatnonzero(rank.ravel() == b))
        w.ravel()[k] = v
        at[b] = np.float32(v)
    s = np.float32(0)
    for b in sorted(at):
        s = np.float32(s + at[b])
    return w, float(s)


def _layers(base):
    return {"in": (8, base), "mid": (base, base), "out": (base, 16)}


class Net:
    def __init__(self, base, S, batch):
        from iskra_amd import Context, _lib
        self.ctx = Context(0)
        self.ws = _lib.WarmStart(self.ctx, levels=1, base=base, side=S, max_batch=batch)
        self.base, self.S, self.batch = base, S, batch
        self.count = batch * (S - 1) * (S - 1)
        self.w = {k: np.zeros((co, 9, ci), np.float32) for k, (ci, co) in _layers(base).items()}

    def box(self, m):
        """1 at pixels at least m from every side."""
        b = np.zeros((self.batch, self.S, self.S), np.float32)
        b[:, m:self.S - m, m:self.S - m] = 1.0
        return b

    def params(self):
        self.ws.set_params(np.concatenate([self.w[k].ravel() for k in ("in", "mid", "out")]))

    def grads(self, x, g):
        """Parameter gradients with the output's gradient at g (powers of two):
        t = o - d with 2 d / count = g to within 2^-22, which bf16 rounds to g."""
        o = self.ws.forward(x).reshape(g.shape)
        d = g.astype(np.float64) * self.count / 2
        t = np.where(g != 0, o - d, o).astype(np.float32)
        _, gr = self.ws.backward(x, t)
        out, k = {}, 0
        for name in ("in", "mid", "out"):
            n = self.w[name].size
            out[name] = gr[k:k + n].reshape(self.w[name].shape)
            k += n
        return out

    def close(self):
        self.ws.close()
        self.ctx.close()


@pytest.fixture
def net(gpu_ready, base, S, batch):
    n = Net(base, S, batch)
    yield n
    n.close()


# both orders of the three layers, channels in whole and in broken blocks of 32
NETS = [(16, 16, 1), (32, 16, 3), (48, 32, 1), (64, 32, 2), (64, 128, 1), (64, 128, 4),
        (32, 128, 4), (80, 64, 1), (256, 64, 1), (320, 16, 1)]


@pytest.mark.parametrize("base,S,batch", NETS)
@pytest.mark.parametrize("layer", ["in", "mid", "out"])
def test_convolution(net, base, S, batch, layer):
    rng = np.random.default_rng(base + S + batch)
    cin, cout = _layers(base)[layer]
    rank = _block_rank(batch * S * S, S, cin, cout)
    if layer == "in":  # one input channel carries the plane
        rank = np.where(np.arange(cin) == 0, rank, -1)
    net.w["in"][:, 4, 0] = 1.0
    for c in range(base):
        net.w["mid"][c, 4, c] = 1.0
    want = np.zeros(cout)
    for c in range(cout if layer != "out" else 1):
        net.w[layer][c], want[c] = _draw(rng, rank)
    net.params()
    if layer == "out":
        o = net.ws.forward(net.box(0)).reshape(batch, S, S)
        assert (o[:, 3:-3, 3:-3] == want[0]).all(), (o[0, 5, 5], want[0])
    else:
        # every channel shows in the output layer's gradient
        g = net.box(5) * 2.0 ** -10
        gr = net.grads(net.box(2), g)["out"][0, 4]
        assert np.array_equal(gr / g.sum(), want), (gr / g.sum(), want)


@pytest.mark.parametrize("base,S,batch", NETS)
@pytest.mark.parametrize("layer", ["mid", "out"])
def test_input_gradient(net, base, S, batch, layer):
    rng = np.random.default_rng(base + S + batch + 1)
    cout, cin = _layers(base)[layer]  # of the gradient's convolution
    rank = _block_rank(batch * S * S, S, cin, cout)
    if layer == "out":  # its gradient has one channel
        rank = np.where(np.arange(cin) == 0, rank, -1)
    want = np.zeros(cout)
    wt = np.zeros((cout, 9, cin), np.float32)
    for c in range(cout):
        wt[c], want[c] = _draw(rng, rank)
    w = np.ascontiguousarray(wt[:, ::-1].transpose(2, 1, 0))  # mirrored taps
    # the layer's input is positive in a box 1 narrower than where its output's
    # gradient is constant
    if layer == "out":
        net.w["in"][:, 4, 0] = 1.0
        for c in range(base):
            net.w["mid"][c, 4, c] = 1.0
        net.w["out"][:] = w
        g = net.box(3) * 2.0 ** 60  # not small beside the output
        x = net.box(5)
        net.params()
        gr = net.grads(x, g)["mid"][:, 4, 0] / (x.sum() * 2.0 ** 60)
    else:
        net.w["in"][:, :, 0] = 1.0  # a plane one pixel wider than x
        net.w["mid"][:] = w
        want[base - 1] = 0.0
        net.w["mid"][:, :, base - 1] = 0.0
        net.w["mid"][:, 4, base - 1] = 2.0 ** 60  # all outputs positive
        net.w["out"][0, 4, :] = 1.0
        g = net.box(1) * 2.0 ** 60
        x = net.box(5)
        net.params()
        gr = net.grads(x, g)["in"][:, 4, 0] / (x.sum() * 2.0 ** 60)
        gr[base - 1] = 0.0
    assert np.array_equal(gr, want), (gr, want)


def _chunks(cin, cout, nseg):
    per = 9 * cin * cout
    fit = max(1, (64 << 20) // 4 // per)
    want = max(1, 1024 // (-(-cout // 32) * -(-cin // 16)))
    most = min(fit, want, nseg)
    return -(-nseg // most)


@pytest.mark.parametrize("base,S,batch", NETS + [(32, 8 * 2, 5), (16, 256, 3), (48, 64, 3)])
def test_weight_gradient(net, base, S, batch):
    rng = np.random.default_rng(base + S + batch + 2)
    net.w["in"][:, 4, 0] = 1.0
    for c in range(base):
        net.w["mid"][c, 4, c] = 1.0
    net.w["out"][0, 4, :] = 1.0
    net.params()
    # at most one pixel in 32, none at the sides: a few pairs of +-BIG among small ones
    nblk = batch * S * S // 32
    p = np.arange(batch * S * S)
    inner = (p % S > 0) & (p % S < S - 2) & (p // S % S > 0) & (p // S % S < S - 2)
    g = np.zeros(batch * S * S)
    pairs = max(1, nblk // 24)
    for k, b in enumerate(rng.permutation(nblk)):
        q = np.flatnonzero(inner[32 * b:32 * b + 32])
        if len(q):
            v = (BIG, -BIG)[k % 2] if k < 2 * pairs else 2.0 ** (k % 4)
            g[32 * b + rng.choice(q)] = v
    g *= 2.0 ** 20
    vals = g.reshape(nblk, 32).sum(1).astype(np.float32)
    got = net.grads(np.ones((batch, S, S), np.float32), g.reshape(batch, S, S))
    for name, (cin, cout) in _layers(base).items():
        spc = _chunks(cin, cout, nblk // 2)
        total = np.float32(0)
        for c0 in range(0, nblk, 2 * spc):
            s = np.float32(0)
            for v in vals[c0:c0 + 2 * spc]:
                s = np.float32(s + v)
            total = np.float32(total + s)
        gr = got[name]
        if name == "in":
            gr = gr[:, :, :1]
        if name == "out":
            gr = gr[:1]
        assert (gr == total).all(), (name, spc, np.unique(gr), total)
