"""The warm-start network's GPU kernels against the FP64 oracle
(oracle/net.py, run with the same bfloat16 roundings as the GPU's storage):
the MFMA operand layout, the forward pass, every parameter gradient, one
Adam step, and tile-wise inference against whole-volume inference."""
import numpy as np
import pytest

from conftest import relL2
from oracle import net as onet

pytestmark = pytest.mark.gpu


def flat(params):
    return np.concatenate([np.concatenate([w.reshape(-1), b.reshape(-1)]) for w, b in params]).astype(np.float32)


def unflat(v):
    out, o = [], 0
    for ws, bs in onet.param_shapes():
        nw, nb = int(np.prod(ws)), int(np.prod(bs))
        out.append([v[o:o + nw].reshape(ws).astype(np.float64), v[o + nw:o + nw + nb].reshape(bs).astype(np.float64)])
        o += nw + nb
    return out


def test_mfma_operand_layout(fm):
    rng = np.random.default_rng(0)
    A = onet.bf16(rng.normal(size=(32, 16)))
    B = onet.bf16(rng.normal(size=(16, 32)))
    net = fm.Net(0)
    dA = fm.DeviceArray.from_host(fm.to_bf16_bits(A))
    dB = fm.DeviceArray.from_host(fm.to_bf16_bits(B))
    dD = fm.DeviceArray((32, 32), np.float32)
    assert net.L.fmvd_net_mfma_layout_test(dA.ptr, dB.ptr, dD.ptr) == 0
    fm.check()
    np.testing.assert_allclose(dD.download(), A @ B, rtol=1e-5, atol=1e-5)


def make_problem(seed, shape=(2, 5, 9, 40)):
    rng = np.random.default_rng(seed)
    params = onet.init_params(seed)
    for p in params:
        p[0] *= 2.0
        p[1][...] = rng.normal(0.0, 0.05, p[1].shape)
    params = unflat(flat(params))  # FP32-representable master weights
    N, D, H, W = shape
    x = onet.bf16(rng.uniform(0.2, 1.5, size=(N, D, H, W, 2)))
    t = rng.uniform(0.2, 1.5, size=(N, D, H, W)).astype(np.float32).astype(np.float64)
    return params, x, t


def oracle_batch(params, x, t):
    """Oracle loss/grads for a batch: the mean over all samples' voxels."""
    N = x.shape[0]
    loss, grads, ys = 0.0, None, []
    for n in range(N):
        l, g, y = onet.loss_and_grads(params, x[n], t[n], quant=True)
        loss += l / N
        ys.append(y)
        g = [[gw / N, gb / N] for gw, gb in g]
        grads = g if grads is None else [[a[0] + b[0], a[1] + b[1]] for a, b in zip(grads, g)]
    return loss, grads, np.stack(ys)


def run_gpu(fm, params, x, t):
    net = fm.Net(1)
    net.set_params(flat(params))
    dx = fm.DeviceArray.from_host(fm.to_bf16_bits(x))
    dt = fm.DeviceArray.from_host(t.astype(np.float32))
    dy = fm.DeviceArray(t.shape, np.float32)
    net.forward(dx, t.shape, dy)
    fm.device_synchronize()
    y = dy.download()
    loss = net.backward(dx, dt, t.shape)
    return net, y, loss, net.grads()


def test_forward_and_gradients_match_oracle(fm):
    params, x, t = make_problem(7)
    net, y, loss, g = run_gpu(fm, params, x, t)
    loss_o, grads_o, y_o = oracle_batch(params, x, t)
    assert relL2(y, y_o) < 2e-3, relL2(y, y_o)
    assert abs(loss - loss_o) < 2e-3 * loss_o
    go = unflat(flat(grads_o).astype(np.float64)) if False else grads_o
    gg = unflat(g)
    for l in range(onet.LAYERS):
        for i in range(2):
            r = relL2(gg[l][i], go[l][i])
            print(f"layer {l + 1} {'W' if i == 0 else 'b'}: relL2 {r:.2e}")
            assert r < 2e-2, (l, i, r)


def test_adam_step_matches_oracle(fm):
    params, x, t = make_problem(11, shape=(1, 4, 6, 33))
    net, _, _, g = run_gpu(fm, params, x, t)
    net.adam(1e-3)
    got = net.params()
    p = unflat(flat(params))
    m = [[np.zeros_like(a), np.zeros_like(b)] for a, b in p]
    v = [[np.zeros_like(a), np.zeros_like(b)] for a, b in p]
    onet.adam_step(p, unflat(g), m, v, 1, lr=1e-3)
    np.testing.assert_allclose(got, flat(p), rtol=0, atol=2e-6)


def test_training_reduces_loss(fm):
    """80 Adam steps at lr 2e-4 on a smoothing task; the FP64 oracle trained
    the same way falls to ~7% of its initial loss."""
    rng = np.random.default_rng(5)
    N, D, H, W = 2, 6, 16, 32
    x = onet.bf16(rng.uniform(0.2, 1.5, size=(N, D, H, W, 2)))
    m = 0.5 * (x[..., 0] + x[..., 1])
    mp = np.pad(m, ((0, 0), (0, 0), (0, 0), (1, 1)))
    t = (0.5 * m + 0.25 * (mp[..., 2:] + mp[..., :-2])).astype(np.float32)
    net = fm.Net(3)
    dx = fm.DeviceArray.from_host(fm.to_bf16_bits(x))
    dt = fm.DeviceArray.from_host(t)
    losses = []
    for _ in range(80):
        losses.append(net.backward(dx, dt, t.shape))
        net.adam(2e-4)
    print("losses", [round(l, 5) for l in losses[::10]], losses[-1])
    assert losses[-1] < 0.5 * losses[0]
    assert np.isfinite(losses).all()


def test_tiled_inference_equals_whole_volume(fm):
    rng = np.random.default_rng(9)
    D, H, W, V = 20, 70, 90, 3
    views = [fm.DeviceArray.from_host(rng.integers(50, 900, size=(D, H, W)).astype(np.uint16)) for _ in range(V)]
    net = fm.Net(4)
    whole = fm.DeviceArray((D, H, W), np.float32)
    tiled = fm.DeviceArray((D, H, W), np.float32)
    net.infer(views, 300.0, whole, tile=(D, H, W, 16))
    net.infer(views, 300.0, tiled, tile=(8, 24, 32, 8))
    a, b = whole.download(), tiled.download()
    assert np.isfinite(a).all() and a.min() >= 1e-3
    assert np.array_equal(a, b)


@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 1, 8, 32), (1, 3, 9, 33), (1, 4, 17, 31), (1, 5, 16, 66),
                                   (3, 90, 4, 5)])
def test_gradients_at_tile_edges(fm, shape):
    """Volumes of one voxel, of whole tiles, of a tile and a remainder on each
    axis, and of more (sample, plane) pairs than CUs.  Tolerance: five times
    the bfloat16 spacing 2^-8, since a stored activation may round to the
    neighbouring bfloat16 value."""
    params, x, t = make_problem(13, shape)
    _, y, loss, g = run_gpu(fm, params, x, t)
    loss_o, grads_o, y_o = oracle_batch(params, x, t)
    assert relL2(y, y_o) < 2e-2
    assert abs(loss - loss_o) < 2e-2 * loss_o
    gg = unflat(g)
    for l in range(onet.LAYERS):
        for i in range(2):
            d, n = np.linalg.norm(gg[l][i] - grads_o[l][i]), np.linalg.norm(grads_o[l][i])
            assert d <= 2e-2 * n + 1e-7, (l, i, d, n)


@pytest.mark.parametrize("shape", [(1, 4, 16, 32), (2, 5, 17, 33), (1, 9, 33, 65), (3, 8, 15, 24)])
def test_edge_layers_at_box_edges(fm, shape):
    """Input layer and the output layer's input gradient at the edges of their 4 x 16 x 32 boxes.  With the blocks'
    weights and biases zero the network is h5 = relu(conv(x)), y = conv(h5): the output is one FP32 sum of bfloat16
    products, so it differs from FP64 by FP32 sums of 27 x 32 terms (1e-6) and rare flips of a bfloat16 rounding
    (2^-8 each); an h1 or a neighbour taken from elsewhere changes it by its own size."""
    params, x, t = make_problem(31, shape)
    for l in range(1, 5):
        params[l][0][...] = 0.0
        params[l][1][...] = 0.0
    net, y, loss, g = run_gpu(fm, params, x, t)
    loss_o, grads_o, y_o = oracle_batch(params, x, t)
    assert np.abs(y - y_o).max() <= 2e-3 * np.abs(y_o).max()
    gg = unflat(g)
    for l in (0, 5):
        for i in range(2):
            assert np.linalg.norm(gg[l][i] - grads_o[l][i]) <= 5e-3 * np.linalg.norm(grads_o[l][i]), (l, i)


@pytest.mark.parametrize("shape", [(1, 1, 1), (16, 8, 32), (17, 9, 33), (33, 23, 66)])
def test_inference_output_layer(fm, shape):
    """Inference's output layer at the edges of its 8 x 32 columns and 16-plane segments, against the oracle and
    against the training path's chain of FP32 sums of the same activations.  The input is small integers (exact in
    bfloat16) and the blocks' weights are zero, so both paths see the same h5; sums of 27 x 32 products in FP32
    differ by at most 864 roundings of 2^-24 of the sum of magnitudes (the oracle with |W6| gives it)."""
    rng = np.random.default_rng(17)
    params, _, _ = make_problem(31, (1,) + shape)
    for l in range(1, 5):
        params[l][0][...] = 0.0
        params[l][1][...] = 0.0
    view = rng.integers(1, 9, size=shape).astype(np.uint16)
    net = fm.Net(1)
    net.set_params(flat(params))
    got = fm.DeviceArray(shape, np.float32)
    net.infer([fm.DeviceArray.from_host(view)], 1.0, got, floor_value=-1e30)
    x = np.stack([view, view], -1).astype(np.float64)[None]
    chain = fm.DeviceArray((1,) + shape, np.float32)
    net.forward(fm.DeviceArray.from_host(fm.to_bf16_bits(x)), (1,) + shape, chain)
    fm.device_synchronize()
    got, chain = got.download(), chain.download()[0]
    want, _ = onet.forward(params, x[0], quant=True)
    err, ref = np.abs(got - want), np.abs(chain - want)
    print(f"{shape}: rms {np.sqrt(np.mean(err**2)):.2e} (chain {np.sqrt(np.mean(ref**2)):.2e}), max {err.max():.2e}")
    params[5][0] = np.abs(params[5][0])
    magnitude = np.abs(onet.forward(params, x[0], quant=True)[0]).max()
    assert np.abs(got.astype(np.float64) - chain).max() <= 864 * 2.0**-24 * magnitude
    assert err.max() <= 2e-3 * np.abs(want).max()


@pytest.mark.parametrize("shape, layers, times", [((4, 64, 128, 128), (0, 5), 1.0), ((8, 1024, 8, 8), (0, 1, 5), 1.6)])
def test_weight_gradients_round_like_row_sums(fm, shape, layers, times):
    """Rounding of the weight gradients: no worse than FP32 sums by rows, of the rows of a plane, and FP64 over the planes.
    The network is one whose gradients have exactly known operands: the input layer reads one voxel and channel, the
    blocks add a constant, the output layer reads one voxel, so that g = bf16(dy w) and every activation follow on the
    host, and the error is that of the sums alone.  With rows of 32 voxels and S steps of rows a block the variance is
    (32 + S) / (W + H) of the row sums' (0.61 of their error at 4 x 64 x 128 x 128, S = 64; one chain over a block would
    have 2.8 times it; in the input layer, whose products have 16 bits, short row sums are exact and the two are near
    each other).  In small planes both add a few rows and matrix instructions that truncate may double the variance (1.4
    times; partial sums over the 8 planes that a cap of 1024 rows gives: more than 2)."""
    rng = np.random.default_rng(5)
    bf = lambda a: onet.bf16(np.asarray(a, np.float32)).astype(np.float32)
    params = [[np.zeros(ws, np.float32), np.zeros(bs, np.float32)] for ws, bs in onet.param_shapes()]
    w1, w6 = bf(rng.uniform(0.2, 1.0, 32)), bf(rng.uniform(0.2, 1.0, 32))
    params[0][0].reshape(27, 32, 2)[13, :, 0] = w1
    params[5][0].reshape(27, 32)[13] = w6
    for l in range(5):
        params[l][1][...] = bf(rng.uniform(0.05, 0.3, 32))
    x = bf(rng.uniform(0.0, 1.0, shape + (2,)))
    net = fm.Net(1)
    net.set_params(flat(params))
    dx = fm.DeviceArray.from_host(fm.to_bf16_bits(x))
    d = fm.DeviceArray(shape, np.float32)
    net.forward(dx, shape, d)
    fm.device_synchronize()
    y = d.download()
    t = (y - rng.normal(0.0, 1.0, shape)).astype(np.float32)
    dy = (2.0 * (y.astype(np.float64) - t) / t.size).astype(np.float32)
    net.backward(dx, fm.DeviceArray.from_host(t), shape)
    got = unflat(net.grads())

    def activation(c, layer):  # channel c of the layer's output
        h = bf(params[0][1][c] + x[..., 0] * w1[c])
        for l in range(1, layer + 1):
            h = bf(h + params[l][1][c])
        return h

    def row_sums(p):  # FP32 along the rows, then along the columns, FP64 over the planes
        s = np.cumsum(np.cumsum(p, -1, dtype=np.float32)[..., -1], -1, dtype=np.float32)[..., -1]
        return s.sum(dtype=np.float64)

    g = [bf(dy * w) for w in w6]
    for l in layers:
        a = [np.ascontiguousarray(x[..., i]) for i in range(2)] if l == 0 else [activation(c, l - 1) for c in range(32)]
        if l == 1:  # 32 x 32 pairs: a few of them
            a = a[:8]
        gpu, ref = [], []
        for co, gv in enumerate(g if l < 5 else [dy]):
            for ci, av in enumerate(a):
                exact = np.dot(gv.reshape(-1).astype(np.float64), av.reshape(-1).astype(np.float64))
                gpu.append(got[l][0].reshape(27, -1, len(a) if l != 1 else 32)[13, co, ci] - exact)
                ref.append(row_sums(gv * av) - exact)
        rms = [float(np.sqrt(np.mean(np.square(e)))) for e in (gpu, ref)]
        print(f"{shape} layer {l + 1}: error {rms[0]:.2e}, row sums {rms[1]:.2e}", flush=True)
        assert rms[0] <= times * rms[1], (l, rms)


@pytest.mark.parametrize("shape", [(1, 1, 1), (2, 16, 32), (5, 17, 33), (16, 40, 64), (18, 9, 40), (33, 47, 95)])
def test_few_boxes_are_shared_by_blocks(fm, shape):
    """Volumes of few boxes and columns, whose rows and planes are dealt to more blocks, give the bits that they have
    among the voxels of a larger batch, which takes one block a box and segments of 16 planes.  The small volume is the
    first sample of that batch."""
    n = -(-2100 * 2048 // int(np.prod(np.ceil(np.array(shape) / (4, 16, 32)) * (4, 16, 32))))
    params, x, _ = make_problem(3, (2,) + shape)
    net = fm.Net(1)
    net.set_params(flat(params))
    for many in (1, min(n, 2100)):
        xs = np.concatenate([x] + [x[:1]] * max(0, many - 2))[:many]
        y = fm.DeviceArray((many,) + shape, np.float32)
        net.forward(fm.DeviceArray.from_host(fm.to_bf16_bits(xs)), (many,) + shape, y)
        fm.device_synchronize()
        if many == 1:
            one = y.download()[0]
    assert np.array_equal(one, y.download()[0])
    view = np.random.default_rng(2).integers(1, 9, shape).astype(np.uint16)
    est = fm.DeviceArray(shape, np.float32)
    net.infer([fm.DeviceArray.from_host(view)], 1.0, est, floor_value=-1e30)
    x = onet.bf16(np.stack([view, view], -1).astype(np.float64))
    want, _ = onet.forward(params, x, quant=True)
    assert relL2(est.download(), want) < 2e-2


def test_failed_allocation_leaves_the_network_usable(fm):
    """A volume that does not fit the device is an error; the next estimate allocates its own activations."""
    rng = np.random.default_rng(4)
    view = fm.DeviceArray.from_host(rng.integers(1, 900, (6, 20, 30)).astype(np.uint16))
    a, b = fm.DeviceArray((6, 20, 30), np.float32), fm.DeviceArray((6, 20, 30), np.float32)
    net = fm.Net(3)
    net.infer([view], 500.0, a)
    dummy = fm.DeviceArray((16,), np.float32)
    with pytest.raises(fm.FmvdError):
        net.forward(dummy, (1, 1000000, 400, 256), dummy)  # 410 GB of input alone: refused before any launch
    net.infer([view], 500.0, b)
    assert np.array_equal(a.download(), b.download())


@pytest.mark.parametrize("shape, tile", [((20, 50, 70), (8, 24, 32, 6)), ((1, 8192, 2200), None)])
def test_tiles_with_the_reach_as_halo(fm, shape, tile):
    """Tiles with a halo of exactly the network's reach, given and as fmvd_net_infer cuts a volume of more than 16 M voxels
    itself: the bits of one tile."""
    view = fm.DeviceArray.from_host(np.random.default_rng(6).integers(1, 900, shape).astype(np.uint16))
    whole, tiled = fm.DeviceArray(shape, np.float32), fm.DeviceArray(shape, np.float32)
    net = fm.Net(3)
    net.infer([view], 500.0, whole, tile=shape + (6,))
    net.infer([view], 500.0, tiled, tile=tile)
    a, b = whole.download(), tiled.download()
    assert np.isfinite(a).all() and a.std() > 0
    assert np.array_equal(a, b)
