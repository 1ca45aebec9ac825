"""GPU checks of the CNN kernels (k_cnn.hip) against the CPU oracle.

Bars:
* each layer, fed the GPU's own BF16 input, reproduces the oracle's BF16
  output except where FP32 accumulation order moves a value across a rounding
  boundary: at most 1% of the values differ, each by at most one BF16 unit or
  (where the 288-term sum cancels) by 1e-3 of the layer's rms;
* the FP32 output y and every parameter gradient agree with the oracle
  end to end (the BF16 activation chain of each side) to rel-L2 1e-2, the loss
  to 1e-5;
* Adam agrees with the oracle's update to FP32 rounding;
* a few hundred Adam steps on a fixed task lower the loss.
"""
import numpy as np
import pytest

from oracle import cnn_oracle as K

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from projects_amd import learned as Lrn


def bf16_bits_to_f32(t):
    u = t.cpu().numpy().view(np.uint16).astype(np.uint32) << 16
    return u.view(np.float32)


def ulp_diff(a, b):
    """Distance in BF16 units between two arrays of BF16 values (as float32)."""
    ia = (a.view(np.uint32) >> 16).astype(np.int64)
    ib = (b.view(np.uint32) >> 16).astype(np.int64)
    ia = np.where(ia & 0x8000, -(ia & 0x7FFF), ia)
    ib = np.where(ib & 0x8000, -(ib & 0x7FFF), ib)
    return np.abs(ia - ib)


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-300))


def make(seed, n=2, H=19, W=45, scale=1.7):
    rng = np.random.default_rng(seed)
    p = Lrn.init_params(seed)
    pd = Lrn.unflatten(p)
    pd["W5"] = pd["W5"] * 5.0
    for k in ("b1", "b2", "b3", "b4", "b5"):
        pd[k][...] = rng.standard_normal(pd[k].shape) * 0.05
    flat = np.concatenate([pd[k].ravel() for k, _ in Lrn.PARAM_SHAPES]).astype(np.float32)
    x = rng.standard_normal((n, H, W)).astype(np.float32) * 2.0
    t = (x + rng.standard_normal((n, H, W)).astype(np.float32) * 0.3).astype(np.float32)
    net = Lrn.Corrector(params=flat, scale=scale)
    return net, {k: v.astype(np.float32) for k, v in pd.items()}, x, t


def test_weight_packing_rounds_like_the_oracle():
    """The kernels' BF16 rounding (the hardware convert) against the oracle's
    integer round-to-nearest-even, bitwise, through the weight packing of the
    three 32 -> 32 layers: exact ties to even and to odd, one unit either side
    of a tie, subnormals (ties included), the largest finites (rounding to
    infinity), signed zeros and infinities, and random floats of every
    exponent."""
    rng = np.random.default_rng(77)
    n = 3 * 9 * K.C * K.C
    hi = rng.integers(0, 1 << 16, n, dtype=np.uint64)
    lo = rng.choice(np.array([0x8000, 0x7FFF, 0x8001, 0x0000, 0xFFFF], np.uint64), n)
    u = (hi << 16) | lo
    special = np.array([0x00008000, 0x00018000, 0x00007FFF, 0x00000001, 0x807F8000, 0x7F7FFFFF, 0x7F7F8000,
                        0x7F7E8000, 0xFF7FFFFF, 0x00000000, 0x80000000, 0x7F800000, 0xFF800000, 0x3F808000,
                        0x3F818000], np.uint64)
    u[:special.size] = special
    u[-4096:] = rng.integers(0, 1 << 32, 4096, dtype=np.uint64)
    w = u.astype(np.uint32).view(np.float32)
    w = np.where(np.isnan(w), np.float32(1.0), w).astype(np.float32)
    net, pd, _, _ = make(5)
    sizes = {name: int(np.prod(shape)) for name, shape in Lrn.PARAM_SHAPES}
    off, flat = 0, net.params.cpu().numpy().copy()
    per = 9 * K.C * K.C
    for name, _ in Lrn.PARAM_SHAPES:
        if name in ("W2", "W3", "W4"):
            l = int(name[1]) - 2
            flat[off:off + per] = w[l * per:(l + 1) * per]
        off += sizes[name]
    net.params.copy_(torch.from_numpy(flat))
    net.pack()
    torch.cuda.synchronize()
    packed = net.packed.cpu().numpy().view(np.uint16)
    for l in range(3):
        W = w[l * per:(l + 1) * per].reshape(K.C, K.C, 9)  # [co][ci][tap]
        want = (K.bf16(W).view(np.uint32) >> 16).astype(np.uint16)
        fwd = packed[l * 2 * per:l * 2 * per + per].reshape(9, K.C, K.C)  # [tap][co][ci]
        assert np.array_equal(fwd, want.transpose(2, 0, 1)), l


def test_forward_layers_match_oracle():
    net, pd, x, _ = make(1)
    xg = torch.from_numpy(x).cuda()
    y, stats = net.forward(xg, train=True)
    torch.cuda.synchronize()
    acts = net._buffers(*x.shape, True)[0]
    a = [bf16_bits_to_f32(t) for t in acts]
    # layer 1 from x; layers 2-4 from the GPU's previous activation
    c = K.forward(pd, x, net.scale)
    wq = c["wq"]
    expect = [c["a1"]]
    for l in (2, 3, 4):
        z = K.conv3x3(a[l - 2], wq[f"W{l}"]) + wq[f"b{l}"]
        expect.append(K.bf16(np.maximum(z, 0.0)))
    for l in range(4):
        e = expect[l].astype(np.float32)
        d = ulp_diff(a[l], e)
        tol = np.maximum(np.abs(e) * 2.0 ** -7, 1e-3 * np.sqrt(np.mean(e.astype(np.float64) ** 2)))
        print(f"a{l + 1}: max ulp {d.max()}, off {np.mean(d > 0):.2e}", flush=True)
        assert np.mean(d > 0) < 0.01 and (np.abs(a[l] - e) <= tol).all(), l
    r = K.conv3x3(a[3], wq["W5"][None])[..., 0] + wq["b5"][0]
    yn = x / np.float32(net.scale) + r
    assert rel(y.cpu().numpy(), yn * net.scale) < 1e-5
    s = stats.cpu().numpy()
    assert np.allclose(s[:, 0], (r ** 2).reshape(2, -1).sum(1), rtol=1e-4)
    assert np.allclose(s[:, 1], ((x / np.float32(net.scale)).astype(np.float64) ** 2).reshape(2, -1).sum(1),
                       rtol=1e-4)
    # end to end against the oracle's own BF16 chain
    assert rel(y.cpu().numpy(), c["y"] * net.scale) < 1e-2


@pytest.mark.parametrize("shape", [(3, 37, 70), (1, 16, 32), (2, 5, 7), (1, 130, 200)])
def test_fused_inference_is_bitwise_forward(shape):
    """The fused kernel (all layers in LDS, halo recomputation) gives bitwise
    the layer-by-layer forward's output, borders and ragged tiles included."""
    net, _, _, _ = make(6)
    x = torch.randn(shape, device="cuda") * 2.0
    y1, s1 = net.forward(x)
    y2, s2 = net.infer(x)
    torch.cuda.synchronize()
    assert torch.equal(y1, y2)
    assert torch.allclose(s1, s2, rtol=1e-4)


@pytest.mark.parametrize("shape", [(3, 37, 70), (1, 16, 32), (2, 5, 7), (1, 130, 200)])
def test_inference_forward_is_bitwise_training_forward(shape):
    """forward() for inference (activation buffers aliased: the first layer
    fused into the second, a1 never stored) gives bitwise the outputs and
    per-image sums of the training forward (five layer kernels, every
    activation stored), borders and ragged tiles included."""
    net, _, _, _ = make(6)
    x = torch.randn(shape, device="cuda") * 2.0
    y1, s1 = net.forward(x, train=True)
    y1, s1 = y1.clone(), s1.clone()
    y2, s2 = net.forward(x)
    torch.cuda.synchronize()
    assert torch.equal(y1, y2)
    assert torch.equal(s1, s2)


def test_backward_matches_oracle():
    net, pd, x, t = make(2)
    xg, tg = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    net.forward(xg, train=True)
    net.backward(xg, tg)
    torch.cuda.synchronize()
    acts = [bf16_bits_to_f32(a) for a in net._buffers(*x.shape, True)[0]]
    # oracle backward on the GPU's activations: differences are accumulation order
    c = K.forward(pd, x, net.scale)
    for l in range(4):
        c[f"a{l + 1}"] = acts[l]
    yn = net._buffers(*x.shape, True)[2].cpu().numpy()
    c["y"] = yn
    loss, g = K.loss_and_backward(pd, c, t, net.scale)
    assert abs(float(net.loss.cpu()) - loss) <= 1e-5 * loss
    gg = Lrn.unflatten(net.grads.cpu().numpy())
    for k in g:
        e = rel(gg[k], g[k])
        print(f"grad {k}: rel-L2 {e:.2e}", flush=True)
        assert e < 1e-2, k


def test_adam_matches_oracle():
    rng = np.random.default_rng(3)
    net = Lrn.Corrector(seed=3)
    p0 = net.params.cpu().numpy().astype(np.float64)
    pd = {"p": p0.copy()}
    m, v = {"p": np.zeros_like(p0)}, {"p": np.zeros_like(p0)}
    for step in range(1, 4):
        g = rng.standard_normal(p0.shape).astype(np.float32)
        net.grads.copy_(torch.from_numpy(g))
        net.adam(lr=1e-3)
        pd, m, v = K.adam(pd, {"p": g.astype(np.float64)}, m, v, step)
    torch.cuda.synchronize()
    got = net.params.cpu().numpy()
    assert np.max(np.abs(got - pd["p"])) < 1e-6


def test_training_lowers_loss():
    """Learn to remove a fixed 3x3 blur residual: the loss falls by 4x."""
    rng = np.random.default_rng(4)
    net = Lrn.Corrector(seed=4, scale=1.0)
    n, H, W = 8, 32, 64
    tgt = rng.standard_normal((n, H, W)).astype(np.float32)
    k = np.array([[1, 2, 1], [2, 4, 2], [1, 2, 1]], np.float32) / 16.0
    pad = np.pad(tgt, ((0, 0), (1, 1), (1, 1)))
    x = sum(k[i, j] * pad[:, i:i + H, j:j + W] for i in range(3) for j in range(3)).astype(np.float32)
    xg, tg = torch.from_numpy(x).cuda(), torch.from_numpy(tgt).cuda()
    first = float(net.train_step(xg, tg, lr=2e-3).cpu())
    for _ in range(300):
        net.train_step(xg, tg, lr=2e-3)
    last = float(net.train_step(xg, tg, lr=2e-3).cpu())
    print(f"loss {first:.4f} -> {last:.4f}", flush=True)
    assert last < first / 4


def test_fallback_keeps_plain_image():
    net, _, x, _ = make(5, n=3, H=16, W=32)
    xg = torch.from_numpy(x).cuda()
    net.threshold = 0.0  # every correction is "too large"
    y, used = net.correct(xg)
    torch.cuda.synchronize()
    assert not bool(used.any()) and torch.equal(y, xg)
    net.threshold = 1e9
    y, used = net.correct(xg)
    assert bool(used.all()) and not torch.equal(y, xg)


def test_trained_network_beats_sparse_gridrec():
    """Train on gridrec pairs (24 / 240 angles, 128^2 phantoms with texture) and
    compare on held-out phantoms: the corrected sparse-angle images are closer
    to the dense-angle gridrec than the plain sparse-angle ones."""
    inp, tgt = Lrn.make_pairs(512, 128, 24, 240, seed=9, n_tex=32, tex_fmax=12.0)
    net = Lrn.Corrector(seed=9, scale=float(tgt.std()))
    hist, steps, _ = Lrn.train(net, inp, tgt, steps=400, batch=16, lr=2e-3)
    vi, vt = Lrn.make_pairs(32, 128, 24, 240, seed=9, n_tex=32, tex_fmax=12.0, slice0=100000)
    vy, used = net.correct(vi)
    torch.cuda.synchronize()
    plain = np.mean([Lrn.psnr(vi[i], vt[i]) for i in range(32)])
    learned = np.mean([Lrn.psnr(vy[i], vt[i]) for i in range(32)])
    print(f"loss {hist[0][1]:.4f} -> {hist[-1][1]:.4f}; held-out PSNR plain {plain:.2f} dB, learned {learned:.2f} dB",
          flush=True)
    assert bool(used.all())
    assert learned > plain + 1.0


def _window(a, y0, x0, w, halo):
    """a[..., y0-halo : y0+w+halo, x0-halo : x0+w+halo] clipped to the image,
    and the offsets of the w x w window inside it."""
    H, W = a.shape[-2:]
    ya, xa = max(0, y0 - halo), max(0, x0 - halo)
    yb, xb = min(H, y0 + w + halo), min(W, x0 + w + halo)
    return a[..., ya:yb, xa:xb], y0 - ya, x0 - xa


@pytest.mark.parametrize("fused", [False, True])
def test_inference_2048_slice_matches_oracle(fused):
    """The sparse-angle inference shape: one 2048 x 2048 gridrec image of a
    150-angle, 2048-detector sinogram through the network on the GPU, checked
    against the oracle on windows.  Five 3x3 layers see 5 pixels around each
    output, so the oracle on a window widened by that halo (clipped at the
    image's edges, where both sides pad with zeros) gives the window's exact
    outputs; the windows include two image corners."""
    from projects_amd import gridrec as gr

    n, nang = 2048, 150
    sino = torch.empty((1, nang, n), dtype=torch.float32, device="cuda")
    gr.phantom_sinograms(sino, 77, nang, n, [n / 2], 20, n_tex=64, tex_amp=0.15, tex_fmax=24.0)
    x = Lrn.gridrec_images(sino, n, n / 2)
    assert x.shape == (1, n, n)
    net, pd, _, _ = make(8, scale=float(x.std()))
    y, _ = net.infer(x) if fused else net.forward(x)
    torch.cuda.synchronize()
    xs, ys = x.cpu().numpy(), y.cpu().numpy()
    w, halo = 160, 5
    for y0, x0 in ((0, 0), (n - w, n - w), (n // 2 - w // 2, n // 2 - w // 2), (311, 1500)):
        xw, oy, ox = _window(xs, y0, x0, w, halo)
        c = K.forward(pd, xw, net.scale)
        ref = c["y"][:, oy:oy + w, ox:ox + w] * net.scale
        e = rel(ys[:, y0:y0 + w, x0:x0 + w], ref)
        print(f"window ({y0}, {x0}): rel-L2 vs oracle {e:.2e}", flush=True)
        assert e < 1e-2, (y0, x0, e)


def test_backward_on_512_gridrec_pairs():
    """The training shape: two 512 x 512 gridrec pairs (90-angle input,
    900-angle target of the same phantoms), forward and backward on the GPU,
    against the oracle's backward on the GPU's activations."""
    inp, tgt = Lrn.make_pairs(2, 512, 90, 900, seed=21)
    net, pd, _, _ = make(9, scale=float(tgt.std()))
    net.forward(inp, train=True)
    net.backward(inp, tgt)
    torch.cuda.synchronize()
    x, t = inp.cpu().numpy(), tgt.cpu().numpy()
    acts = [bf16_bits_to_f32(a) for a in net._buffers(*x.shape, True)[0]]
    c = K.forward(pd, x, net.scale)
    yo = c["y"]
    for l in range(4):
        c[f"a{l + 1}"] = acts[l]
    c["y"] = net._buffers(*x.shape, True)[2].cpu().numpy()
    assert rel(c["y"], yo) < 1e-2  # the forward, end to end against the oracle's BF16 chain
    loss, g = K.loss_and_backward(pd, c, t, net.scale)
    print(f"loss GPU {float(net.loss.cpu()):.6e} oracle {loss:.6e}", flush=True)
    assert abs(float(net.loss.cpu()) - loss) <= 1e-5 * loss
    gg = Lrn.unflatten(net.grads.cpu().numpy())
    for k in g:
        e = rel(gg[k], g[k])
        print(f"grad {k}: rel-L2 {e:.2e}", flush=True)
        assert e < 1e-2, k


# the fused backward's 16 x 32 tiles, two rows per wave and eight-row halves:
# single pixels, rows and columns, one short of, exactly and one past a tile,
# several tiles and images
@pytest.mark.parametrize("n,H,W", [(1, 1, 1), (3, 1, 40), (2, 33, 1), (1, 15, 31), (2, 16, 32), (1, 17, 33), (5, 8, 64),
                                   (1, 50, 97)])
def test_backward_tile_edges(n, H, W):
    """Every gradient against the oracle's backward on the GPU's activations.
    Both round dz to bf16, so they differ where an accumulation order moves a
    value across a rounding boundary: one in some hundreds of values by one
    part in 2^8, far below the 2e-3 that one wrong halo pixel would exceed."""
    net, pd, x, t = make(n + H + W, n, H, W)
    xg, tg = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    net.forward(xg, train=True)
    net.backward(xg, tg)
    torch.cuda.synchronize()
    c = K.forward(pd, x, net.scale)
    for l, act in enumerate(net._buffers(*x.shape, True)[0]):
        c[f"a{l + 1}"] = bf16_bits_to_f32(act)
    c["y"] = net._buffers(*x.shape, True)[2].cpu().numpy()
    loss, g = K.loss_and_backward(pd, c, t, net.scale)
    assert abs(float(net.loss.cpu()) - loss) <= 1e-5 * loss
    gg = Lrn.unflatten(net.grads.cpu().numpy())
    for k in g:
        assert np.linalg.norm(gg[k] - g[k]) <= 2e-3 * np.linalg.norm(g[k]), k


# the last layer's backward: 8 x 32 tiles, more of them than workgroups, with
# ragged last rows and columns; a tile's rows and columns short of, exactly and
# past one
@pytest.mark.parametrize("n,H,W", [(1, 7, 31), (2, 8, 32), (1, 9, 33), (4, 130, 300)])
def test_last_layer_backward_tiles(n, H, W):
    """Loss and every gradient against the oracle's, within the bounds of
    test_backward_tile_edges and for its reasons; a second run gives the same
    bits."""
    test_backward_tile_edges(n, H, W)
    net, _, x, t = make(n + H + W, n, H, W)
    xg, tg = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    runs = []
    for _ in range(2):
        net.forward(xg, train=True)
        net.backward(xg, tg)
        torch.cuda.synchronize()
        runs.append((net.grads.clone(), net.loss.clone()))
    assert torch.equal(runs[0][0], runs[1][0]) and torch.equal(runs[0][1], runs[1][1])


# the forward kernel's strips of 56 columns (16-column groups, guard columns)
# and segments of rows (pairs of rows, odd ends): one short of, exactly and one
# past a strip, several segments, images smaller than the halo
FORWARD_SHAPES = [(1, 1, 1), (2, 3, 55), (1, 4, 56), (1, 17, 57), (1, 33, 113), (3, 130, 4), (1, 300, 61), (40, 18, 60)]


@pytest.mark.parametrize("shape", FORWARD_SHAPES)
def test_forward_strips_and_segments(shape):
    """Each layer against the convolution of the GPU's own previous activations:
    equal up to the rounding of a float sum at a bf16 boundary (tolerances of
    test_forward_layers_match_oracle); inference bitwise the training output."""
    net, pd, x, _ = make(sum(shape), *shape)
    xg = torch.from_numpy(x).cuda()
    y, stats = net.forward(xg, train=True)
    torch.cuda.synchronize()
    a = [bf16_bits_to_f32(t) for t in net._buffers(*shape, True)[0]]
    xn = x / np.float32(net.scale)
    prev = K.bf16(xn)[..., None]
    for l in range(4):
        w = K.bf16(pd[f"W{l + 1}"])
        w = w[:, None, :] if l == 0 else w
        e = K.bf16(np.maximum(K.conv3x3(prev, w) + pd[f"b{l + 1}"], 0.0)).astype(np.float32)
        tol = np.maximum(np.abs(e) * 2.0 ** -7, 1e-3 * np.sqrt(np.mean(e.astype(np.float64) ** 2)))
        d = ulp_diff(np.ascontiguousarray(a[l]), np.ascontiguousarray(e))
        assert np.mean(d > 0) < 0.01 and (np.abs(a[l] - e) <= tol).all(), l
        prev = a[l]
    r = K.conv3x3(prev, K.bf16(pd["W5"])[None])[..., 0] + pd["b5"][0]
    assert rel(y.cpu().numpy(), (xn + r) * net.scale) < 1e-5
    s = stats.cpu().numpy().astype(np.float64)
    assert np.allclose(s[:, 0], (r ** 2).reshape(shape[0], -1).sum(1), rtol=1e-4)
    y2, stats2 = net.infer(xg)
    torch.cuda.synchronize()
    assert torch.equal(y, y2) and torch.equal(stats, stats2)


def test_forward_aliased_activations():
    """gr_cnn_forward with a3 in a1's buffer and a4 in a2's: they end holding
    a3 and a4."""
    import ctypes as C

    from projects_amd import gridrec as gr

    net, _, x, _ = make(9, 2, 40, 70)
    xg = torch.from_numpy(x).cuda()
    y, _ = net.forward(xg, train=True)
    acts = net._buffers(2, 40, 70, True)[0]
    b = [torch.zeros_like(acts[0]) for _ in range(2)]
    y2 = torch.empty_like(xg)
    p = lambda t: C.c_void_p(t.data_ptr()) if t is not None else C.c_void_p(None)
    gr._check(gr.lib().gr_cnn_forward(p(net.params), p(net.packed), p(xg), 2, 40, 70, net.scale, p(b[0]), p(b[1]),
                                      p(b[0]), p(b[1]), p(y2), p(None), p(None), p(None), C.c_void_p(0)), "forward")
    torch.cuda.synchronize()
    assert torch.equal(y, y2) and torch.equal(b[0], acts[2]) and torch.equal(b[1], acts[3])


# outputs over the input: the forward kernel reads x with a halo of five pixels
# while other strips of 56 columns and segments of rows are written, so images of
# several of both, and of one
INPLACE_SHAPES = [(1, 20, 30), (2, 75, 130), (3, 300, 61), (1, 16, 300)]


@pytest.mark.parametrize("shape", INPLACE_SHAPES)
def test_forward_in_place(shape):
    """forward, infer and correct with out=x: bitwise the images, sums and
    choices of a separate output."""
    net, _, x, _ = make(sum(shape), *shape)
    xg = torch.from_numpy(x).cuda()
    for train in (True, False):
        y, s = net.forward(xg, train=train)
        y, s = y.clone(), s.clone()
        z = xg.clone()
        out, s2 = net.forward(z, out=z, train=train)
        torch.cuda.synchronize()
        assert out is z and torch.equal(z, y) and torch.equal(s, s2)
    z = xg.clone()
    net.infer(z, out=z)
    assert torch.equal(z, y)
    rel_norm = torch.sqrt(s[:, 0] / s[:, 1])
    for net.threshold in (float(rel_norm.min()), 0.0, 1e9):  # one, none, all kept
        y, used = net.correct(xg)
        z = xg.clone()
        out, used2 = net.correct(z, out=z)
        torch.cuda.synchronize()
        assert out is z and torch.equal(z, y) and torch.equal(used, used2)
        for i in range(shape[0]):
            assert bool(used[i]) or torch.equal(z[i], xg[i])


@pytest.mark.parametrize("shape", INPLACE_SHAPES)
def test_c_entries_in_place(shape):
    """The C entries with y or yn at x, or part of the way over it: bitwise the
    outputs of separate buffers, the activations and sums among them."""
    import ctypes as C

    from projects_amd import gridrec as gr

    net, _, x, _ = make(sum(shape), *shape)
    n, H, W = shape
    xg = torch.from_numpy(x).cuda()
    y0, s0 = net.forward(xg, train=True)
    acts, work, yn0, _ = net._buffers(n, H, W, True)
    y0, s0, yn0 = y0.clone(), s0.clone(), yn0.clone()
    a4 = acts[3].clone()
    L = gr.lib()
    p = lambda t: C.c_void_p(t.data_ptr()) if t is not None else C.c_void_p(None)
    npx = n * H * W

    def forward(xv, y, yn, a, st=None, wk=None):
        gr._check(L.gr_cnn_forward(p(net.params), p(net.packed), p(xv), n, H, W, net.scale, *[p(t) for t in a], p(y),
                                   p(yn), p(st), p(wk), C.c_void_p(gr._stream_handle(None))), "gr_cnn_forward")
        torch.cuda.synchronize()

    def room(shift):  # a copy of x and an output `shift` floats further on
        buf = torch.zeros(npx + abs(shift), device="cuda")
        xv = buf[max(-shift, 0):max(-shift, 0) + npx].view(shape)
        xv.copy_(xg)
        return xv, buf[max(shift, 0):max(shift, 0) + npx].view(shape)

    for shift in (0, 1, -W, npx // 2):
        xv, out = room(shift)
        forward(xv, out, None, acts)
        assert torch.equal(out, y0) and torch.equal(acts[3], a4), shift
        xv, out = room(shift)
        other, st = torch.empty_like(xg), torch.empty_like(s0)
        forward(xv, other, out, acts, st, work)
        assert torch.equal(out, yn0) and torch.equal(other, y0) and torch.equal(st, s0), shift
        xv, out = room(shift)
        forward(xv, out, other, [acts[0], acts[1], acts[0], acts[1]])
        assert torch.equal(out, y0) and torch.equal(other, yn0) and torch.equal(acts[1], a4), shift
        xv, out = room(shift)
        gr._check(L.gr_cnn_infer(p(net.params), p(net.packed), p(xv), n, H, W, net.scale, p(out), p(None), p(None),
                                 C.c_void_p(gr._stream_handle(None))), "gr_cnn_infer")
        torch.cuda.synchronize()
        assert torch.equal(out, y0), shift


def test_forward_in_place_captured():
    """In-place inference as a graph on a stream of its own: every replay, with
    other work in between, gives the eager images."""
    net, _, x, _ = make(4, 2, 75, 130)
    xg = torch.from_numpy(x).cuda()
    y, _ = net.forward(xg)
    y = y.clone()
    s = torch.cuda.Stream()
    z = xg.clone()
    s.wait_stream(torch.cuda.current_stream())
    net.forward(z, out=z, stream=s)
    s.synchronize()
    assert torch.equal(z, y)
    z.copy_(xg)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        net.forward(z, out=z)
    for _ in range(3):
        z.copy_(xg)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(z, y)
        torch.randn(1 << 20, device="cuda").mul_(2.0)
        net.forward(torch.ones_like(xg))
        torch.cuda.synchronize()


# one value whose square no float sum of a workgroup's pixels can hold beside
# theirs: 2^26 against squares below one
@pytest.mark.parametrize("n,H,W,hot", [(1, 8, 32, 0), (1, 8, 32, 255), (3, 40, 70, 4321), (40, 128, 128, 77)])
def test_loss_of_uneven_errors(n, H, W, hot):
    """The loss against a sum in 64 bits.  Sums in double round twice, to a
    workgroup's float partial and to the result, by 2^-24 each."""
    net = Lrn.Corrector(params=np.zeros(28353, np.float32), scale=1.0)  # yn = x
    x = np.random.default_rng(hot).uniform(0.5, 0.99, (n, H, W)).astype(np.float32)
    x.reshape(-1)[hot] = 8192.0
    xg, t = torch.from_numpy(x).cuda(), torch.zeros((n, H, W), device="cuda")
    net.forward(xg, train=True)
    net.backward(xg, t)
    torch.cuda.synchronize()
    loss = np.mean(x.astype(np.float64) ** 2)
    assert abs(float(net.loss.cpu()) - loss) <= 2.0 ** -23 * loss
    g = Lrn.unflatten(net.grads.cpu().numpy())
    db5 = np.sum(2.0 * x.astype(np.float64)) / x.size
    assert abs(float(g["b5"][0]) - db5) <= 2.0 ** -20 * np.sum(np.abs(2.0 * x)) / x.size


def test_forward_and_infer_keep_their_sums():
    """The sums forward() returned are still its image's after infer() on
    another, and the other way round."""
    net, _, x, _ = make(8, 2, 40, 70)
    a, b = torch.from_numpy(x).cuda(), torch.from_numpy(3.0 * x).cuda()
    want = [net.forward(v, train=True)[1].clone() for v in (a, b)]
    s1 = net.forward(a)[1]
    s2 = net.infer(b)[1]
    torch.cuda.synchronize()
    assert torch.equal(s1, want[0]) and torch.equal(s2, want[1])
    net.forward(b)
    torch.cuda.synchronize()
    assert torch.equal(s2, want[1])


# segments of eight rows at least, and more than 64 of them
@pytest.mark.parametrize("shape", [(1, 8, 8), (1, 9, 60), (2, 15, 57), (1, 2100, 20)])
def test_forward_short_segments(shape):
    test_forward_strips_and_segments(shape)


# the sums' partials stay within the documented work sizes, short segments or not
@pytest.mark.parametrize("shape", [(1, 8, 8), (3, 16, 32), (2, 40, 57), (1, 64, 64), (1, 256, 256), (1, 2100, 20), (2, 1100, 64)])
def test_infer_work_stays_in_its_size(shape):
    import ctypes as C

    from projects_amd import gridrec as gr

    net, _, x, _ = make(sum(shape), *shape)
    n, H, W = shape
    L = gr.lib()
    size = L.gr_cnn_infer_work_bytes(n, H, W)
    assert size == 8 * n * ((W + 31) // 32) * ((H + 15) // 16)
    xg = torch.from_numpy(x).cuda()
    work = torch.full((size + 65536,), 0x5A, dtype=torch.uint8, device="cuda")
    y, st = torch.empty_like(xg), torch.empty((n, 2), dtype=torch.float32, device="cuda")
    p = lambda t: C.c_void_p(t.data_ptr())
    gr._check(L.gr_cnn_infer(p(net.params), p(net.packed), p(xg), n, H, W, net.scale, p(y), p(st), p(work),
                             C.c_void_p(gr._stream_handle(None))), "gr_cnn_infer")
    torch.cuda.synchronize()
    assert bool((work[size:] == 0x5A).all())
    y1, s1 = net.forward(xg, train=True)
    torch.cuda.synchronize()
    assert torch.equal(y, y1) and torch.equal(st, s1)
