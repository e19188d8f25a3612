"""The warm-start network's kernels at the edges of their tiles: remainders of
rows, columns and channels, the smallest and largest tile forms, non-finite
values.  References are the operations' definitions in 64 bits on the CPU."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _call(name, *args):
    import torch
    from imexlb._lib import lib
    rc = getattr(lib(), "imexlb_nn_" + name)(
        *[C.c_void_p(a.data_ptr()) if isinstance(a, torch.Tensor) else a for a in args], None)
    assert rc == 0, (name, rc)


def _conv64(x, w, b=None):
    N, ci, H, W = x.shape
    xp = np.zeros((N, ci, H + 2, W + 2))
    xp[:, :, 1:-1, 1:-1] = x
    y = np.zeros((N, w.shape[0], H, W))
    for k in range(9):
        y += np.einsum("oc,nchw->nohw", w[:, :, k // 3, k % 3], xp[:, :, k // 3:k // 3 + H, k % 3:k % 3 + W])
    return y if b is None else y + b[None, :, None, None]


# tile forms: 16-column (W <= 16), 4 x 32 (few blocks), 8 x 32 (512 blocks and more)
SHAPES = [(1, 1, 1, 1, 1), (2, 3, 5, 9, 7), (1, 15, 31, 8, 16), (1, 16, 32, 4, 17), (2, 17, 33, 5, 33),
          (1, 33, 65, 3, 32), (3, 8, 3, 2, 70), (1, 100, 4, 1, 40), (20, 5, 31, 61, 97), (9, 17, 65, 121, 64)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("relu", [0, 1])
def test_conv3x3_at_tile_edges(shape, relu):
    import torch
    N, ci, co, H, W = shape
    print(f"[nn] conv3x3 {shape} relu {relu}", flush=True)
    rng = np.random.default_rng(5)
    x = rng.normal(0, 1, (N, ci, H, W)).astype(np.float32)
    w = rng.normal(0, 1, (co, ci, 3, 3)).astype(np.float32)
    b = rng.normal(0, 1, co).astype(np.float32)
    xd, wd, bd = (torch.tensor(v, device="cuda") for v in (x, w, b))
    out = torch.full((N, co, H, W), 7.0, device="cuda")
    _call("conv3x3", xd, wd, bd, out, N, ci, co, H, W, relu)
    ref = _conv64(x.astype(np.float64), w.astype(np.float64), b.astype(np.float64))
    size = _conv64(np.abs(x).astype(np.float64), np.abs(w).astype(np.float64), np.abs(b).astype(np.float64))
    # FP32 summation bound: one rounding of 2^-24 per term, and a few more
    tol = (9 * ci + 8) * 2.0 ** -24 * size
    err = np.abs(out.cpu().numpy() - (np.maximum(ref, 0) if relu else ref))
    assert (err <= tol).all(), (err / tol).max()


@pytest.mark.parametrize("shape", [(1, 5, 6, 20, 40), (1, 18, 34, 9, 16), (4, 3, 7, 200, 180)])
def test_conv3x3_non_finite_values(shape):
    """Infinities, NaN and overflowing products behave as in FP32."""
    import torch
    N, ci, co, H, W = shape
    print(f"[nn] conv3x3 non-finite {shape}", flush=True)
    rng = np.random.default_rng(6)
    x = rng.normal(0, 1, (N, ci, H, W)).astype(np.float32)
    w = rng.integers(-3, 4, (co, ci, 3, 3)).astype(np.float32)
    x[0, 0, 3, 3], x[0, 1, H - 1, W - 1], x[0, 2, 5, 9] = np.nan, np.inf, -np.inf
    x[N - 1, 1, 7, 12] = 3.4e38
    out = torch.empty((N, co, H, W), device="cuda")
    _call("conv3x3", torch.tensor(x, device="cuda"), torch.tensor(w, device="cuda"), None, out, N, ci, co, H, W, 0)
    with np.errstate(all="ignore"):
        ref = _conv64(x.astype(np.float64), w.astype(np.float64))
        small = np.where(np.isfinite(x) & (np.abs(x) < 1e30), x, 0).astype(np.float64)
        ref32 = ref.astype(np.float32)
    got = out.cpu().numpy()
    big = np.abs(ref) > 1e30  # products of 3.4e38: overflow depends on the order of the sum
    assert (np.isnan(got) == np.isnan(ref))[~big].all()
    assert np.array_equal(got[np.isinf(ref)], ref32[np.isinf(ref)])
    plain = np.isfinite(ref) & ~big
    size = _conv64(np.abs(small), np.abs(w).astype(np.float64))
    assert (np.abs(got[plain] - ref[plain]) <= ((9 * ci + 8) * 2.0 ** -24 * size)[plain]).all()


# channel groups of 16 and 32 on either side and past them, ragged tiles, one
# and two tile halves, tile counts around the reduction's 32 loads in flight
DW_SHAPES = [(1, 1, 1, 1, 1), (3, 15, 16, 8, 16), (2, 16, 17, 9, 17), (2, 17, 15, 16, 33), (1, 33, 34, 31, 5),
             (2, 20, 40, 260, 190), (1, 3, 65, 65, 500), (2, 40, 9, 100, 300)]


@pytest.mark.parametrize("shape", DW_SHAPES)
def test_weight_gradient_at_tile_edges(shape):
    import torch
    from imexlb._lib import lib
    N, ci, co, H, W = shape
    print(f"[nn] conv3x3_dw {shape}", flush=True)
    rng = np.random.default_rng(7)
    x = rng.normal(0, 1, (N, ci, H, W)).astype(np.float32)
    g = rng.normal(0, 1, (N, co, H, W)).astype(np.float32)
    start = rng.normal(0, 1, (co, ci, 3, 3)).astype(np.float32)

    def dw64(x, g):
        xp = np.zeros((N, ci, H + 2, W + 2))
        xp[:, :, 1:-1, 1:-1] = x
        r = np.zeros((co, ci, 3, 3))
        for k in range(9):
            s = xp[:, :, k // 3:k // 3 + H, k % 3:k % 3 + W].transpose(1, 0, 2, 3).reshape(ci, -1)
            r[:, :, k // 3, k % 3] = g.astype(np.float64).transpose(1, 0, 2, 3).reshape(co, -1) @ s.T
        return r

    xd, gd = torch.tensor(x, device="cuda"), torch.tensor(g, device="cuda")
    n = lib().imexlb_nn_conv3x3_dw_work(ci, co, H, W)
    work = torch.empty(n, device="cuda")
    dw = torch.tensor(start, device="cuda")
    _call("conv3x3_dw_ordered", xd, gd, dw, work, n, N, ci, co, H, W)
    again = torch.tensor(start, device="cuda")
    _call("conv3x3_dw_ordered_noalloc", xd, gd, again, N, ci, co, H, W)
    assert torch.equal(dw, again)
    loose = torch.tensor(start, device="cuda")
    _call("conv3x3_dw", xd, gd, loose, N, ci, co, H, W)
    # one rounding of 2^-24 per product and per tile
    tiles = -(-H // 16) * -(-W // 16)
    tol = (N * H * W + tiles + 4) * 2.0 ** -24 * (dw64(np.abs(x), np.abs(g)) + np.abs(start))
    for got in (dw, loose):
        err = np.abs(got.cpu().numpy() - (dw64(x, g) + start))
        assert (err <= tol).all(), (err / tol).max()


# rows of 256 pixels: one ragged, exactly one, more than a batch of loads in
# flight, images shorter than a batch
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 3, 15, 17), (3, 5, 16, 16), (2, 7, 131, 129), (5, 4, 16, 112),
                                   (1, 33, 16, 1040)])
def test_bias_gradient(shape):
    import torch
    N, C_, H, W = shape
    rng = np.random.default_rng(8)
    g = rng.normal(0, 1, shape).astype(np.float32)
    db = torch.empty(C_, device="cuda")
    _call("bias_grad", torch.tensor(g, device="cuda"), db, N, C_, H, W)
    # the order of the sum: thread t adds pixels t, t + 256, ..., then a tree
    rows = -(-H * W // 256)
    v = np.zeros((N, C_, rows * 256), np.float32)
    v[:, :, :H * W] = g.reshape(N, C_, -1)
    v = v.reshape(N, C_, rows, 256).transpose(1, 0, 2, 3).reshape(C_, N * rows, 256)
    s = np.zeros((C_, 256), np.float32)
    for k in range(N * rows):
        s += v[:, k]
    o = 128
    while o:
        s[:, :o] += s[:, o:2 * o]
        o //= 2
    assert np.array_equal(db.cpu().numpy(), s[:, 0])


@pytest.mark.parametrize("n", [1, 255, 1024, 1025, 131072, 131073, 400003])
def test_mse(n):
    import torch
    rng = np.random.default_rng(9)
    p, t = (rng.normal(0, 1, n).astype(np.float32) for _ in range(2))
    g, loss = torch.empty(n, device="cuda"), torch.full((1,), 0.5, device="cuda")
    _call("mse", torch.tensor(p, device="cuda"), torch.tensor(t, device="cuda"), g, n, loss)
    d = p - t
    assert np.array_equal(g.cpu().numpy(), np.float32(2) * d / np.float32(n))
    ref = 0.5 + np.mean(d.astype(np.float64) ** 2)
    # each term rounded twice, at most 128 additions to the loss
    assert abs(loss.item() - ref) <= 130 * 2.0 ** -24 * ref


@pytest.mark.parametrize("shape", [(1, 1, 1, 1, 1), (2, 5, 33, 9, 33), (1, 40, 7, 6, 16), (1, 17, 64, 70, 31),
                                   (9, 32, 65, 121, 64)])
@pytest.mark.parametrize("gated", [False, True])
def test_data_gradient_equals_flipped_convolution(shape, gated):
    import torch
    N, ci, co, H, W = shape
    g = torch.Generator("cuda").manual_seed(10)
    r = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    dz, w, gate = r(N, co, H, W), r(co, ci, 3, 3), r(N, ci + 5, H, W)
    wt, ref, dx = torch.empty(ci, co, 3, 3, device="cuda"), r(N, ci, H, W), r(N, ci, H, W)
    _call("flip_weights", w, wt, ci, co)
    _call("conv3x3", dz, wt, None, ref, N, co, ci, H, W, 0)
    _call("conv3x3_dgrad", dz, w, gate if gated else None, ci + 5, 3, dx, N, ci, co, H, W)
    if gated:
        ref = torch.where(gate[:, 3:3 + ci] > 0, ref, torch.zeros_like(ref))
    assert torch.equal(dx, ref)


@pytest.mark.parametrize("shape", [(2, 5, 33, 9, 33), (1, 40, 70, 6, 16), (3, 17, 18, 70, 31)])
def test_joined_entries_equal_their_parts(shape):
    """Output into a channel slice; weight and bias gradient in one launch."""
    import torch
    from imexlb._lib import lib
    N, ci, co, H, W = shape
    g = torch.Generator("cuda").manual_seed(11)
    r = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    x, w, b, dz = r(N, ci, H, W), r(co, ci, 3, 3), r(co), r(N, co, H, W)
    ref, wide = torch.empty(N, co, H, W, device="cuda"), r(N, co + 9, H, W)
    keep = wide.clone()
    _call("conv3x3", x, w, b, ref, N, ci, co, H, W, 1)
    _call("conv3x3_into", x, w, b, wide, co + 9, 4, N, ci, co, H, W, 1)
    assert torch.equal(wide[:, 4:4 + co], ref)
    assert torch.equal(wide[:, :4], keep[:, :4]) and torch.equal(wide[:, 4 + co:], keep[:, 4 + co:])
    n = lib().imexlb_nn_conv3x3_dw_work(ci, co, H, W)
    work = torch.empty(n, device="cuda")
    dw, dw2 = torch.zeros_like(w), torch.zeros_like(w)
    db, db2 = torch.empty_like(b), torch.empty_like(b)
    _call("conv3x3_dw_ordered", x, dz, dw, work, n, N, ci, co, H, W)
    _call("bias_grad", dz, db, N, co, H, W)
    _call("conv3x3_grads", x, dz, dw2, db2, work, n, N, ci, co, H, W)
    assert torch.equal(dw, dw2) and torch.equal(db, db2)


# odd and even widths, one pixel, rows longer than a wave's 128 pixels, more
# rows than blocks of a small launch; buffers that start off 16 bytes
@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 3, 5, 7), (1, 4, 3, 64), (2, 5, 2, 131), (1, 3, 9, 258)])
@pytest.mark.parametrize("shift", [0, 1])
def test_pooling_and_upsampling(shape, shift):
    import torch
    N, C_, h, w = shape
    g = torch.Generator("cuda").manual_seed(12)

    def r(*s):
        n = int(np.prod(s))
        return torch.randn(n + shift, generator=g, device="cuda")[shift:].view(s)

    f = np.float32
    big, low = r(N, C_ + 6, 2 * h, 2 * w), r(N, C_, h, w)
    B, Lo = big.cpu().numpy(), low.cpu().numpy()
    sl = B[:, 4:4 + C_]
    quad = ((sl[..., 0::2, 0::2] + sl[..., 0::2, 1::2]) + (sl[..., 1::2, 0::2] + sl[..., 1::2, 1::2]))
    out = r(N, C_, h, w)
    _call("pool2_from", big, C_ + 6, 4, out, N, C_, h, w)
    assert np.array_equal(out.cpu().numpy(), f(0.25) * quad)
    gate = r(N, C_ + 2, h, w)
    _call("up2_bwd_gate", big, C_ + 6, 4, gate, C_ + 2, 1, out, N, C_, h, w)
    assert np.array_equal(out.cpu().numpy(), np.where(gate.cpu().numpy()[:, 1:1 + C_] > 0, quad, f(0)))
    _call("up2_bwd", big, out, N, C_, h, w, C_ + 6, 4)
    assert np.array_equal(out.cpu().numpy(), quad)
    din, gate2 = r(N, C_, 2 * h, 2 * w), r(N, C_ + 1, 2 * h, 2 * w)
    spread = f(0.25) * Lo.repeat(2, 2).repeat(2, 3)
    _call("pool2_bwd", low, din, N, C_, h, w)
    assert np.array_equal(din.cpu().numpy(), spread)
    _call("pool2_bwd_join", low, big, C_ + 6, 4, gate2, C_ + 1, 1, din, N, C_, h, w)
    assert np.array_equal(din.cpu().numpy(), np.where(gate2.cpu().numpy()[:, 1:] > 0, spread + sl, f(0)))
    wide = r(N, C_ + 3, 2 * h, 2 * w)
    keep = wide.cpu().numpy()
    _call("up2", low, wide, N, C_, h, w, C_ + 3, 2)
    keep[:, 2:2 + C_] = Lo.repeat(2, 2).repeat(2, 3)
    assert np.array_equal(wide.cpu().numpy(), keep)


# the tiles: 16 columns (narrow images, few and many blocks), 32 columns four
# rows with chunks ahead, 8 rows, 16 rows, 64 channels a block; chunks of 16
# and 32 channels, one to nine of them; ragged sizes and channel counts
BF16_SHAPES = [(1, 16, 3, 1, 1), (1, 48, 40, 9, 16), (80, 32, 8, 41, 13), (2, 96, 32, 5, 33), (1, 288, 33, 7, 40),
               (3, 16, 31, 130, 190), (9, 32, 64, 130, 62), (12, 80, 30, 130, 200), (16, 32, 32, 134, 260)]


def _bf16_ref(x, w, b):
    """Exact products in FP64 of bf16 values (torch's float64 on the CPU)."""
    return _conv64(x.astype(np.float64), w.astype(np.float64), b.astype(np.float64))


@pytest.mark.parametrize("shape", BF16_SHAPES)
def test_bf16_convolution_at_tile_edges(shape):
    import torch
    N, ci, co, H, W = shape
    print(f"[nn] conv3x3_bf16 {shape}", flush=True)
    g = torch.Generator().manual_seed(13)
    x = torch.randn(N, H, W, ci, generator=g).to(torch.bfloat16)
    w = (torch.randn(co, ci, 3, 3, generator=g) / np.sqrt(9 * ci)).to(torch.bfloat16).float()
    b = torch.randn(co, generator=g)
    cop = 32 * -(-co // 32)
    wp = torch.empty(ci * 9 * cop, dtype=torch.bfloat16, device="cuda")
    wd, bd, xd = w.cuda(), b.cuda(), x.cuda()
    _call("pack_weights_bf16", wd, wp, ci, co, ci, cop)
    few = max(1, min(N, 2))  # (the reference of a few images; the rest by repetition)
    xd[few:] = xd[:1]
    ref = _bf16_ref(xd[:few].cpu().float().permute(0, 3, 1, 2).numpy(), w.numpy(), b.numpy())
    size = _bf16_ref(xd[:few].cpu().float().abs().permute(0, 3, 1, 2).numpy(), w.abs().numpy(), b.abs().numpy())
    wide = torch.full((N, H, W, co + 3), 7.0, dtype=torch.bfloat16, device="cuda")
    f32 = torch.empty(N, co, H, W, device="cuda")
    _call("conv3x3_bf16", xd, wp, bd, wide, N, ci, co, cop, H, W, co + 3, 2, 0, 0)
    _call("conv3x3_bf16", xd, wp, bd, f32, N, ci, co, cop, H, W, 0, 0, 1, 1)
    # FP32 sums of exact products, then one rounding to bf16
    tol = (9 * ci + 8) * 2.0 ** -24 * size
    got = f32[:few].cpu().numpy()
    assert (np.abs(got - np.maximum(ref, 0)) <= tol).all()
    full = wide.float().cpu().numpy().transpose(0, 3, 1, 2)
    assert (full[:, :2] == 7).all() and (full[:, 2 + co:] == 7).all()
    assert (np.abs(full[:few, 2:2 + co] - ref) <= 2.0 ** -8 * np.abs(ref) + 2 * tol).all()
    for k in range(few, N):
        assert torch.equal(f32[k], f32[0]) and torch.equal(wide[k], wide[0])


@pytest.mark.parametrize("shape", [(1, 32, 16, 16, 4, 6), (1, 16, 32, 40, 34, 18), (2, 64, 32, 32, 66, 70),
                                   (9, 64, 64, 64, 130, 66), (5, 32, 32, 96, 260, 130)])
def test_bf16_joined_layer_equals_its_parts(shape):
    """Upsampled and skip channels from their own buffers, and the pooled
    output, against the separate calls: the same bits."""
    import torch
    N, cl, cs, co, H, W = shape
    print(f"[nn] conv3x3_bf16_join {shape}", flush=True)
    g = torch.Generator("cuda").manual_seed(14)
    bf = lambda *s: torch.randn(s, generator=g, device="cuda").to(torch.bfloat16)  # noqa: E731
    low, skip, b = bf(N, H // 2, W // 2, cl), bf(N, H, W, cs), torch.randn(co, generator=g, device="cuda")
    ci, cop = cl + cs, 32 * -(-co // 32)
    wp = torch.empty(ci * 9 * cop, dtype=torch.bfloat16, device="cuda")
    _call("pack_weights_bf16", torch.randn(co, ci, 3, 3, generator=g, device="cuda") / np.sqrt(9 * ci), wp, ci, co, ci,
          cop)
    cat = torch.empty(N, H, W, ci, dtype=torch.bfloat16, device="cuda")
    _call("up2_bf16", low, cat, N, cl, H // 2, W // 2, ci, 0)
    cat[..., cl:] = skip
    ref, out = bf(N, H, W, co), bf(N, H, W, co)
    pref, pool = bf(N, H // 2, W // 2, co), bf(N, H // 2, W // 2, co)
    _call("conv3x3_bf16", cat, wp, b, ref, N, ci, co, cop, H, W, co, 0, 1, 0)
    _call("pool2_bf16", ref, pref, N, co, H // 2, W // 2, co, 0)
    _call("conv3x3_bf16_join", low, cl, skip, cs, wp, b, out, pool, N, co, cop, H, W, co, 0, 1, 0)
    assert torch.equal(out, ref) and torch.equal(pool, pref)
