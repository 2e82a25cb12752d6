"""GPU convolution kernels of the learned L3 operator (BF16 MFMA, FP32
accumulation) against the FP64 oracle (oracle/conv_oracle.py) on the same
bf16-rounded inputs; tolerances stated per test."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def S():
    import torch
    import _native as N
    N.init_device()
    import surrogate as S
    return S


def _dev_bf16(a):
    import torch
    from oracle import conv_oracle as CO
    bits = CO.bf16_bits(np.ascontiguousarray(a, np.float32))
    return torch.from_numpy(bits.view(np.int16)).view(torch.bfloat16).cuda()


def _rel(g, r):
    return float(np.max(np.abs(g - r)) / max(np.max(np.abs(r)), 1e-30))


# the kernels chosen by channel counts: 16-channel K stages (cin 16, 48), the
# pipelined 32-channel stages with 128 x 32 tiles (cout <= 32) and 64 x 64
# tiles, the weight gradient's 32 x 32, 32-multiple and general kernels
SHAPES = [(2, 5, 6, 7, 16, 32), (1, 8, 8, 4, 32, 16), (1, 3, 3, 3, 16, 48), (1, 9, 7, 11, 48, 80),
          (2, 4, 6, 8, 32, 32), (1, 5, 6, 7, 64, 96), (1, 7, 5, 9, 96, 32),
          (1, 6, 8, 10, 16, 32), (1, 5, 7, 9, 32, 16), (2, 3, 4, 5, 16, 16),
          # 128-voxel blocks of whole rows, W from 2 to 64
          (2, 3, 4, 32, 32, 32), (1, 3, 2, 64, 64, 16), (1, 2, 64, 2, 96, 32),
          # a larger volume: 32768 voxels, 128 outputs
          (2, 8, 32, 64, 32, 128),
          # 2^18 voxels: 4096-voxel parts in the weight gradient, and the
          # forward kernel with one sub-stage per barrier pair (the smaller
          # volumes above take three): 256 x 32 blocks of 64 x 32 waves (up to
          # 32 outputs, also with 16 input channels), 64 x 64 blocks beyond
          (1, 8, 128, 256, 32, 32), (1, 8, 128, 256, 16, 32), (1, 8, 128, 256, 64, 64),
          (2, 8, 64, 128, 128, 128)]


@pytest.mark.parametrize("shape", SHAPES)
def test_conv_forward(S, shape):
    """Y = conv(X; W) + b, relu off and on: 1e-5 of max |Y| (FP32 sums of
    exact bf16 products)."""
    import torch
    from oracle import conv_oracle as CO
    nb, D, H, W, ci, co = shape
    rng = np.random.default_rng(sum(shape))
    X = CO.bf16_round(rng.standard_normal((nb, D, H, W, ci)).astype(np.float32))
    Wk = CO.bf16_round((0.2 * rng.standard_normal((27, co, ci))).astype(np.float32))
    b = rng.standard_normal(co).astype(np.float32)
    ref = CO.conv3d(X, Wk, b)
    for relu in (False, True):
        Y, Yb = S.conv3d(_dev_bf16(X), _dev_bf16(Wk), torch.from_numpy(b).cuda(), relu=relu)
        torch.cuda.synchronize()
        r = np.maximum(ref, 0) if relu else ref
        assert _rel(Y.cpu().numpy(), r) < 1e-5
        # the bf16 copy is the rounded FP32 output
        yb = Yb.float().cpu().numpy()
        np.testing.assert_array_equal(yb, CO.bf16_round(Y.cpu().numpy()))


@pytest.mark.parametrize("shape", SHAPES)
def test_conv_gradients(S, shape):
    """Input and weight gradients against the oracle: 1e-5 of the max; the
    weight gradient is added to what dW holds."""
    import torch
    from oracle import conv_oracle as CO
    nb, D, H, W, ci, co = shape
    rng = np.random.default_rng(7 + sum(shape))
    X = CO.bf16_round(rng.standard_normal((nb, D, H, W, ci)).astype(np.float32))
    Wk = CO.bf16_round((0.2 * rng.standard_normal((27, co, ci))).astype(np.float32))
    dY = CO.bf16_round(rng.standard_normal((nb, D, H, W, co)).astype(np.float32))
    dX, _ = S.conv3d_bwd_data(_dev_bf16(dY), _dev_bf16(Wk))
    torch.cuda.synchronize()
    assert _rel(dX.cpu().numpy(), CO.conv3d_bwd_data(dY, Wk)) < 1e-5
    base = rng.standard_normal((27, co, ci)).astype(np.float32)
    dW = torch.from_numpy(base.copy()).cuda()
    S.conv3d_bwd_weight(_dev_bf16(X), _dev_bf16(dY), dW)
    torch.cuda.synchronize()
    ref = CO.conv3d_bwd_weight(X, dY)
    assert _rel(dW.cpu().numpy() - base, ref) < 1e-5


# edges of the passes as a network calls them: partial tiles in x, y and z, 8-
# and 16-wide tiles, output counts off the tiles, one plane, one voxel, 352
# channels (the tap-by-tap kernel).  Most forward passes here have few tiles
# and split their sum; MARCH_TILES holds the marching kernel's own edges
MARCH = [(1, 3, 19, 33, 32, 48), (2, 5, 17, 8, 64, 96), (1, 33, 9, 40, 32, 80),
         (1, 1, 1, 1, 32, 16), (3, 1, 30, 23, 64, 32), (1, 7, 34, 17, 160, 32),
         (2, 4, 12, 20, 256, 64), (1, 2, 9, 16, 352, 16), (5, 17, 33, 40, 64, 64),
         (4, 9, 40, 47, 32, 32), (3, 10, 33, 31, 128, 128), (4, 9, 33, 31, 192, 64)]


@pytest.mark.parametrize("shape", MARCH)
def test_conv_march_edges(S, shape):
    """Forward and input gradient against the oracle: 1e-5 of the max (FP32
    sums of exact bf16 products), and operands that are only 8-byte aligned,
    which take another kernel, within twice that."""
    import ctypes
    import torch
    import _native as N
    from oracle import conv_oracle as CO
    nb, D, H, W, ci, co = shape
    rng = np.random.default_rng(11 + sum(shape))
    X = CO.bf16_round(rng.standard_normal((nb, D, H, W, ci)).astype(np.float32))
    Wk = CO.bf16_round((0.2 * rng.standard_normal((27, co, ci))).astype(np.float32))
    b = rng.standard_normal(co).astype(np.float32)
    Xd, Wd, bd = _dev_bf16(X), _dev_bf16(Wk), torch.from_numpy(b).cuda()
    Y, Yb = S.conv3d(Xd, Wd, bd, relu=True)
    ref = np.maximum(CO.conv3d(X, Wk, b), 0)
    assert _rel(Y.cpu().numpy(), ref) < 1e-5
    np.testing.assert_array_equal(Yb.float().cpu().numpy(), CO.bf16_round(Y.cpu().numpy()))
    off = torch.empty(Xd.numel() + 4, dtype=torch.bfloat16, device="cuda")
    off[4:] = Xd.reshape(-1)
    Yo = torch.empty_like(Y)
    p = lambda t, o=0: ctypes.c_void_p(t.data_ptr() + o)  # noqa: E731
    N.check(N.lib().gm_conv3d_fwd((ctypes.c_int32 * 6)(*shape), p(off, 8), p(Wd), p(bd), 1,
                                  p(Yo), None, None))
    torch.cuda.synchronize()
    assert _rel(Yo.cpu().numpy(), Y.cpu().numpy()) < 2e-5
    dY = CO.bf16_round(rng.standard_normal((nb, D, H, W, co)).astype(np.float32))
    dX, _ = S.conv3d_bwd_data(_dev_bf16(dY), Wd, want_bf16=False)
    torch.cuda.synchronize()
    assert _rel(dX.cpu().numpy(), CO.conv3d_bwd_data(dY, Wk)) < 1e-5


# the weight gradient's column kernel on every tile shape, on one z segment and
# on several, with ragged columns; then the tap-by-tap ones on many small
# images (32 and 16 channels, 32 outputs, multiples of 32, others), the number
# of voxels off their stages (test_conv_plan checks the kernels)
WGRAD_TILES = [(1, 1, 14, 38, 16, 16), (1, 9, 13, 18, 48, 16), (7, 1, 17, 17, 32, 64),
               (2, 9, 17, 18, 128, 32), (1, 1, 5, 25, 48, 16), (1, 9, 5, 27, 16, 48),
               (3, 1, 9, 17, 96, 80), (5, 9, 9, 17, 32, 80)]
WGRAD_TAPS = [(300, 1, 1, 1, 32, 32), (201, 2, 1, 1, 32, 16), (601, 1, 2, 2, 16, 32),
              (901, 1, 2, 1, 16, 16), (901, 2, 1, 2, 96, 32), (131, 2, 2, 1, 64, 96),
              (701, 1, 1, 2, 48, 80)]


@pytest.mark.parametrize("shape", WGRAD_TILES + WGRAD_TAPS)
def test_conv_weight_gradient_kernels(S, shape):
    """Added to what dW holds: 1e-5 of the max against the oracle (FP32 sums
    of exact bf16 products)."""
    import torch
    from oracle import conv_oracle as CO
    nb, D, H, W, ci, co = shape
    rng = np.random.default_rng(19 + sum(shape))
    X = CO.bf16_round(rng.standard_normal((nb, D, H, W, ci)).astype(np.float32))
    dY = CO.bf16_round(rng.standard_normal((nb, D, H, W, co)).astype(np.float32))
    base = rng.standard_normal((27, co, ci)).astype(np.float32)
    dW = torch.from_numpy(base.copy()).cuda()
    S.conv3d_bwd_weight(_dev_bf16(X), _dev_bf16(dY), dW)
    torch.cuda.synchronize()
    assert _rel(dW.cpu().numpy() - base, CO.conv3d_bwd_weight(X, dY)) < 1e-5


def test_conv_weight_gradient_large_image(S):
    """An image of more than 2^31 bytes: gradients at a few voxels, the first
    and last and those around byte 2^31 among them, against their own sums."""
    import torch
    D, H, W, ci, co = 130, 512, 512, 32, 16
    gen = torch.Generator(device="cuda").manual_seed(2)
    X = torch.randn((1, D, H, W, ci), generator=gen, device="cuda", dtype=torch.bfloat16)
    assert X.numel() * 2 > 2 ** 31
    dY = torch.zeros((1, D, H, W, co), dtype=torch.bfloat16, device="cuda")
    edge = 2 ** 31 // (2 * ci)
    v = torch.cat([torch.tensor([0, edge - 1, edge, D * H * W - 1]),
                   torch.randint(0, D * H * W, (300,), generator=torch.Generator().manual_seed(3))]
                  ).unique().cuda()
    g = torch.randn((len(v), co), generator=gen, device="cuda").bfloat16()
    dY.view(-1, co)[v] = g
    dW = torch.zeros((27, co, ci), device="cuda")
    S.conv3d_bwd_weight(X, dY, dW)
    z, y, x = v // (H * W), v // W % H, v % W
    for tap in range(27):
        zz, yy, xx = z + tap // 9 - 1, y + tap // 3 % 3 - 1, x + tap % 3 - 1
        ok = (zz >= 0) & (zz < D) & (yy >= 0) & (yy < H) & (xx >= 0) & (xx < W)
        rows = X.view(-1, ci)[((zz * H + yy) * W + xx)[ok]].double()
        ref = (g[ok].double().t() @ rows).cpu().numpy()
        assert _rel(dW[tap].cpu().numpy(), ref) < 1e-5, tap


# the weight gradient's edges: partial 16 x 4 and 8 x 8 columns, segments of
# one plane and cut volumes, an odd number of columns, channel tiles off 32,
# one voxel
WGRAD = [(1, 1, 1, 1, 16, 16), (1, 1, 5, 17, 32, 16), (3, 2, 7, 8, 64, 48), (1, 37, 9, 15, 16, 80),
         (2, 70, 6, 18, 32, 32), (5, 17, 33, 21, 48, 32), (3, 9, 13, 34, 96, 64)]


@pytest.mark.parametrize("shape", WGRAD)
def test_conv_weight_gradient_edges(S, shape):
    """Added to what dW holds: 1e-5 of the max against the oracle (FP32 sums
    of exact bf16 products), and operands that are only 8-byte aligned, which
    take another kernel, within twice that."""
    import ctypes
    import torch
    import _native as N
    from oracle import conv_oracle as CO
    nb, D, H, W, ci, co = shape
    rng = np.random.default_rng(13 + sum(shape))
    X = CO.bf16_round(rng.standard_normal((nb, D, H, W, ci)).astype(np.float32))
    dY = CO.bf16_round(rng.standard_normal((nb, D, H, W, co)).astype(np.float32))
    base = rng.standard_normal((27, co, ci)).astype(np.float32)
    ref = CO.conv3d_bwd_weight(X, dY)
    Xd, dYd = _dev_bf16(X), _dev_bf16(dY)
    dW = torch.from_numpy(base.copy()).cuda()
    S.conv3d_bwd_weight(Xd, dYd, dW)
    off = torch.empty(Xd.numel() + 4, dtype=torch.bfloat16, device="cuda")
    off[4:] = Xd.reshape(-1)
    dWo = torch.zeros((27, co, ci), dtype=torch.float32, device="cuda")
    N.check(N.lib().gm_conv3d_bwd_weight((ctypes.c_int32 * 6)(*shape),
                                         ctypes.c_void_p(off.data_ptr() + 8),
                                         ctypes.c_void_p(dYd.data_ptr()),
                                         ctypes.c_void_p(dWo.data_ptr()), None))
    torch.cuda.synchronize()
    assert _rel(dW.cpu().numpy() - base, ref) < 1e-5
    assert _rel(dWo.cpu().numpy(), ref) < 2e-5


# every tile shape of the marching kernel, on one z segment and on several
# (test_conv_plan checks that), with ragged x and y edges
MARCH_TILES = [
    (1, 1, 6, 5, 64, 16), (1, 4, 6, 7, 64, 16), (1, 1, 5, 5, 32, 16), (1, 4, 11, 5, 32, 16),
    (15, 1, 39, 5, 160, 64), (11, 11, 10, 5, 64, 96), (11, 1, 25, 5, 32, 96),
    (9, 4, 10, 5, 32, 64), (15, 1, 19, 10, 64, 96), (3, 8, 18, 9, 64, 64),
    (16, 1, 10, 20, 64, 96), (11, 8, 5, 17, 64, 32), (11, 1, 41, 6, 160, 128),
    (2, 12, 50, 35, 64, 64), (14, 1, 9, 10, 64, 96), (3, 4, 9, 10, 64, 96),
    (9, 1, 10, 9, 32, 128), (6, 4, 9, 9, 32, 48), (10, 1, 59, 9, 64, 128),
    (3, 35, 57, 9, 64, 32), (15, 1, 33, 9, 32, 128), (4, 15, 17, 10, 32, 96),
    (13, 1, 35, 9, 32, 64), (3, 16, 9, 10, 32, 48)]


@pytest.mark.parametrize("shape", MARCH_TILES)
def test_conv_march_tiles(S, shape):
    """The marching kernel without a workspace: FP32 output within 1e-5 of the
    oracle's max (FP32 sums of exact bf16 products), the bf16 outputs (with
    and without the FP32 one) its rounding, and the bits of the tap-by-tap
    kernel, which an output off 16 bytes takes."""
    import ctypes
    import torch
    import _native as N
    from oracle import conv_oracle as CO
    nb, D, H, W, ci, co = shape
    rng = np.random.default_rng(17 + sum(shape))
    X = CO.bf16_round(rng.standard_normal((nb, D, H, W, ci)).astype(np.float32))
    Wk = CO.bf16_round((0.2 * rng.standard_normal((27, co, ci))).astype(np.float32))
    b = rng.standard_normal(co).astype(np.float32)
    Xd, Wd, bd = _dev_bf16(X), _dev_bf16(Wk), torch.from_numpy(b).cuda()
    out = torch.full((nb * D * H * W * co + 2,), -7.0, device="cuda")
    Y = torch.empty((nb, D, H, W, co), device="cuda")
    Yb, Yo = (torch.empty(Y.shape, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    p = lambda t, o=0: ctypes.c_void_p(t.data_ptr() + o)  # noqa: E731
    sh, L = (ctypes.c_int32 * 6)(*shape), N.lib()
    N.check(L.gm_conv3d_fwd(sh, p(Xd), p(Wd), p(bd), 1, p(Y), p(Yb), None))
    N.check(L.gm_conv3d_fwd_bf16(sh, p(Xd), p(Wd), p(bd), 1, p(Yo), None, 0, None))
    N.check(L.gm_conv3d_fwd(sh, p(Xd), p(Wd), p(bd), 1, p(out, 8), None, None))
    torch.cuda.synchronize()
    Yn = Y.cpu().numpy()
    assert _rel(Yn, np.maximum(CO.conv3d(X, Wk, b), 0)) < 1e-5
    np.testing.assert_array_equal(Yb.float().cpu().numpy(), CO.bf16_round(Yn))
    np.testing.assert_array_equal(Yo.float().cpu().numpy(), CO.bf16_round(Yn))
    out = out.cpu().numpy()
    np.testing.assert_array_equal(out[2:], Yn.reshape(-1))
    assert (out[:2] == -7.0).all()


def test_two_layer_training_gradients(S):
    """Gradients of L = 0.5 |conv(relu(conv(X)+b1))+b2 - T|^2 through the
    kernels: with the oracle fed the same bf16-rounded intermediates, 1e-5;
    against the oracle's all-FP64 gradients, 3e-2 (bf16 activations)."""
    import torch
    from oracle import conv_oracle as CO
    rng = np.random.default_rng(5)
    nb, D, H, W, ci, ch, co = 2, 6, 5, 4, 16, 32, 16
    X = CO.bf16_round(rng.standard_normal((nb, D, H, W, ci)).astype(np.float32))
    W1 = CO.bf16_round((0.1 * rng.standard_normal((27, ch, ci))).astype(np.float32))
    W2 = CO.bf16_round((0.1 * rng.standard_normal((27, co, ch))).astype(np.float32))
    b1 = (0.1 * rng.standard_normal(ch)).astype(np.float32)
    b2 = (0.1 * rng.standard_normal(co)).astype(np.float32)
    T = rng.standard_normal((nb, D, H, W, co)).astype(np.float32)
    Z1, A1b = S.conv3d(_dev_bf16(X), _dev_bf16(W1), torch.from_numpy(b1).cuda(), relu=True)
    Y, _ = S.conv3d(A1b, _dev_bf16(W2), torch.from_numpy(b2).cuda())
    R = Y - torch.from_numpy(T).cuda()
    Rb = S.to_bf16(R.contiguous())
    dW2 = torch.zeros((27, co, ch), dtype=torch.float32, device="cuda")
    S.conv3d_bwd_weight(A1b, Rb, dW2)
    dA1, _ = S.conv3d_bwd_data(Rb, _dev_bf16(W2))
    dZ1 = dA1 * (Z1 > 0)
    dZ1b = S.to_bf16(dZ1.contiguous())
    dW1 = torch.zeros((27, ch, ci), dtype=torch.float32, device="cuda")
    S.conv3d_bwd_weight(_dev_bf16(X), dZ1b, dW1)
    torch.cuda.synchronize()
    # matched: the oracle on the GPU's own bf16 intermediates
    a1 = A1b.float().cpu().numpy()
    rb = Rb.float().cpu().numpy()
    dz1b = dZ1b.float().cpu().numpy()
    assert _rel(dW2.cpu().numpy(), CO.conv3d_bwd_weight(a1, rb)) < 1e-5
    assert _rel(dA1.cpu().numpy(), CO.conv3d_bwd_data(rb, W2)) < 1e-5
    assert _rel(dW1.cpu().numpy(), CO.conv3d_bwd_weight(X, dz1b)) < 1e-5
    # unmatched: all-FP64 chain rule of the oracle
    _, (gW1, gb1, gW2, gb2), _ = CO.two_layer_loss(X, W1, b1, W2, b2, T)
    assert _rel(dW2.cpu().numpy(), gW2) < 3e-2
    assert _rel(dW1.cpu().numpy(), gW1) < 3e-2


def test_adam(S):
    import torch
    from oracle import conv_oracle as CO
    rng = np.random.default_rng(9)
    n = 5000
    w = rng.standard_normal(n).astype(np.float32)
    m = np.zeros(n, np.float32)
    v = np.zeros(n, np.float32)
    tw, tm, tv = (torch.from_numpy(a.copy()).cuda() for a in (w, m, v))
    twb = torch.empty(n, dtype=torch.bfloat16, device="cuda")
    lr, b1, b2, eps = 1e-2, 0.9, 0.999, 1e-8
    w64, m64, v64 = w.astype(np.float64), m.astype(np.float64), v.astype(np.float64)
    for step in (1, 2, 3):
        g = rng.standard_normal(n).astype(np.float32)
        S.adam(tw, twb, torch.from_numpy(g).cuda(), tm, tv, step, lr, b1, b2, eps)
        m64 = b1 * m64 + (1 - b1) * g
        v64 = b2 * v64 + (1 - b2) * g.astype(np.float64) ** 2
        w64 = w64 - lr * (m64 / (1 - b1 ** step)) / (np.sqrt(v64 / (1 - b2 ** step)) + eps)
    torch.cuda.synchronize()
    assert float(np.max(np.abs(tw.cpu().numpy() - w64))) < 1e-5
    np.testing.assert_array_equal(twb.float().cpu().numpy(), CO.bf16_round(tw.cpu().numpy()))
