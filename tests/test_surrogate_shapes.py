"""CPU trace of the operator network's forward and backward passes: every
kernel wrapper is replaced by a shape-checking stand-in, so a wiring mistake
(a tensor handed to the wrong level) fails here instead of on the GPU."""
import pytest


class _Shapes:
    """Stand-ins of the surrogate module's kernel calls (CPU tensors)."""

    def __init__(self, torch):
        self.t = torch
        self.seams = 0  # fused passes taken

    def conv3d(self, X, Wk, bias=None, relu=False, want_bf16=True, want_f32=True):
        assert X.dim() == 5 and Wk.shape == (27, Wk.shape[1], X.shape[4]), (X.shape, Wk.shape)
        assert X.shape[4] % 16 == 0 and Wk.shape[1] % 16 == 0
        Y = self.t.empty(X.shape[:4] + (Wk.shape[1],))
        return Y if want_f32 else None, Y.to(self.t.bfloat16)

    def conv3d_bwd_data(self, dY, Wk, want_bf16=True):
        assert dY.shape[4] == Wk.shape[1]
        return self.t.empty(dY.shape[:4] + (Wk.shape[2],)), None

    def conv3d_bwd_weight(self, X, dY, dW):
        assert X.shape[:4] == dY.shape[:4] and dW.shape == (27, dY.shape[4], X.shape[4])
        return dW

    def relu_bwd(self, dA, A, dA2=None):
        assert A is None or A.shape == dA.shape, (A.shape, dA.shape)
        assert dA2 is None or dA2.shape == dA.shape, (dA2.shape, dA.shape)
        return self.t.empty(dA.shape), self.t.empty(dA.shape)

    def bias_grad(self, dZ, db):
        assert db.numel() == dZ.shape[-1]

    def relu_bias_bwd(self, dA, A, db, dA2=None):
        self.bias_grad(dA, db)
        return self.relu_bwd(dA, A, dA2)[1]

    def relu_bias_net(self, dA, A, db, dA2=None, pooled=False):
        assert A.dtype == self.t.bfloat16 and db.numel() == A.shape[-1]
        assert (self.pool2(A) if pooled else A).shape == dA.shape, (A.shape, dA.shape)
        assert dA2 is None or (dA2.shape[:4] == A.shape[:4] and dA2.shape[4] >= A.shape[4])
        self.seams += 1
        return self.t.empty(A.shape)

    def pool2(self, X):
        assert all(s % 2 == 0 for s in X.shape[1:4])
        return self.t.empty(X.shape[:1] + tuple(s // 2 for s in X.shape[1:4]) + X.shape[4:])

    def pool2_bwd(self, dY):
        return self.t.empty(dY.shape[:1] + tuple(2 * s for s in dY.shape[1:4]) + dY.shape[4:])

    up2 = pool2_bwd

    def up2_bwd(self, dY):
        return self.pool2(dY)

    def up2_bwd_of(self, dY, c0):
        assert 0 < c0 < dY.shape[4]
        self.seams += 1
        return self.pool2(dY[..., c0:])

    def up2_concat(self, A, X):
        self.seams += 1
        return self.concat(A, self.up2(X))

    def concat(self, A, B):
        assert A.shape[:4] == B.shape[:4], (A.shape, B.shape)
        return self.t.empty(A.shape[:4] + (A.shape[4] + B.shape[4],))

    def split(self, dY, ca):
        return (self.t.empty(dY.shape[:4] + (ca,)),
                self.t.empty(dY.shape[:4] + (dY.shape[4] - ca,)))

    def mse(self, Y, target, loss):
        assert target.numel() == Y.numel() // Y.shape[-1]
        return self.t.empty(Y.shape)

    def to_bf16(self, a):
        return a.to(self.t.bfloat16)

    def zeros(self, shape, dtype=None):
        return self.t.zeros(shape)


@pytest.mark.parametrize("channels,window", [((16, 32), (8, 8, 8)), ((16, 32, 32), (16, 32, 32)),
                                             ((32, 64, 128, 128), (32, 64, 64))])
def test_unet_pass_shapes(monkeypatch, channels, window):
    torch = pytest.importorskip("torch")
    import surrogate as S
    f = _Shapes(torch)
    for name in ("conv3d", "conv3d_bwd_data", "conv3d_bwd_weight", "relu_bwd", "bias_grad",
                 "relu_bias_bwd", "pool2", "pool2_bwd", "up2", "up2_bwd", "concat", "split", "mse",
                 "to_bf16", "relu_bias_net", "up2_bwd_of", "up2_concat"):
        monkeypatch.setattr(S, name, getattr(f, name))
    monkeypatch.setattr(S, "_zeros", f.zeros)
    monkeypatch.setattr(torch.Tensor, "cuda", lambda self, *a, **k: self)
    net = S.UNet(channels=channels, seed=0)
    X = torch.empty((2,) + window + (16,), dtype=torch.bfloat16)
    Y = net.forward(X)
    assert Y.shape == (2,) + window + (16,)
    net.backward(torch.empty(Y.shape))
    # the passes a device runs: two seams a decoder level, a backward pass a
    # layer but the head
    assert f.seams == 2 * (len(channels) - 1) + len(net.layers()) - 1


def test_seam_wrappers_check_their_operands(monkeypatch):
    """relu_bias_net and up2_bwd_of hand raw pointers to kernels that index
    every operand by one shape: operands of other shapes, dtypes or strides
    are refused before a launch (CPU tensors, a library that records it)."""
    torch = pytest.importorskip("torch")
    import surrogate as S

    class Lib:
        launched = 0

        def __getattr__(self, name):
            def call(*a):
                self.launched += 1
                return 0
            return call

    lib = Lib()
    monkeypatch.setattr(S.N, "lib", lambda: lib)
    monkeypatch.setattr(S, "_stream", lambda: None)

    def check(t, dtype, name):  # S._check, but for the device
        if t.dtype != dtype or not t.is_contiguous():
            raise ValueError(name)

    monkeypatch.setattr(S, "_check", check)
    f = lambda *s: torch.zeros(s)  # noqa: E731
    A = f(2, 4, 6, 8, 32).bfloat16()
    dA, half, wide, db = f(2, 4, 6, 8, 32), f(2, 2, 3, 4, 32), f(2, 4, 6, 8, 96), f(32)
    for k, ok in enumerate([(dA, A, db), (dA, A, db, dA), (dA, A, db, wide),
                            (half, A, db, wide, True), (half, A, db, None, True)]):
        S.relu_bias_net(*ok)
        assert lib.launched == k + 1
    odd = f(1, 3, 4, 4, 16)
    lib.launched = 0
    for bad in [(half, A, db), (dA, A, db, None, True), (f(1, 4, 6, 8, 32), A, db),
                (f(2, 4, 6, 8, 16), A, db), (f(2 * 4 * 6 * 8 * 32), A, db),
                (dA, A.float(), db), (dA, A.transpose(2, 3), db), (dA, A, f(16)),
                (dA, A, db.double()), (dA, A, db, half), (dA, A, db, f(2, 4, 6, 8, 16)),
                (dA, A, db, wide.bfloat16()), (dA, A, db, wide[..., :64]),
                (dA, A, db, f(2, 4, 6, 8)), (half, A, db, half, True),
                (f(1, 1, 2, 2, 16), odd.bfloat16(), f(16), None, True)]:
        with pytest.raises(ValueError):
            S.relu_bias_net(*bad)
    for dY, c0 in [(wide, 96), (wide, -1), (wide, 200), (odd, 0), (wide[..., 32:], 0)]:
        with pytest.raises(ValueError):
            S.up2_bwd_of(dY, c0)
    assert lib.launched == 0
    assert S.up2_bwd_of(wide, 32).shape == (2, 2, 3, 4, 64) and lib.launched == 1
