"""Which kernel a convolution takes (gm_conv3d_plan, host code only)."""
import ctypes
import os

import pytest

import _native as N
from test_gpu_conv import MARCH_TILES, WGRAD_TAPS, WGRAD_TILES


def _plan(shape, kind=0):
    if not os.path.exists(N.LIB_PATH):
        pytest.skip("libgomelt.so is not built (make -C go-melt_amd/csrc)")
    out = (ctypes.c_int32 * 7)()
    N.check(N.lib().gm_conv3d_plan(kind, (ctypes.c_int32 * 6)(*shape), out))
    return tuple(out)


def test_march_tiles_cover_the_kernel():
    """The GPU test's shapes take every tile shape, with one z segment and
    with several, and none divides its tile."""
    seen = set()
    for s in MARCH_TILES:
        kernel, xt, yw, nt, wv, step, nz = _plan(s)
        assert kernel == 2, s
        assert s[3] % xt and s[2] % (wv * (16 // xt) * yw), s
        seen.add((xt, yw, nt, wv, step, nz > 1))
    tiles = {(16, 2, 2, 8, 9), (16, 4, 1, 4, 9), (16, 2, 1, 4, 9), (8, 1, 2, 4, 9),
             (8, 1, 1, 4, 9), (16, 2, 2, 8, 3), (16, 1, 4, 8, 1), (16, 1, 2, 8, 3),
             (16, 1, 2, 4, 3), (16, 2, 1, 4, 3), (8, 1, 2, 4, 3), (8, 1, 1, 4, 3)}
    assert seen == {t + (many,) for t in tiles for many in (False, True)}


# images smaller than a column's tile, or just past one: padding them cost up
# to 49 times the tap-by-tap kernel's time
@pytest.mark.parametrize("shape,kernel", [
    ((4096, 1, 1, 1, 128, 128), 1), ((2048, 2, 2, 2, 64, 64), 1), ((512, 4, 4, 2, 256, 128), 1),
    ((64, 256, 1, 1, 192, 64), 1), ((8, 17, 17, 17, 256, 128), 1),
    ((20000000, 1, 1, 1, 32, 32), 1), ((3, 13, 27, 35, 48, 80), 0), ((4, 8, 16, 16, 16, 32), 1),
    ((16, 32, 64, 64, 32, 32), 2), ((16, 32, 64, 64, 96, 32), 2), ((16, 16, 32, 32, 192, 64), 2),
    ((16, 4, 8, 8, 128, 128), 2), ((1, 32, 64, 64, 32, 32), 2)])
def test_forward_kernel_by_shape(shape, kernel):
    assert _plan(shape)[0] == kernel


def test_weight_gradient_shapes_cover_the_kernels():
    seen = set()
    for s in WGRAD_TILES:
        kernel, xt, it, _, _, _, nz = _plan(s, 1)
        assert kernel == 2 and s[3] % xt and s[2] % (64 // xt), s
        seen.add((xt, it, nz > 1))
    assert seen == {(xt, it, many) for xt in (8, 16) for it in (1, 2) for many in (False, True)}
    assert [_plan(s, 1)[0] for s in WGRAD_TAPS] == [1, 1, 1, 1, 1, 1, 0]


@pytest.mark.parametrize("shape,kernel", [
    ((4096, 1, 1, 1, 128, 128), 1), ((2048, 2, 2, 2, 256, 128), 1), ((512, 4, 4, 4, 192, 64), 1),
    ((864, 9, 1, 1, 48, 256), 0), ((1, 130, 512, 512, 32, 32), 1), ((3, 13, 27, 35, 48, 80), 2),
    ((16, 32, 64, 64, 32, 32), 2), ((16, 32, 64, 64, 96, 32), 2), ((16, 16, 32, 32, 64, 64), 2),
    ((16, 8, 16, 16, 128, 128), 2), ((16, 4, 8, 8, 128, 128), 2)])
def test_weight_gradient_kernel_by_shape(shape, kernel):
    assert _plan(shape, 1)[0] == kernel
