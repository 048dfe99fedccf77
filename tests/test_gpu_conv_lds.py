"""The LDS-staged convolution against float64 and, bitwise, against the
single-wave kernel it stands beside (reached through one split of the split
entry point, whose K order is the same)."""
import ctypes as C

import pytest
import torch

from natrix_amd import _lib

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def _p(t):
    return C.c_void_p(t.data_ptr())


def _s():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


# tiles are 16 or 8 rows x 16 columns x 32, 64 or 128 output channels: one
# pixel, one tile, one more and one less on a side; every channel pair of the
# network and pairs that take the narrow forms
@pytest.mark.parametrize("n,h,w,ci,co", [
    (1, 1, 1, 32, 32), (1, 16, 16, 32, 64), (2, 17, 15, 64, 64), (1, 15, 33, 64, 32),
    (1, 9, 17, 64, 192), (2, 16, 20, 96, 32), (1, 8, 16, 96, 64), (1, 7, 31, 128, 32),
    (1, 12, 18, 128, 64), (2, 8, 8, 128, 256), (1, 20, 16, 128, 384), (1, 9, 15, 192, 64),
    (1, 17, 17, 192, 128), (3, 4, 4, 256, 256), (1, 18, 31, 256, 64), (1, 11, 19, 384, 128),
    (1, 8, 17, 384, 64), (1, 6, 10, 192, 96)])
@pytest.mark.parametrize("relu", [0, 1])
def test_conv_lds(gpu, n, h, w, ci, co, relu):
    g = torch.Generator().manual_seed(n * h * w + ci + co)
    x = torch.randn(n, h, w, ci, generator=g).to(BF)
    wt = (torch.randn(co, 9, ci, generator=g) / (3 * ci ** 0.5)).to(BF)
    b = torch.randn(co, generator=g)
    y = torch.full((n, h, w, co), float("nan"), dtype=BF, device="cuda")
    z = torch.full_like(y, float("nan"))
    work = torch.empty(n * h * w * co, device="cuda")
    xd, wd, bd = x.cuda(), wt.cuda(), b.cuda()
    _lib.call("nx_conv3x3_fwd", _p(xd), _p(wd), _p(bd), _p(y), n, h, w, ci, co, relu, _s())
    _lib.call("nx_conv3x3_fwd_split", _p(xd), _p(wd), _p(bd), _p(z), _p(work), 1, n, h, w, ci, co,
              relu, _s())
    assert torch.equal(y, z)
    # every product is exact in float32; 9 ci of them are summed, one bias
    # added and the sum rounded to bfloat16
    xp = torch.nn.functional.pad(x.double(), (0, 0, 1, 1, 1, 1))
    ref, mag = b.double().expand(n, h, w, co).clone(), b.double().abs().expand(n, h, w, co).clone()
    for t in range(9):
        xt = xp[:, t // 3:t // 3 + h, t % 3:t % 3 + w]
        ref += xt @ wt[:, t].double().t()
        mag += xt.abs() @ wt[:, t].double().abs().t()
    ref = ref.relu() if relu else ref
    err = (y.double().cpu() - ref).abs()
    assert bool((err <= 9 * ci * 2.0 ** -24 * mag + 2.0 ** -8 * ref.abs()).all())


@pytest.mark.parametrize("n,h,w,ci,co", [(1, 6, 7, 128, 128), (1, 1, 43, 128, 64),
                                         (5, 1, 17, 256, 256), (2, 1, 43, 256, 128)])
def test_either_side_of_the_pixel_line(gpu, n, h, w, ci, co):
    """The last image that is not staged and the first that is (cin / 3 pixels)."""
    test_conv_lds(gpu, n, h, w, ci, co, 1)


def test_conv_without_bias_and_infinities(gpu):
    """No bias (the input gradient's call); an infinite pixel reaches its 3 x 3
    neighbourhood and nothing else."""
    n, h, w, ci, co = 1, 19, 21, 32, 32
    x = torch.zeros(n, h, w, ci, dtype=BF, device="cuda")
    x[0, 16, 16, 5] = float("inf")
    wt = torch.ones(co, 9, ci, dtype=BF, device="cuda")
    y = torch.full((n, h, w, co), float("nan"), dtype=BF, device="cuda")
    _lib.call("nx_conv3x3_fwd", _p(x), _p(wt), None, _p(y), n, h, w, ci, co, 0, _s())
    want = torch.zeros(n, h, w, co, dtype=BF)
    want[0, 15:18, 15:18] = float("inf")
    assert torch.equal(y.cpu(), want)
