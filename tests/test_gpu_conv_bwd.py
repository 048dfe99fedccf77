"""Backward kernels of the network's layers against float64 sums on the CPU of
the same bfloat16 values.  Tolerances: every output is a float32 sum of n
products of bfloat16 values (exact in float32), so whatever its order it lies
within n 2^-24 of the exact sum, relative to the sum of the magnitudes."""
import ctypes as C

import pytest
import torch

from natrix_amd import _lib
from natrix_amd.learned import unet as U

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def _p(t):
    return C.c_void_p(t.data_ptr())


def _s():
    return C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _wgrad(x, dy, splits):
    n, h, w, ci = x.shape
    co = dy.shape[3]
    dw = torch.full((co, 9, ci), float("nan"), device="cuda")
    work = torch.full((splits * co * 9 * ci,), float("nan"), device="cuda")
    _lib.call("nx_conv3x3_wgrad", _p(x), _p(dy), _p(dw), _p(work), splits, n, h, w, ci, co, _s())
    return dw


def _taps(x):
    """x moved by each tap, zero outside the image: [9] of [N, H, W, C]."""
    n, h, w, _ = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    return [xp[:, t // 3:t // 3 + h, t % 3:t % 3 + w] for t in range(9)]


# tiles are 8 rows x 16 columns x 32 channels: one pixel, one tile exactly, one
# more and one less on each side, channels that do not fill a tile or need
# several, splits beyond the number of tiles
@pytest.mark.parametrize("n,h,w,ci,co,splits", [
    (1, 1, 1, 8, 8, 1), (1, 8, 16, 32, 32, 1), (2, 9, 17, 32, 64, 3), (3, 7, 15, 64, 32, 2),
    (1, 4, 4, 96, 32, 7), (2, 16, 33, 40, 24, 64), (1, 23, 31, 128, 96, 5),
    (2, 40, 48, 32, 32, 30)])
def test_wgrad_edges(gpu, n, h, w, ci, co, splits):
    g = torch.Generator().manual_seed(n + h * w + ci * co)
    x = torch.randn(n, h, w, ci, generator=g).to(BF)
    dy = torch.randn(n, h, w, co, generator=g).to(BF)
    dw = _wgrad(x.cuda(), dy.cuda(), splits).double().cpu()
    again = _wgrad(x.cuda(), dy.cuda(), splits).double().cpu()
    assert torch.equal(dw, again)
    d = dy.double().reshape(-1, co)
    for t, xt in enumerate(_taps(x.double())):
        xt = xt.reshape(-1, ci)
        ref, mag = d.t() @ xt, d.abs().t() @ xt.abs()
        assert bool(((dw[:, t] - ref).abs() <= n * h * w * 2.0 ** -24 * mag).all()), t


def test_wgrad_keeps_infinities_where_they_are(gpu):
    """An infinite activation in the last column and row reaches only the taps
    that see it there: nothing beyond the image multiplies it by zero."""
    n, h, w, ci, co = 1, 9, 13, 32, 32
    g = torch.Generator().manual_seed(5)
    x = torch.randn(n, h, w, ci, generator=g).to(BF)
    dy = torch.randn(n, h, w, co, generator=g).to(BF).abs() + 0.5
    x[0, h - 1, w - 1, 3] = float("inf")
    dw = _wgrad(x.cuda(), dy.to(BF).cuda(), 2).cpu()
    for t in range(9):
        # pixel (y, x) sees (h - 1, w - 1) at tap t if it is inside the image
        y, xx = h - 1 - (t // 3 - 1), w - 1 - (t % 3 - 1)
        seen = y < h and xx < w
        assert bool(torch.isinf(dw[:, t, 3]).all()) == seen, t
        assert bool(torch.isfinite(dw[:, t, :3]).all()) and bool(torch.isfinite(dw[:, t, 4:]).all())


@pytest.mark.parametrize("rows,c", [(1, 32), (63, 8), (64, 256), (65, 64), (1000, 24), (777, 5),
                                    (70000, 128), (300, 513)])
def test_row_passes(gpu, rows, c):
    """Column sums alone and with ReLU's gradient: the gradient bitwise, the sums
    within float32 summation; 5 and 513 channels take the one-channel form."""
    g = torch.Generator().manual_seed(rows + c)
    y = torch.randn(rows, c, generator=g).to(BF).relu()
    dy = torch.randn(rows, c, generator=g).to(BF)
    yd, dyd = y.cuda(), dy.cuda()
    dz = torch.full_like(dyd, float("nan"))
    db = torch.full((c,), float("nan"), device="cuda")
    work = torch.full((1024 * c,), float("nan"), device="cuda")
    _lib.call("nx_relu_bwd_colsum", _p(yd), _p(dyd), _p(dz), _p(db), _p(work), rows, c, _s())
    want = torch.where(y > 0, dy, torch.zeros_like(dy))
    assert torch.equal(dz.cpu(), want)
    out = torch.full((c,), float("nan"), device="cuda")
    _lib.call("nx_colsum", _p(dz), _p(out), _p(work), rows, c, _s())
    bound = rows * 2.0 ** -24 * want.double().abs().sum(0)
    for got in (db, out):
        assert bool(((got.double().cpu() - want.double().sum(0)).abs() <= bound).all())


@pytest.mark.parametrize("pixels,c", [(1, 32), (130, 32), (5000, 64), (999, 12)])
def test_head_backward(gpu, pixels, c):
    g = torch.Generator().manual_seed(pixels + c)
    x = torch.randn(1, 1, pixels, c, generator=g).to(BF)
    w, b = torch.randn(c, generator=g), torch.zeros(1)
    dout = torch.randn(1, 1, pixels, generator=g)
    xg, wg, bg = (t.cuda().requires_grad_(True) for t in (x, w, b))
    U.HeadFn.apply(xg, wg, bg).backward(dout.cuda())
    assert torch.equal(xg.grad.cpu(), (dout[..., None] * w).to(BF))
    terms = dout.double()[0, 0][:, None] * x.double()[0, 0]
    # one more rounding: a product of float32 and bfloat16 is not exact
    bound = (pixels + 1) * 2.0 ** -24 * terms.abs().sum(0)
    assert bool(((wg.grad.double().cpu() - terms.sum(0)).abs() <= bound).all())
    assert abs(float(bg.grad) - float(dout.double().sum())) <= \
        pixels * 2.0 ** -24 * float(dout.double().abs().sum())


@pytest.mark.parametrize("rows,c", [(3, 1032), (70, 2048), (130, 2056), (3, 15361), (65, 20000)])
def test_row_passes_of_many_channels(gpu, rows, c):
    """Rows as wide as a block and wider (256 threads of one or eight channels),
    beyond what a block's LDS would hold."""
    g = torch.Generator().manual_seed(rows + c)
    y = torch.randn(rows, c, generator=g).to(BF)
    dy = torch.randn(rows, c, generator=g).to(BF)
    w, dout = torch.randn(c, generator=g), torch.randn(rows, generator=g)
    yd, dyd, wd, dd = y.cuda(), dy.cuda(), w.cuda(), dout.cuda()
    dz = torch.full_like(dyd, float("nan"))
    db, dwb = (torch.full((c + i,), float("nan"), device="cuda") for i in (0, 1))
    work = torch.full((1024 * (c + 1),), float("nan"), device="cuda")
    _lib.call("nx_relu_bwd_colsum", _p(yd), _p(dyd), _p(dz), _p(db), _p(work), rows, c, _s())
    want = torch.where(y > 0, dy, torch.zeros_like(dy))
    assert torch.equal(dz.cpu(), want)
    unit = rows * 2.0 ** -24
    assert bool(((db.double().cpu() - want.double().sum(0)).abs() <=
                 unit * want.double().abs().sum(0)).all())
    _lib.call("nx_colsum", _p(dyd), _p(db), _p(work), rows, c, _s())
    assert bool(((db.double().cpu() - dy.double().sum(0)).abs() <=
                 unit * dy.double().abs().sum(0)).all())
    _lib.call("nx_head_bwd", _p(yd), _p(wd), _p(dd), _p(dz), _p(dwb), _p(work), rows, c, _s())
    assert torch.equal(dz.cpu(), (dout[:, None] * w).to(BF))
    terms = dout.double()[:, None] * y.double()
    assert bool(((dwb[:c].double().cpu() - terms.sum(0)).abs() <=
                 (rows + 1) * 2.0 ** -24 * terms.abs().sum(0)).all())
    assert abs(float(dwb[c]) - float(dout.double().sum())) <= unit * float(dout.double().abs().sum())


@pytest.mark.parametrize("n,h,w,ca,cb", [(1, 2, 2, 8, 16), (2, 6, 10, 64, 32), (1, 4, 2, 5, 3),
                                         (3, 8, 4, 24, 12)])
def test_movers_wide_and_single(gpu, n, h, w, ca, cb):
    """Pool, upsample and concat, forward and backward, with channel counts that
    take 16-byte accesses and counts that do not, against torch on the CPU."""
    g = torch.Generator().manual_seed(n * h * w + ca)
    x = torch.randn(n, h, w, ca, generator=g).to(BF)
    s = torch.randn(n, h, w, cb, generator=g).to(BF)
    d = torch.randn(n, h, w, ca, generator=g).to(BF)
    xg, sg = (t.cuda().requires_grad_(True) for t in (x, s))
    p = U.Pool2Fn.apply(xg)
    f = x.float().view(n, h // 2, 2, w // 2, 2, ca)
    want = (((f[:, :, 0, :, 0] + f[:, :, 0, :, 1]) + f[:, :, 1, :, 0]) + f[:, :, 1, :, 1]) * 0.25
    assert torch.equal(p.detach().cpu(), want.to(BF))
    u = U.Up2Fn.apply(p)
    assert torch.equal(u.detach().cpu(),
                       want.to(BF).repeat_interleave(2, 1).repeat_interleave(2, 2))
    y = U.ConcatFn.apply(u, sg)
    assert torch.equal(y.detach().cpu(), torch.cat([u.detach().cpu(), s], 3))
    dy = torch.cat([d, s], 3).contiguous()
    y.backward(dy.cuda())
    assert torch.equal(sg.grad.cpu(), s)
    e = d.float().view(n, h // 2, 2, w // 2, 2, ca)
    up = (((e[:, :, 0, :, 0] + e[:, :, 0, :, 1]) + e[:, :, 1, :, 0]) + e[:, :, 1, :, 1]).to(BF)
    pool = (up.float() * 0.25).to(BF)
    assert torch.equal(xg.grad.cpu(), pool.repeat_interleave(2, 1).repeat_interleave(2, 2))


def test_relu_gradient_alone(gpu):
    """nx_relu_bwd, the gradient without the bias sums that the layers take with it."""
    g = torch.Generator().manual_seed(2)
    y = torch.randn(3, 257, generator=g).to(BF).relu()
    dy = torch.randn(3, 257, generator=g).to(BF)
    yd, dyd = y.cuda(), dy.cuda()
    dz = torch.full_like(dyd, float("nan"))
    _lib.call("nx_relu_bwd", _p(yd), _p(dyd), _p(dz), dy.numel(), _s())
    assert torch.equal(dz.cpu(), torch.where(y > 0, dy, torch.zeros_like(dy)))
