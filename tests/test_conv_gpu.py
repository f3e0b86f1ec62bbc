"""Parity of the HIP convolution path (through the C-ABI and through the
operator) with the oracle and with torch's conv2d on the CPU.

Tolerance: 1e-3 relative to the largest magnitude of the expected tensor (the
bound the task states for the convolution) for the fp32 products and for the
split-bf16 products (two bf16 per operand, three products); 1e-2 for plain bf16
operands, whose rounding alone (2^-9 per operand) puts a sum of products about
2e-3 off.  im2col / col2im are copies and sums in the reference's order and
must be bit-exact."""
import ctypes

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from mobulaop_amd import native
from oracle import conv as oracle
import abi_util as abi

pytestmark = pytest.mark.gpu
CONV_TOL = 1e-3
# option "conv_compute" -> tolerance
MODES = {'fp32': (0, 1e-3), 'bf16': (1, 1e-2), 'bf16x3': (2, 1e-3)}


@pytest.fixture(params=sorted(MODES))
def compute(request):
    """Runs the test once per way of forming the products; yields the tolerance."""
    mode, tol = MODES[request.param]
    native.set_option('conv_compute', mode)
    yield tol
    native.set_option('conv_compute', 0)


def _ci(*vals):
    return [ctypes.c_int(int(v)) for v in vals]


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _call(name, *args, extents=()):
    lib = native.library()
    native.begin_call(None, list(extents))
    getattr(lib, name)(ctypes.c_int(0), *args)
    native.end_call(name)


def _close(got, want, what, tol=CONV_TOL):
    got, want = got.detach().cpu().double().numpy(), want.detach().cpu().double().numpy()
    assert got.shape == want.shape and np.isfinite(got).all(), what
    err = np.abs(got - want).max()
    assert err <= tol * max(np.abs(want).max(), 1e-30), '{}: max abs error {} vs scale {}'.format(
        what, err, np.abs(want).max())


@pytest.mark.parametrize('case', [
    (2, 3, 4, (2, 3), (0, 1), (1, 2), (1, 1)),
    (5, 17, 13, (3, 3), (1, 1), (1, 1), (1, 1)),
    (3, 20, 16, (3, 2), (2, 0), (2, 1), (1, 2)),
    (2, 12, 12, (3, 3), (2, 2), (1, 2), (2, 2)),
])
def test_unfold_and_fold_bit_exact(case):
    C, H, W, kernel, pad, stride, dil = case
    rng = np.random.default_rng(21)
    im = rng.standard_normal((C, H, W)).astype(np.float32)
    want_col = oracle.im2col(im, kernel, pad, stride, dil)
    OH, OW = want_col.shape[1:]
    geo = _ci(H, W, kernel[0], kernel[1], pad[0], pad[1], stride[0], stride[1], dil[0], dil[1], OH, OW)
    d_im = torch.from_numpy(im).cuda()
    d_col = torch.full(want_col.shape, float('nan'), device='cuda')
    _call('im2col_341af5d3', ctypes.c_int(d_col.numel()), _ptr(d_im), *geo, _ptr(d_col))
    assert np.array_equal(d_col.cpu().numpy(), want_col)
    g = rng.standard_normal(want_col.shape).astype(np.float32)
    d_g = torch.from_numpy(g).cuda()
    d_back = torch.full(im.shape, float('nan'), device='cuda')
    _call('col2im_341af5d3', ctypes.c_int(d_back.numel()), _ptr(d_g), *geo, _ptr(d_back))
    assert np.array_equal(d_back.cpu().numpy(), oracle.col2im(g, im.shape, kernel, pad, stride, dil))


SHAPES = [
    # N, C, H, W, D, kernel, pad, stride, dilation
    (2, 2, 3, 4, 3, (2, 3), (0, 1), (1, 2), (1, 1)),       # opzoo/Convolution/test_conv.py:10-14
    (1, 3, 9, 9, 5, (3, 3), (1, 1), (1, 1), (1, 1)),
    (3, 8, 17, 13, 20, (3, 2), (2, 1), (2, 1), (1, 2)),     # ragged tiles, dilation
    (2, 64, 28, 28, 160, (3, 3), (1, 1), (1, 1), (1, 1)),   # several tiles in every dimension
    (4, 32, 30, 30, 140, (5, 5), (2, 2), (2, 2), (1, 1)),
    (5, 16, 14, 14, 24, (1, 1), (0, 0), (1, 1), (1, 1)),    # pointwise
    (4, 38, 4, 3, 166, (1, 3), (2, 0), (2, 1), (1, 1)),     # 4 x 1 outputs: a step of the weight gradient spans images
    (9, 5, 2, 2, 7, (2, 2), (0, 0), (1, 1), (1, 1)),        # one output pixel per image
]


@pytest.mark.parametrize('shape', SHAPES)
def test_convolution_through_the_abi(shape, compute):
    N, C, H, W, D, kernel, pad, stride, dil = shape
    tol = compute
    g = torch.Generator().manual_seed(31)
    x = torch.randn(N, C, H, W, generator=g)
    w = torch.randn(D, C, *kernel, generator=g) * 0.1
    b = torch.randn(D, generator=g)
    xr, wr, br = (t.clone().requires_grad_(True) for t in (x, w, b))
    y_ref = F.conv2d(xr, wr, br, stride=stride, padding=pad, dilation=dil)
    dy = torch.randn(y_ref.shape, generator=g)
    y_ref.backward(dy)
    if x.numel() * D < 5e6:   # the oracle agrees with torch at sizes it finishes quickly
        y_o = oracle.conv2d_forward(x.numpy(), w.numpy(), b.numpy(), pad, stride, dil)
        assert np.abs(y_o - y_ref.detach().numpy()).max() <= 1e-4 * max(1.0, float(y_ref.detach().abs().max()))
    xd, wd, bd, dyd = x.cuda(), w.cuda(), b.cuda(), dy.cuda()
    geo = _ci(N, C, H, W, D, kernel[0], kernel[1], pad[0], pad[1], stride[0], stride[1], dil[0], dil[1])
    y = torch.full(y_ref.shape, float('nan'), device='cuda')
    _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(xd), _ptr(wd), _ptr(bd), ctypes.c_int(1),
          *geo, _ptr(y))
    _close(y, y_ref, 'y', tol)
    dx = torch.full(x.shape, float('nan'), device='cuda')
    _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dyd), _ptr(wd), ctypes.c_int(0),
          *geo, _ptr(dx))
    _close(dx, xr.grad, 'dx', tol)
    dw = torch.full(w.shape, float('nan'), device='cuda')
    _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw.numel()), _ptr(dyd), _ptr(xd), ctypes.c_int(0),
          *geo, _ptr(dw))
    _close(dw, wr.grad, 'dw', tol)
    db = torch.full((D,), float('nan'), device='cuda')
    _call('conv2d_backward_bias_cd239a08', ctypes.c_int(D), _ptr(dyd), ctypes.c_int(0), ctypes.c_int(N),
          ctypes.c_int(y.shape[2] * y.shape[3]), _ptr(db))
    _close(db, br.grad, 'db', tol)
    # accumulate variants add to what is there
    dx2 = torch.ones_like(dx)
    _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx2.numel()), _ptr(dyd), _ptr(wd), ctypes.c_int(1),
          *geo, _ptr(dx2))
    _close(dx2 - 1, xr.grad, 'dx accumulate', tol)
    dw2 = torch.ones_like(dw)
    _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw2.numel()), _ptr(dyd), _ptr(xd), ctypes.c_int(1),
          *geo, _ptr(dw2))
    _close(dw2 - 1, wr.grad, 'dw accumulate', tol)


def test_operator_matches_torch_autograd(mobula):
    mobula.op.load('Convolution')
    torch.manual_seed(41)
    x = torch.randn(2, 2, 3, 4, device='cuda', requires_grad=True)       # test_conv.py:10-14
    w = torch.randn(3, 2, 2, 3, device='cuda', requires_grad=True)
    b = torch.randn(3, device='cuda', requires_grad=True)
    y = mobula.op.Conv2D(x=x, weight=w, bias=b, channels=3, kernel_size=(2, 3), strides=(1, 2), padding=(0, 1))
    dy = torch.rand_like(y)
    y.backward(dy)
    xr, wr, br = (t.detach().cpu().requires_grad_(True) for t in (x, w, b))
    yr = F.conv2d(xr, wr, br, stride=(1, 2), padding=(0, 1))
    yr.backward(dy.cpu())
    for got, want, what in ((y, yr, 'y'), (x.grad, xr.grad, 'dx'), (w.grad, wr.grad, 'dw'), (b.grad, br.grad, 'db')):
        _close(got, want, what)
    # without bias
    y2 = mobula.op.Conv2D(x=x.detach(), weight=w.detach(), channels=3, kernel_size=(2, 3), strides=(1, 2),
                          padding=(0, 1))
    _close(y2, F.conv2d(xr.detach(), wr.detach(), None, stride=(1, 2), padding=(0, 1)), 'y without bias')


def test_resnet_block_shape_properties(compute):
    # C_in = C_out = 256, 3x3, pad 1 at a reduced batch and map: linearity in x and
    # the adjoint identity <conv(x), dy> = <x, dx> tie forward and backward together
    N, C, H, W, D = 4, 256, 28, 28, 256
    g = torch.Generator().manual_seed(51)
    x = torch.randn(N, C, H, W, generator=g).cuda()
    w = (torch.randn(D, C, 3, 3, generator=g) * (2.0 / (C * 9)) ** 0.5).cuda()
    dy = torch.randn(N, D, H, W, generator=g).cuda()
    geo = _ci(N, C, H, W, D, 3, 3, 1, 1, 1, 1, 1, 1)
    y = torch.empty(N, D, H, W, device='cuda')
    _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(x), _ptr(w), _ptr(w), ctypes.c_int(0), *geo,
          _ptr(y))
    _close(y, F.conv2d(x.cpu(), w.cpu(), padding=1), 'y', compute)
    dx = torch.empty_like(x)
    _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dy), _ptr(w), ctypes.c_int(0), *geo,
          _ptr(dx))
    dw = torch.empty_like(w)
    _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw.numel()), _ptr(dy), _ptr(x), ctypes.c_int(0), *geo,
          _ptr(dw))
    lhs = float((y.double() * dy.double()).sum())
    if compute <= 1e-3:
        bound = 1e-4 * abs(lhs)
    else:
        # operands rounded to bf16: the three sums round different tensors, and the terms
        # cancel in lhs itself, so the scale is the one of Cauchy-Schwarz
        bound = 1e-3 * float(y.double().norm() * dy.double().norm())
    assert abs(lhs - float((x.double() * dx.double()).sum())) <= bound
    assert abs(lhs - float((w.double() * dw.double()).sum())) <= bound


@pytest.mark.parametrize('mode', ['fp32', 'bf16x3', 'bf16'])
def test_full_cfg5_against_torch(mode):
    # BASELINE configuration 5 at its full size: N=32, 256 -> 256 channels, 56 x 56, 3 x 3,
    # stride 1, pad 1; y, dx and dw against torch's conv2d and its autograd on the CPU, 1e-3
    # (1e-2 with operands rounded to bf16)
    N, C, H, W, D = 32, 256, 56, 56, 256
    g = torch.Generator().manual_seed(1005)
    xh = torch.randn(N, C, H, W, generator=g)
    wh = torch.randn(D, C, 3, 3, generator=g) * (2.0 / (C * 9)) ** 0.5   # Kaiming-normal
    dyh = torch.randn(N, D, H, W, generator=g)
    xr, wr = xh.clone().requires_grad_(True), wh.clone().requires_grad_(True)
    print('cfg5: torch conv2d on the CPU ...', flush=True)
    yr = F.conv2d(xr, wr, padding=1)
    yr.backward(dyh)
    native.set_option('conv_compute', MODES[mode][0])
    try:
        x, w, dy = xh.cuda(), wh.cuda(), dyh.cuda()
        geo = _ci(N, C, H, W, D, 3, 3, 1, 1, 1, 1, 1, 1)
        y = torch.empty(N, D, H, W, device='cuda')
        _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(x), _ptr(w), _ptr(w), ctypes.c_int(0), *geo,
              _ptr(y))
        _close(y, yr, 'cfg5 y ' + mode, MODES[mode][1])
        dx = torch.empty_like(x)
        _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dy), _ptr(w), ctypes.c_int(0), *geo,
              _ptr(dx))
        _close(dx, xr.grad, 'cfg5 dx ' + mode, MODES[mode][1])
        dw = torch.empty_like(w)
        _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw.numel()), _ptr(dy), _ptr(x), ctypes.c_int(0),
              *geo, _ptr(dw))
        _close(dw, wr.grad, 'cfg5 dw ' + mode, MODES[mode][1])
    finally:
        native.set_option('conv_compute', 0)


@pytest.mark.parametrize('shape', [
    # N, C, H, W, D, kernel, pad, stride, dilation
    (3, 40, 24, 24, 72, (3, 3), (1, 1), (1, 1), (1, 1)),    # rows of four: the 16-byte conversion
    (2, 33, 19, 21, 50, (3, 2), (2, 0), (1, 1), (1, 1)),    # odd rows: the element-wise conversion
    (4, 64, 56, 56, 64, (3, 3), (1, 1), (1, 1), (1, 1)),    # planes longer than one conversion span
    (1, 3, 12, 12, 5, (3, 3), (1, 1), (1, 1), (1, 1)),      # N * C odd: the sets of planes end off a 256-byte boundary
    (3, 5, 9, 11, 7, (3, 3), (1, 1), (1, 1), (1, 1)),       # likewise with an odd grid width
    (1, 4, 70, 71, 6, (3, 3), (1, 1), (1, 1), (1, 1)),      # the element-wise conversion over planes of two spans
    (3, 8, 17, 13, 20, (3, 2), (2, 1), (2, 1), (1, 2)),     # strides and dilation: the gathered weight gradient
    (4, 32, 30, 30, 140, (5, 5), (2, 2), (2, 2), (1, 1)),   # several channel blocks and row tiles, strides
    (2, 70, 23, 17, 200, (3, 3), (1, 1), (1, 1), (1, 1)),   # channels not a multiple of 32
])
def test_split_operands_keep_every_cross_term(shape):
    # Two bf16 per fp32 and three products (head x head, head x tail, tail x head) leave errors of
    # about 2^-16 of the operands; leaving out one cross term would leave about 2^-9, the error
    # of operands rounded to bf16.  Reference: the same sums in float64.
    N, C, H, W, D, kernel, pad, stride, dil = shape
    g = torch.Generator().manual_seed(77)
    x = torch.randn(N, C, H, W, generator=g)
    w = torch.randn(D, C, *kernel, generator=g) * 0.1
    xr, wr = x.double().requires_grad_(True), w.double().requires_grad_(True)
    y_ref = F.conv2d(xr, wr, None, stride=stride, padding=pad, dilation=dil)
    dy = torch.randn(y_ref.shape, generator=g)
    y_ref.backward(dy.double())
    try:
        native.set_option('conv_compute', 1)
        _leave_nan_patterns_in_the_workspace()
        native.set_option('conv_compute', 2)
        xd, wd, dyd = x.cuda(), w.cuda(), dy.cuda()
        geo = _ci(N, C, H, W, D, kernel[0], kernel[1], pad[0], pad[1], stride[0], stride[1], dil[0], dil[1])
        y = torch.full(y_ref.shape, float('nan'), device='cuda')
        _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(xd), _ptr(wd), _ptr(wd), ctypes.c_int(0),
              *geo, _ptr(y))
        _close(y, y_ref, 'y', 3e-5)
        dx = torch.full(x.shape, float('nan'), device='cuda')
        _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dyd), _ptr(wd), ctypes.c_int(0),
              *geo, _ptr(dx))
        _close(dx, xr.grad, 'dx', 3e-5)
        dw = torch.full(w.shape, float('nan'), device='cuda')
        _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw.numel()), _ptr(dyd), _ptr(xd), ctypes.c_int(0),
              *geo, _ptr(dw))
        _close(dw, wr.grad, 'dw', 3e-5)
    finally:
        native.set_option('conv_compute', 0)


def test_random_shapes_in_every_mode():
    # sixty seeded shapes (channel counts around the 32-channel blocks, strides, dilation, padding
    # beyond the kernel, widths with and without 16-byte rows), each in one of the three ways of
    # forming the products, against torch's float64 convolution and its autograd
    tol = {0: 2e-5, 2: 3e-5}
    done = 0
    for case in range(80):
        rng = np.random.default_rng(5000 + case)
        N, C, D = int(rng.integers(1, 5)), int(rng.choice([1, 3, 8, 31, 32, 33, 64, 70])), int(rng.choice([1, 5, 32, 100, 129, 260]))
        H, W = int(rng.integers(1, 40)), int(rng.integers(1, 40))
        if rng.integers(0, 2):
            W = (W + 3) // 4 * 4
        kh, kw = int(rng.integers(1, 4)), int(rng.integers(1, 4))
        ph, pw = int(rng.integers(0, 3)), int(rng.integers(0, 3))
        sh, sw = (1, 1) if rng.integers(0, 3) else (int(rng.integers(1, 3)), int(rng.integers(1, 3)))
        dh, dw_ = (1, 1) if rng.integers(0, 3) else (int(rng.integers(1, 3)), int(rng.integers(1, 3)))
        mode = int(rng.integers(0, 3))
        if H + 2 * ph < dh * (kh - 1) + 1 or W + 2 * pw < dw_ * (kw - 1) + 1:
            continue
        g = torch.Generator().manual_seed(5000 + case)
        x = torch.randn(N, C, H, W, generator=g)
        w = torch.randn(D, C, kh, kw, generator=g) * 0.2
        xr, wr = x.double().requires_grad_(True), w.double().requires_grad_(True)
        y_ref = F.conv2d(xr, wr, None, stride=(sh, sw), padding=(ph, pw), dilation=(dh, dw_))
        dy = torch.randn(y_ref.shape, generator=g)
        y_ref.backward(dy.double())
        what = 'case {}: mode {} N{} C{} {}x{} D{} k{}x{} p{},{} s{},{} d{},{}'.format(
            case, mode, N, C, H, W, D, kh, kw, ph, pw, sh, sw, dh, dw_)
        print(what, flush=True)
        native.set_option('conv_compute', mode)
        try:
            xd, wd, dyd = x.cuda(), w.cuda(), dy.cuda()
            geo = _ci(N, C, H, W, D, kh, kw, ph, pw, sh, sw, dh, dw_)
            y = torch.full(y_ref.shape, float('nan'), device='cuda')
            _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(xd), _ptr(wd), _ptr(wd), ctypes.c_int(0),
                  *geo, _ptr(y))
            dx = torch.full(x.shape, float('nan'), device='cuda')
            _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dyd), _ptr(wd), ctypes.c_int(0),
                  *geo, _ptr(dx))
            dw = torch.full(w.shape, float('nan'), device='cuda')
            _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw.numel()), _ptr(dyd), _ptr(xd), ctypes.c_int(0),
                  *geo, _ptr(dw))
        finally:
            native.set_option('conv_compute', 0)
        if mode == 1:
            # operands rounded to bf16 are off by up to 2^-9 each: the bound is a share of the sum of
            # the terms' magnitudes, which a sum that cancels can be far below
            xa, wa = x.double().abs().requires_grad_(True), w.double().abs().requires_grad_(True)
            ya = F.conv2d(xa, wa, None, stride=(sh, sw), padding=(ph, pw), dilation=(dh, dw_))
            ya.backward(dy.double().abs())
            for got, want, mag, name in ((y, y_ref, ya, ' y'), (dx, xr.grad, xa.grad, ' dx'), (dw, wr.grad, wa.grad, ' dw')):
                err = float((got.cpu().double() - want.detach()).abs().max())
                assert err <= 2.0 ** -7 * float(mag.detach().max()), what + name
        else:
            _close(y, y_ref, what + ' y', tol[mode])
            _close(dx, xr.grad, what + ' dx', tol[mode])
            _close(dw, wr.grad, what + ' dw', tol[mode])
        done += 1
    assert done >= 60


def _leave_nan_patterns_in_the_workspace():
    # The bf16 products keep copies of their operands in the calling thread's workspace, which
    # is not cleared between calls: a product of NaN inputs (conv_compute must be 1) leaves NaN
    # bit patterns behind, so a later call that read bytes it had not written itself would show.
    x = torch.full((2, 32, 40, 40), float('nan'), device='cuda')
    w = torch.full((32, 32, 3, 3), float('nan'), device='cuda')
    y = torch.empty(2, 32, 40, 40, device='cuda')
    geo = _ci(2, 32, 40, 40, 32, 3, 3, 1, 1, 1, 1, 1, 1)
    _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(x), _ptr(w), _ptr(w), ctypes.c_int(0), *geo,
          _ptr(y))
    dw = torch.empty_like(w)
    _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw.numel()), _ptr(y), _ptr(x), ctypes.c_int(0), *geo,
          _ptr(dw))
    torch.cuda.synchronize()


@pytest.mark.parametrize('case', [
    # N, C, H, W, D, kernel, pad, stride, dilation
    (3, 64, 20, 20, 96, (3, 3), (1, 1), (1, 1), (1, 1)),      # 128-row tiles
    (2, 70, 23, 17, 200, (3, 3), (1, 1), (1, 1), (1, 1)),     # 256-row tiles, channels not a multiple of 32
    (2, 40, 19, 21, 130, (5, 3), (2, 0), (1, 1), (1, 2)),     # dilation, uneven padding
    (2, 33, 30, 26, 300, (3, 3), (1, 1), (2, 2), (1, 1)),     # strides: two row tiles, gathered weight gradient
    (9, 256, 28, 28, 256, (3, 3), (1, 1), (1, 1), (1, 1)),    # several images to a tile, K cut into pieces
    (1, 16, 60, 60, 16, (1, 1), (0, 0), (1, 1), (1, 1)),      # one tap
    (2, 8, 96, 96, 12, (3, 3), (1, 1), (1, 1), (1, 1)),       # planes of several spans in the padded copies
    (1, 8, 70, 104, 8, (1, 3), (0, 1), (1, 1), (1, 1)),       # likewise, no padded rows
    (1, 3, 12, 12, 5, (3, 3), (1, 1), (1, 1), (1, 1)),        # N * C odd: the padded copies end off a 256-byte boundary
    (3, 5, 9, 11, 7, (3, 3), (1, 1), (1, 1), (1, 1)),         # likewise, odd grid width (the scalar copy)
    (2, 20, 20, 20, 100, (3, 3), (1, 1), (1, 1), (1, 1)),     # 128-row tiles with channels not a multiple of 32
    (1, 6, 21, 20, 9, (1, 2), (0, 0), (1, 1), (1, 1)),        # an odd shift without padding
    (1, 4, 70, 71, 6, (3, 3), (1, 1), (1, 1), (1, 1)),        # odd width: the scalar copy over planes of two spans
    (1, 2, 3, 4100, 4, (3, 3), (1, 1), (1, 1), (1, 1)),       # grid rows longer than a span
])
def test_bf16_mode_is_exact_on_bf16_valued_operands(case):
    # Mode 1 rounds both operands of every product to bf16 and accumulates in fp32: against
    # the same products of the rounded operands in fp32 only the order of the sums differs,
    # well inside the 1e-3 bound (the 1e-2 of the other tests is the rounding of the inputs)
    N, C, H, W, D, k, pad, stride, dil = case
    g = torch.Generator().manual_seed(61)
    x = torch.randn(N, C, H, W, generator=g)
    w = torch.randn(D, C, *k, generator=g) * 0.1
    rnd = lambda t: t.bfloat16().float()
    xr, wr = rnd(x).requires_grad_(True), rnd(w).requires_grad_(True)
    yr = F.conv2d(xr, wr, padding=pad, stride=stride, dilation=dil)
    dy = torch.randn(yr.shape, generator=g)
    yr.backward(rnd(dy))
    native.set_option('conv_compute', 1)
    try:
        _leave_nan_patterns_in_the_workspace()
        xd, wd, dyd = x.cuda(), w.cuda(), dy.cuda()
        geo = _ci(N, C, H, W, D, k[0], k[1], pad[0], pad[1], stride[0], stride[1], dil[0], dil[1])
        y = torch.empty(yr.shape, device='cuda')
        _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(xd), _ptr(wd), _ptr(wd), ctypes.c_int(0),
              *geo, _ptr(y))
        dx = torch.empty_like(xd)
        _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dyd), _ptr(wd), ctypes.c_int(0),
              *geo, _ptr(dx))
        dw = torch.empty_like(wd)
        _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw.numel()), _ptr(dyd), _ptr(xd), ctypes.c_int(0),
              *geo, _ptr(dw))
        # accumulate: twice the gradient on top of what is there
        dw2 = dw.clone()
        _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw.numel()), _ptr(dyd), _ptr(xd), ctypes.c_int(1),
              *geo, _ptr(dw2))
        dx2 = dx.clone()
        _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dyd), _ptr(wd), ctypes.c_int(1),
              *geo, _ptr(dx2))
    finally:
        native.set_option('conv_compute', 0)
    _close(y, yr.detach(), 'y', 1e-4)
    _close(dx, xr.grad, 'dx', 1e-4)
    _close(dw, wr.grad, 'dw', 1e-4)
    _close(dw2, 2 * wr.grad, 'dw accumulated', 1e-4)
    _close(dx2, 2 * xr.grad, 'dx accumulated', 1e-4)


@pytest.mark.parametrize('mode', ['bf16', 'bf16x3', 'three parts', 'halves'])
@pytest.mark.parametrize('case', [
    # N, C, H, W, D, kernel, pad, stride, dilation
    (2, 70, 23, 18, 40, (3, 3), (1, 1), (2, 2), (1, 1)),    # phases of one, two and four taps
    (3, 20, 17, 31, 33, (5, 4), (2, 0), (2, 1), (1, 1)),
    (2, 24, 20, 19, 48, (1, 1), (0, 0), (2, 2), (1, 1)),    # a single tap: all pixels in one go
    (2, 24, 21, 20, 48, (3, 3), (2, 1), (2, 4), (2, 1)),    # a filter of every second row: odd rows meet no tap; four phases of columns
    (2, 17, 19, 23, 20, (3, 4), (1, 2), (3, 2), (2, 3)),    # stride and dilation without a common factor
    (300, 16, 3, 2, 20, (2, 2), (1, 0), (4, 2), (1, 1)),    # fewer rows than phases; a tile spans hundreds of images
    (1, 130, 40, 37, 20, (7, 7), (3, 3), (4, 4), (1, 1)),   # sixteen phases, the most
    (2, 18, 30, 30, 20, (6, 5), (2, 2), (5, 4), (1, 1)),    # twenty: all taps
    (1, 600, 16, 16, 600, (3, 3), (1, 1), (2, 2), (1, 1)),  # cut along K; few pixels, all taps with three parts and halves
    (4, 40, 40, 41, 130, (3, 3), (1, 1), (2, 2), (1, 1)),   # cut along K: phases of 36, 18 and nine steps into as many pieces
    (9, 33, 45, 38, 44, (5, 5), (2, 2), (2, 2), (1, 1)),
])
def test_data_gradient_of_strided_products(case, mode):
    """Every phase of the strides with its own taps, against the products of the same operands in 64 bits; what the gradient
    is added to; an infinite weight reaches no pixels of other phases."""
    N, C, H, W, D, k, pad, stride, dil = case
    g = torch.Generator().manual_seed(62)
    w = torch.randn(D, C, *k, generator=g) * 0.1
    shape = (N, C, H, W)
    y_shape = F.conv2d(torch.zeros(1, C, H, W), w, padding=pad, stride=stride, dilation=dil).shape
    dy = torch.randn((N,) + y_shape[1:], generator=g)
    rnd = (lambda t: t.bfloat16().double()) if mode == 'bf16' else (lambda t: t.double())
    want = torch.nn.grad.conv2d_input(shape, rnd(w), rnd(dy), stride=stride, padding=pad, dilation=dil)
    # terms are rounded to 2^-16 of an operand with two parts, sums to fp32 otherwise; of the largest result
    tol = 2e-5 if mode == 'bf16x3' else 2e-6
    native.set_option('conv_compute', {'bf16': 1, 'bf16x3': 2}.get(mode, 0))
    native.set_option('conv_fp32_split', {'three parts': 2, 'halves': 3}.get(mode, 1))
    try:
        _leave_nan_patterns_in_the_workspace()
        geo = _ci(N, C, H, W, D, k[0], k[1], pad[0], pad[1], stride[0], stride[1], dil[0], dil[1])
        dyd = dy.cuda()

        def run(weight, dx, accumulate):
            _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dyd), _ptr(weight), ctypes.c_int(accumulate), *geo,
                  _ptr(dx))
            return dx
        wd = w.cuda()
        dx = run(wd, torch.full(shape, float('nan'), device='cuda'), 0)
        _close(dx, want, 'dx', tol)
        _close(run(wd, dx.clone(), 1), 2 * want, 'dx accumulated', tol)
        if mode == 'bf16' and stride[0] * stride[1] <= 16 and k != (1, 1):   # (its phase it meets beyond dy's border, too)
            wd[:, :, 0, 0] = float('inf')
            got = run(wd, torch.empty(shape, device='cuda'), 0).cpu()
            phase = ((torch.arange(H) + pad[0]) % stride[0] == 0)[:, None] & ((torch.arange(W) + pad[1]) % stride[1] == 0)
            assert torch.isfinite(got[:, :, ~phase]).all()
    finally:
        native.set_option('conv_compute', 0)
        native.set_option('conv_fp32_split', 1)


def test_strided_data_gradient_where_phases_reach_too_far():
    """So many images that the offsets of a phase's tiles would pass 2^31 and those of whole images do not: all taps, walked one
    by one (tests/test_conv_phases.py has the rule)."""
    N, C, H, W, D = 21398, 4, 14, 14, 512
    g = torch.Generator(device='cuda').manual_seed(5)
    w = torch.randn((D, C, 3, 3), generator=g, device='cuda') * 0.1
    dy = torch.randn((N, D, 7, 7), generator=g, device='cuda')
    dx = torch.full((N, C, H, W), float('nan'), device='cuda')
    native.set_option('conv_compute', 2)
    try:
        _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dy), _ptr(w), ctypes.c_int(0),
              *_ci(N, C, H, W, D, 3, 3, 1, 1, 2, 2, 1, 1), _ptr(dx))
    finally:
        native.set_option('conv_compute', 0)
    assert torch.isfinite(dx).all()
    for n in (0, 1, N // 2, N - 1):
        want = torch.nn.grad.conv2d_input((1, C, H, W), w.double().cpu(), dy[n:n + 1].double().cpu(), stride=2, padding=1)
        _close(dx[n:n + 1], want, 'image %d' % n, 2e-5)   # (two parts: terms to 2^-16 of an operand)


def test_errors_surface_as_exceptions():
    x = torch.zeros(1, 1, 4, 4, device='cuda')
    w = torch.zeros(1, 1, 3, 3, device='cuda')
    y = torch.zeros(1, 1, 2, 2, device='cuda')
    geo = _ci(1, 1, 4, 4, 1, 3, 3, 0, 0, 1, 1, 1, 1)
    with pytest.raises(RuntimeError):   # wrong output element count
        _call('conv2d_forward_c6a7aa85', ctypes.c_int(3), _ptr(x), _ptr(w), _ptr(w), ctypes.c_int(0), *geo, _ptr(y))
    with pytest.raises(RuntimeError):   # window larger than the padded input
        _call('conv2d_forward_c6a7aa85', ctypes.c_int(4), _ptr(x), _ptr(w), _ptr(w), ctypes.c_int(0),
              *_ci(1, 1, 2, 2, 1, 3, 3, 0, 0, 1, 1, 1, 1), _ptr(y))
    lib = native.library()
    native.begin_call(None, [])
    lib.conv2d_forward_c6a7aa85(ctypes.c_int(-1), ctypes.c_int(4), _ptr(x), _ptr(w), _ptr(w), ctypes.c_int(0), *geo,
                                _ptr(y))
    with pytest.raises(RuntimeError):   # host buffers are not staged for the convolution
        native.end_call('conv2d_forward')
    # the library stays usable
    _call('conv2d_forward_c6a7aa85', ctypes.c_int(4), _ptr(x), _ptr(w), _ptr(w), ctypes.c_int(0), *geo, _ptr(y))


@pytest.mark.parametrize('shape', [
    # the fp32 kernels that stage patches of the map: tiles of 32, 64 and 128 rows, their edges, and what chunks,
    # strides and image borders do to them  (N, C, H, W, D, kernel, pad, stride, dilation)
    (2, 3, 40, 37, 64, (7, 7), (3, 3), (2, 2), (1, 1)),     # a first layer; planes that are no multiple of four
    (9, 3, 5, 6, 65, (3, 3), (1, 1), (1, 1), (1, 1)),       # tiles span images; one row past a tile
    (3, 1, 33, 64, 32, (5, 1), (2, 0), (1, 1), (1, 1)),     # one channel, rows that divide a tile
    (2, 19, 24, 30, 33, (3, 3), (1, 1), (2, 3), (1, 1)),    # strides that differ: six classes of dx
    (1, 40, 21, 26, 24, (3, 2), (2, 1), (3, 2), (2, 3)),    # dilation against stride: classes without taps
    (2, 8, 16, 16, 130, (1, 1), (0, 0), (2, 2), (1, 1)),    # pointwise at a stride: three classes of dx are zero
    (5, 33, 11, 11, 17, (1, 1), (0, 0), (1, 1), (1, 1)),    # pointwise, few rows
    (1, 5, 60, 250, 40, (3, 9), (0, 4), (1, 1), (1, 1)),    # rows longer than a tile
])
def test_fp32_products_from_patches(shape):
    N, C, H, W, D, kernel, pad, stride, dil = shape
    g = torch.Generator().manual_seed(77)
    x, w = torch.randn(N, C, H, W, generator=g), torch.randn(D, C, *kernel, generator=g)
    b = torch.randn(D, generator=g)
    xr, wr = x.double().requires_grad_(True), w.double().requires_grad_(True)
    y_ref = F.conv2d(xr, wr, b.double(), stride=stride, padding=pad, dilation=dil)
    dy = torch.randn(y_ref.shape, generator=g)
    y_ref.backward(dy.double())
    xd, wd, bd, dyd = x.cuda(), w.cuda(), b.cuda(), dy.cuda()
    geo = _ci(N, C, H, W, D, kernel[0], kernel[1], pad[0], pad[1], stride[0], stride[1], dil[0], dil[1])
    y = torch.full(y_ref.shape, float('nan'), device='cuda')
    _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(xd), _ptr(wd), _ptr(bd), ctypes.c_int(1), *geo, _ptr(y))
    _close(y, y_ref, 'y', 1e-5)
    for start, accumulate in ((float('nan'), 0), (1.0, 1)):
        dx, dw = torch.full(x.shape, start, device='cuda'), torch.full(w.shape, start, device='cuda')
        _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dyd), _ptr(wd), ctypes.c_int(accumulate),
              *geo, _ptr(dx))
        _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw.numel()), _ptr(dyd), _ptr(xd), ctypes.c_int(accumulate),
              *geo, _ptr(dw))
        _close(dx - accumulate, xr.grad, 'dx', 1e-5)
        _close(dw - accumulate, wr.grad, 'dw', 1e-5)
    db = torch.empty(D, device='cuda')
    _call('conv2d_backward_bias_cd239a08', ctypes.c_int(D), _ptr(dyd), ctypes.c_int(0), ctypes.c_int(N),
          ctypes.c_int(y.shape[2] * y.shape[3]), _ptr(db))
    _close(db, dy.double().sum((0, 2, 3)), 'db', 1e-5)


@pytest.mark.parametrize('channels,filters', [(16, 128), (32, 130), (48, 100), (128, 16), (130, 32), (100, 48)])
def test_fp32_gathered_products_of_few_steps(channels, filters):
    """Tiles of one, two and three K steps (the loop requests two ahead), rows and columns that end
    within a tile; the weight gradient's slices are one K step each."""
    g = torch.Generator().manual_seed(78)
    x, w = torch.randn(3, channels, 9, 15, generator=g), torch.randn(filters, channels, 1, 1, generator=g)
    dy = torch.randn(3, filters, 9, 15, generator=g)
    xr, wr = x.double().requires_grad_(True), w.double().requires_grad_(True)
    y_ref = F.conv2d(xr, wr)
    y_ref.backward(dy.double())
    geo = _ci(3, channels, 9, 15, filters, 1, 1, 0, 0, 1, 1, 1, 1)
    xd, wd, dyd = x.cuda(), w.cuda(), dy.cuda()
    y = torch.full(dy.shape, float('nan'), device='cuda')
    _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(xd), _ptr(wd), _ptr(wd), ctypes.c_int(0), *geo, _ptr(y))
    _close(y, y_ref, 'y', 1e-5)
    for start, accumulate in ((float('nan'), 0), (1.0, 1)):
        dx, dw = torch.full(x.shape, start, device='cuda'), torch.full(w.shape, start, device='cuda')
        _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dyd), _ptr(wd), ctypes.c_int(accumulate),
              *geo, _ptr(dx))
        _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw.numel()), _ptr(dyd), _ptr(xd), ctypes.c_int(accumulate),
              *geo, _ptr(dw))
        _close(dx - accumulate, xr.grad, 'dx', 1e-5)
        _close(dw - accumulate, wr.grad, 'dw', 1e-5)


@pytest.mark.parametrize('channels,filters,kernel', [(512, 512, 3), (256, 256, 7)])
def test_weights_of_more_than_two_million_elements(channels, filters, kernel):
    """The gathered products read a rearranged copy of the weights from the workspace: all of it is written."""
    g = torch.Generator().manual_seed(79)
    x = torch.randn(1, channels, 14, 14, generator=g)
    w = torch.randn(filters, channels, kernel, kernel, generator=g)
    dy = torch.randn(1, filters, 14, 14, generator=g)
    xr = x.double().requires_grad_(True)
    y_ref = F.conv2d(xr, w.double(), padding=kernel // 2)
    y_ref.backward(dy.double())
    geo = _ci(1, channels, 14, 14, filters, kernel, kernel, kernel // 2, kernel // 2, 1, 1, 1, 1)
    xd, wd, dyd = x.cuda(), w.cuda(), dy.cuda()
    y, dx = torch.empty(dy.shape, device='cuda'), torch.empty(x.shape, device='cuda')
    abi.poison_workspace(128 << 20)
    _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(xd), _ptr(wd), _ptr(wd), ctypes.c_int(0), *geo, _ptr(y))
    _close(y, y_ref, 'y', 1e-5)
    abi.poison_workspace(128 << 20)
    _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dyd), _ptr(wd), ctypes.c_int(0), *geo, _ptr(dx))
    _close(dx, xr.grad, 'dx', 1e-5)


def test_bias_gradient_can_be_recorded_first():
    """Without a workspace, which cannot be had while a stream is being captured, one workgroup per filter
    adds the images up."""
    dy = torch.randn(5, 3, 7, 9, generator=torch.Generator().manual_seed(80))
    dyd, db, stream = dy.cuda(), torch.zeros(3, device='cuda'), torch.cuda.Stream()
    torch.cuda.synchronize()
    native.release_workspace()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        native.begin_call(torch.cuda.current_stream().cuda_stream, [])
        native.library().conv2d_backward_bias_cd239a08(ctypes.c_int(0), *_ci(3), _ptr(dyd), *_ci(0, 5, 63), _ptr(db))
        native.end_call('conv2d_backward_bias')
    for _ in range(3):
        db.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        _close(db, dy.double().sum((0, 2, 3)), 'db', 1e-5)
        dyd.add_(0)   # (ordinary work between the replays)


@pytest.mark.parametrize('wanted', ['x w b', 'w b', 'b'])
@pytest.mark.parametrize('shape', [
    (2, 3, 70, 66, 7, 3, 1),       # planes of ten runs, the last of twelve pixels
    (3, 16, 65, 63, 130, 1, 1),    # odd planes: no whole quads
    (5, 34, 9, 7, 3, 3, 2),
    (300, 16, 3, 3, 66, 3, 1),     # many small planes
    (4, 64, 31, 33, 256, 3, 1),    # high tiles for both gradients
])
def test_bias_gradient_beside_the_others(mobula, shape, wanted, compute):
    """The bias's gradient rides in launches of the other gradients where there are any: 64-bit sums, rounded once (half a unit
    of the result; 2^-40 of the sum of magnitudes for the 64-bit additions, of which there are fewer than 2^12)."""
    mobula.op.load('Convolution')
    N, C, H, W, D, K, stride = shape
    gen = torch.Generator().manual_seed(sum(shape))
    x = torch.randn(N, C, H, W, generator=gen).cuda().requires_grad_('x' in wanted)
    w = (torch.randn(D, C, K, K, generator=gen) / (C * K * K) ** 0.5).cuda().requires_grad_('w' in wanted)
    b = torch.randn(D, generator=gen).cuda().requires_grad_(True)
    y = mobula.op.Conv2D(x, w, b, channels=D, kernel_size=(K, K), strides=(stride, stride), padding=(K // 2, K // 2))
    dy = torch.randn(y.shape, generator=gen).cuda() + 0.5
    y.backward(dy)
    exact, size = dy.double().sum((0, 2, 3)), dy.double().abs().sum((0, 2, 3))
    assert ((b.grad.double() - exact).abs() <= 2.0 ** -24 * exact.abs() + 2.0 ** -40 * size).all()
    xr, wr, br = (t.detach().cpu().requires_grad_(t.requires_grad) for t in (x, w, b))
    F.conv2d(xr, wr, br, stride=stride, padding=K // 2).backward(dy.cpu())
    if 'x' in wanted:
        _close(x.grad, xr.grad, 'dx', compute)
    if 'w' in wanted:
        _close(w.grad, wr.grad, 'dw', compute)


def test_bias_gradient_that_finds_no_room_beside_the_others(mobula):
    """A recorded call cannot grow the workspace: one that was warmed up without a bias leaves none for its sums (an image of
    one pixel has as many sums as filters).  They are 64-bit sums all the same (the bound of
    test_bias_gradient_beside_the_others)."""
    N, D = 65000, 336
    mobula.op.load('Convolution')
    gen = torch.Generator().manual_seed(8)
    x, w = torch.randn(N, 1, 1, 1, generator=gen).cuda(), torch.randn(D, 1, 1, 1, generator=gen).cuda().requires_grad_(True)
    b = torch.zeros(D, device='cuda', requires_grad=True)
    dy = torch.randn(N, D, 1, 1, generator=gen).cuda()
    dy[1::2] = 1e-3 * dy[1::2] - dy[0::2]   # (terms that nearly cancel)

    def gradients(*inputs):
        y = mobula.op.Conv2D(*inputs, channels=D, kernel_size=(1, 1))
        return torch.autograd.grad(y, inputs[1:], dy)

    stream = torch.cuda.Stream()
    try:
        with torch.cuda.stream(stream):
            native.release_workspace()
            alone, = gradients(x, w)
            torch.cuda.synchronize()
            assert native.workspace_bytes() < 8 * N * D
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                dw, db = gradients(x, w, b)
            for _ in range(3):
                dw.zero_()
                db.zero_()
                torch.cuda.synchronize()
                graph.replay()
                torch.cuda.synchronize()
                assert torch.equal(dw, alone)
                exact, size = dy.double().sum((0, 2, 3)), dy.double().abs().sum((0, 2, 3))
                assert ((db.double() - exact).abs() <= 2.0 ** -24 * exact.abs() + 2.0 ** -40 * size).all()
            del graph
    finally:
        native.unpin_workspace()


@pytest.mark.parametrize('mode', ['bf16', 'bf16x3'])
def test_both_gradients_in_a_workspace_that_holds_the_operands_of_one(mode):
    """The gradients of one call share their operands where the workspace can hold both; where it cannot
    grow they are made one after the other, with the same bits."""
    native.set_option('conv_compute', MODES[mode][0])
    N, C, H, W, D = 24 if mode == 'bf16' else 12, 32, 56, 56, 512
    g = torch.Generator(device='cuda').manual_seed(81)
    x, w = torch.randn(N, C, H, W, generator=g, device='cuda'), torch.randn(D, C, 3, 3, generator=g, device='cuda')
    dy = torch.randn(N, D, H, W, generator=g, device='cuda')
    geo = _ci(N, C, H, W, D, 3, 3, 1, 1, 1, 1, 1, 1)
    lib, stream = native.library(), torch.cuda.Stream()

    def both(dx, dw, on=None):
        native.begin_call(on, [])
        lib.mobula_hip_conv2d_backward(ctypes.c_int(0), _ptr(dy), _ptr(x), _ptr(w), *geo, _ptr(dx), _ptr(dw))
        native.end_call('conv2d_backward')
    try:
        want, single, got = ([torch.full_like(t, float('nan')) for t in (x, w)] for _ in range(3))
        torch.cuda.synchronize()
        both(*want)
        roomy = native.workspace_bytes()
        native.release_workspace()
        _call('conv2d_backward_data_ecf81c91', ctypes.c_int(x.numel()), _ptr(dy), _ptr(w), ctypes.c_int(0), *geo,
              _ptr(single[0]))
        _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(w.numel()), _ptr(dy), _ptr(x), ctypes.c_int(0), *geo,
              _ptr(single[1]))
        held = native.workspace_bytes()
        assert held < roomy / 1.25   # (a workspace is made a quarter larger than asked for)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            both(*got, on=torch.cuda.current_stream().cuda_stream)
        for _ in range(3):
            for t in got:
                t.fill_(float('nan'))
            graph.replay()
            torch.cuda.synchronize()
            for a, b, c in zip(got, want, single):
                assert torch.equal(a, b) and torch.equal(a, c)
            both(*single)   # an ordinary call between the replays: the recorded graph holds the workspace where it is
            assert native.workspace_bytes() == held
        del graph
    finally:
        native.unpin_workspace()
        native.set_option('conv_compute', 0)


@pytest.mark.parametrize('shape', [
    # K steps of the products from patches that end in padding: taps x channels that fill no whole step, chunks of
    # channels that end past the last one, chunks of pixels that end past the plane
    (2, 3, 20, 21, 64, (7, 7), (3, 3), (2, 2), (1, 1)),
    (3, 1, 33, 64, 32, (5, 1), (2, 0), (1, 1), (1, 1)),
    (2, 32, 24, 26, 33, (3, 3), (1, 1), (2, 2), (1, 1)),
    (2, 50, 19, 23, 40, (3, 3), (1, 1), (1, 1), (1, 1)),
    (5, 33, 11, 11, 17, (1, 1), (0, 0), (1, 1), (1, 1)),
    # gathered products: channels (of dy: filters) that fill no whole step of sixteen
    (2, 69, 9, 15, 250, (3, 3), (1, 1), (1, 1), (1, 1)),
    (3, 130, 9, 15, 140, (1, 1), (0, 0), (1, 1), (1, 1)),
])
def test_an_infinity_stays_an_infinity_in_fp32_products(shape):
    """What pads a K step is zero times zero: one infinite element of an operand makes the results that it
    belongs to infinite, of the right sign, and no other."""
    N, C, H, W, D, kernel, pad, stride, dil = shape
    g = torch.Generator().manual_seed(82)
    x, w = torch.randn(N, C, H, W, generator=g), torch.randn(D, C, *kernel, generator=g)
    geo = _ci(N, C, H, W, D, kernel[0], kernel[1], pad[0], pad[1], stride[0], stride[1], dil[0], dil[1])

    def check(got, want, what):
        got = got.cpu().double()
        assert not got.isnan().any(), what
        assert torch.equal(got == float('inf'), want == float('inf')) and torch.equal(got == -float('inf'), want == -float('inf')), what
        finite = want.isfinite()
        if finite.any():
            _close(got[finite], want[finite], what, 1e-5)
    for at in ((0, 0, 0, 0), (N - 1, C - 1, H - 1, W - 1), (N // 2, C // 2, H // 2, W // 2), (0, C - 1, 1, 2)):
        xi = x.clone()
        xi[at] = float('inf')
        xr, wr = x.double().requires_grad_(True), w.double().requires_grad_(True)
        conv = lambda a, b: F.conv2d(a, b, stride=stride, padding=pad, dilation=dil)   # noqa: E731
        y_ref = conv(xi.double(), wr)
        dy = torch.randn(y_ref.shape, generator=g)
        (dw_ref,) = torch.autograd.grad(y_ref, wr, dy.double())
        y, dw, dx = torch.empty(dy.shape, device='cuda'), torch.empty(w.shape, device='cuda'), torch.empty(x.shape, device='cuda')
        xd, wd, dyd = xi.cuda(), w.cuda(), dy.cuda()
        _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(xd), _ptr(wd), _ptr(wd), ctypes.c_int(0), *geo, _ptr(y))
        check(y, y_ref.detach(), 'y')
        _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw.numel()), _ptr(dyd), _ptr(xd), ctypes.c_int(0), *geo, _ptr(dw))
        check(dw, dw_ref, 'dw')
        dyi = dy.clone()
        dyi[at[0], at[1] % D, min(at[2], dy.shape[2] - 1), min(at[3], dy.shape[3] - 1)] = float('inf')
        (dx_ref,) = torch.autograd.grad(conv(xr, w.double()), xr, dyi.double())
        dyd = dyi.cuda()
        _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dyd), _ptr(wd), ctypes.c_int(0), *geo, _ptr(dx))
        check(dx, dx_ref, 'dx')


@pytest.fixture
def split_always():
    native.set_option('conv_fp32_split', 2)
    yield
    native.set_option('conv_fp32_split', 1)


def _three_products(geo, x, w, dy, dx0=None, dw0=None):
    """y, dx, dw through the C-ABI; dx0, dw0: added to."""
    y = torch.full(dy.shape, float('nan'), device='cuda')
    dx = torch.full(x.shape, float('nan'), device='cuda') if dx0 is None else dx0.clone()
    dw = torch.full(w.shape, float('nan'), device='cuda') if dw0 is None else dw0.clone()
    _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(x), _ptr(w), _ptr(w), ctypes.c_int(0), *geo, _ptr(y))
    _call('conv2d_backward_data_ecf81c91', ctypes.c_int(dx.numel()), _ptr(dy), _ptr(w), ctypes.c_int(dx0 is not None), *geo,
          _ptr(dx))
    _call('conv2d_backward_weight_ecf81c91', ctypes.c_int(dw.numel()), _ptr(dy), _ptr(x), ctypes.c_int(dw0 is not None), *geo,
          _ptr(dw))
    return y, dx, dw


@pytest.mark.parametrize('shape', [
    # N, C, H, W, D, kernel, pad, stride, dilation
    (1, 1, 1, 1, 1, (1, 1), (0, 0), (1, 1), (1, 1)),         # one multiply-add
    (3, 16, 5, 3, 64, (1, 1), (0, 0), (1, 1), (1, 1)),       # 15 pixels an image: a step of K meets two and three images
    (40, 17, 2, 2, 65, (2, 2), (1, 1), (1, 1), (1, 1)),      # 9 pixels, rows and channels one past a tile and a block
    (2, 15, 16, 16, 128, (3, 3), (1, 1), (1, 1), (1, 1)),    # whole steps of pixels and rows of two workgroups' tiles
    (2, 33, 19, 21, 193, (3, 2), (2, 0), (1, 1), (1, 1)),    # odd planes: the element-wise conversion
    (4, 64, 24, 28, 256, (3, 3), (1, 1), (1, 1), (1, 1)),    # columns in whole tiles, rows too
    (3, 48, 23, 17, 257, (3, 3), (0, 1), (2, 2), (1, 1)),    # strides: taps that reach no pixel
    (2, 24, 30, 22, 40, (3, 2), (2, 1), (2, 1), (1, 2)),     # strides and dilation
    (5, 20, 7, 9, 130, (5, 5), (6, 2), (1, 3), (1, 1)),      # padding beyond the kernel
])
def test_fp32_products_of_three_parts(shape, split_always):
    """fp32 products from three bf16 parts per operand: exact products but for at most 2^-24 of them, and at most six fp32
    roundings for sixteen of K, each of 2^-24 of a sum no larger than the result's own scale."""
    N, C, H, W, D, kernel, pad, stride, dil = shape
    g = torch.Generator().manual_seed(91)
    x, w = torch.randn(N, C, H, W, generator=g), torch.randn(D, C, *kernel, generator=g)
    xr, wr = x.double().requires_grad_(True), w.double().requires_grad_(True)
    y_ref = F.conv2d(xr, wr, None, stride=stride, padding=pad, dilation=dil)
    dy = torch.randn(y_ref.shape, generator=g)
    y_ref.backward(dy.double())
    geo = _ci(N, C, H, W, D, kernel[0], kernel[1], pad[0], pad[1], stride[0], stride[1], dil[0], dil[1])
    _leave_nan_patterns_in_the_workspace()
    xd, wd, dyd = x.cuda(), w.cuda(), dy.cuda()
    got = _three_products(geo, xd, wd, dyd)
    terms = C * kernel[0] * kernel[1], D * kernel[0] * kernel[1], dy[:, 0].numel()
    for a, b, k, what in zip(got, (y_ref.detach(), xr.grad, wr.grad), terms, ('y', 'dx', 'dw')):
        error = ((a.cpu().double() - b).norm() / b.norm()).item()
        assert error <= 2.0 ** -24 * (1 + (6 * (k / 16 + 1)) ** 0.5), (what, error)
    # added to what is there; the same bits a second time
    start = torch.randn(x.shape, generator=g).cuda(), torch.randn(w.shape, generator=g).cuda()
    again = _three_products(geo, xd, wd, dyd, *start)
    assert torch.equal(again[0], got[0])
    assert torch.equal(again[1], start[0] + got[1]) and torch.equal(again[2], start[1] + got[2])


@pytest.mark.parametrize('scale_x,scale_w,odd', [
    (1.0, 1.0, float('inf')), (1.0, 1.0, -float('inf')), (1.0, 1.0, float('nan')),
    (1.0, 1.0, 3e38), (1.0, 1.0, 1e-40), (1.0, 1.0, 2.0 ** -110),
    (2.0 ** -60, 2.0 ** -60, None),     # every operand in range, the products' last parts not
    (2.0 ** 60, 2.0 ** 55, None), (2.0 ** -96, 2.0 ** 40, None), (0.0, 1.0, None),
])
def test_values_that_three_parts_do_not_stand_for(scale_x, scale_w, odd, split_always):
    """Operands outside the range of the parts are multiplied by the fp32 kernels: the results are those that the option
    gives without parts, which in these sizes take the same kernels."""
    N, C, H, W, D = 2, 64, 24, 28, 128
    geo = _ci(N, C, H, W, D, 3, 3, 1, 1, 1, 1, 1, 1)
    g = torch.Generator(device='cuda').manual_seed(92)
    x = torch.randn(N, C, H, W, generator=g, device='cuda') * scale_x
    w = torch.randn(D, C, 3, 3, generator=g, device='cuda') * scale_w
    dy = torch.randn(N, D, H, W, generator=g, device='cuda') * scale_x
    if odd is not None:
        x[1, 3, 5, 7] = odd
        dy[0, 9, 20, 1] = odd
    got = _three_products(geo, x, w, dy)
    native.set_option('conv_fp32_split', 0)
    want = _three_products(geo, x, w, dy)
    for a, b, what in zip(got, want, ('y', 'dx', 'dw')):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf()), what
        fine = b.isfinite()
        if fine.any() and b[fine].abs().max() > 0:
            scale = b[fine].double().norm()
            assert ((a[fine].double() - b[fine].double()).norm() / scale).item() <= 2e-6, what
        else:
            assert torch.equal(a[fine], b[fine]), what


@pytest.mark.parametrize('place,a,b', [
    # one product of two elements, the others of these tensors being zero
    ('one', 1.005 * 2.0 ** 70, 2.0 ** 70),      # an infinity; of the parts' products +inf and -inf
    ('one', -1.005 * 2.0 ** 70, 2.0 ** 70),
    ('one', 1.998 * 2.0 ** 63, 2.0 ** 64),      # finite; with the head rounded up 2^128
    ('one', 1.998 * 2.0 ** 50, 2.0 ** 50),      # finite, and formed from parts
    # sums of terms of one size, of one sign (of both, what overflows on the way depends on the order of the sum,
    # which neither way states): all overflow; none does
    ('all', 2.0 ** 63, 2.0 ** 62), ('all', 2.0 ** 50, 2.0 ** 50),
])
def test_fp32_products_and_sums_that_overflow(place, a, b, split_always):
    """Results are finite, infinite and NaN where the fp32 kernels' are, and these operands' (a product of
    few bits, sums that are whole multiples of one) the same to the bit."""
    N, C, H, W, D = 2, 64, 24, 28, 128
    geo = _ci(N, C, H, W, D, 3, 3, 1, 1, 1, 1, 1, 1)
    sign = (torch.arange(D, device='cuda') % 3 - 1.5).sign()   # of a filter's weights and of its dy

    def make(value, *shape):
        if place == 'all':
            return torch.full(shape, value, device='cuda')
        t = torch.zeros(shape, device='cuda')
        t[0, 5, 1, 1] = value
        return t
    x, w = make(a, N, C, H, W), make(b, D, C, 3, 3) * sign.reshape(D, 1, 1, 1)
    for dy in make(a, N, D, H, W), make(b, N, D, H, W):
        dy *= sign.reshape(D, 1, 1)
        native.set_option('conv_fp32_split', 2)
        got = _three_products(geo, x, w, dy)
        native.set_option('conv_fp32_split', 0)
        for p, q, what in zip(got, _three_products(geo, x, w, dy), ('y', 'dx', 'dw')):
            assert torch.equal(p.isnan(), q.isnan()) and torch.equal(p.nan_to_num(0.0), q.nan_to_num(0.0)), what
            assert torch.equal(p.isinf(), q.isinf()), what


def _errors_of_both_ways(shape):
    """Errors (2-norm, relative) against 64 bits of y, dx and dw of a layer, from parts and by the fp32 kernels."""
    N, C, H, W, D, kernel, pad, stride, dil = shape
    g = torch.Generator().manual_seed(94)
    x, w = torch.randn(N, C, H, W, generator=g), torch.randn(D, C, *kernel, generator=g)
    xr, wr = x.double().requires_grad_(True), w.double().requires_grad_(True)
    y_ref = F.conv2d(xr, wr, None, stride=stride, padding=pad, dilation=dil)
    dy = torch.randn(y_ref.shape, generator=g)
    y_ref.backward(dy.double())
    geo = _ci(N, C, H, W, D, kernel[0], kernel[1], pad[0], pad[1], stride[0], stride[1], dil[0], dil[1])
    errors = []
    for option in 2, 0:
        native.set_option('conv_fp32_split', option)
        got = _three_products(geo, x.cuda(), w.cuda(), dy.cuda())
        errors.append([((a.cpu().double() - b).norm() / b.norm()).item() for a, b in zip(got, (y_ref.detach(), xr.grad, wr.grad))])
    return errors


@pytest.mark.parametrize('shape', [
    # N, C, H, W, D, kernel, pad, stride, dilation: sums of sixteen terms (y, dx, dw in turn) and of more
    (4, 16, 24, 28, 64, (1, 1), (0, 0), (1, 1), (1, 1)),
    (4, 64, 24, 28, 16, (1, 1), (0, 0), (1, 1), (1, 1)),
    (1, 64, 4, 4, 130, (1, 1), (0, 0), (1, 1), (1, 1)),
    (2, 48, 23, 17, 64, (3, 3), (1, 1), (2, 2), (1, 1)),     # dx: 64 to 256 terms
    (4, 64, 24, 28, 256, (3, 3), (1, 1), (1, 1), (1, 1)),
    (2, 256, 20, 21, 130, (5, 5), (2, 2), (1, 1), (1, 1)),
    (24, 384, 13, 13, 500, (3, 3), (1, 1), (2, 2), (1, 1)),   # dx: phases, whose sums are cut as those of all taps would be
])
def test_sums_of_parts_are_no_further_off_than_the_fp32_kernels(shape, split_always):
    for parts, fp32, what in zip(*_errors_of_both_ways(shape), ('y', 'dx', 'dw')):
        assert parts <= fp32, (what, parts, fp32)


@pytest.mark.parametrize('hw', [(8, 16), (11, 13)])
@pytest.mark.parametrize('channel', [0, 15, 16, 40, 63, 64, 79])
def test_every_wavefront_of_a_conversion_tells_what_it_found(channel, hw, split_always):
    """An infinity anywhere in a tile of 64 pixels x 64 channels sends the product to the fp32 kernels, where it stays one (its
    parts would make it NaN)."""
    N, C, D = 2, 80, 64
    g = torch.Generator(device='cuda').manual_seed(97)
    w = torch.rand(D, C, 1, 1, generator=g, device='cuda') + 0.5
    y = torch.empty(N, D, *hw, device='cuda')
    for pixel in 0, 31, 32, 63, hw[0] * hw[1] - 1:
        x = torch.randn(N, C, *hw, generator=g, device='cuda')
        x.view(N, C, -1)[1, channel, pixel] = float('inf')
        _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(x), _ptr(w), _ptr(w), ctypes.c_int(0),
              *_ci(N, C, *hw, D, 1, 1, 0, 0, 1, 1, 1, 1), _ptr(y))
        got = y.view(N, D, -1)
        assert (got[1, :, pixel] == float('inf')).all()
        assert torch.isfinite(got).sum().item() == got.numel() - D


def test_one_product_of_parts_is_within_two_half_units(split_always):
    """What six products of parts leave out of one of fp32 is at most 2^-24 of it, and the result's rounding another
    2^-24 (the fp32 kernels': the rounding alone)."""
    N, D, P = 1, 64, 64 * 64
    g = torch.Generator().manual_seed(95)
    x, w = torch.rand(N, 1, 64, 64, generator=g) + 1, torch.rand(D, 1, 1, 1, generator=g) + 1
    y = torch.empty(N, D, 64, 64, device='cuda')
    xd, wd = x.cuda(), w.cuda()
    _call('conv2d_forward_c6a7aa85', ctypes.c_int(y.numel()), _ptr(xd), _ptr(wd), _ptr(wd), ctypes.c_int(0),
          *_ci(N, 1, 64, 64, D, 1, 1, 0, 0, 1, 1, 1, 1), _ptr(y))
    want = w.double().reshape(D, 1) * x.double().reshape(1, P)
    off = ((y.cpu().double().reshape(D, P) - want) / want).abs().max().item()
    assert off <= 2.0 ** -23 * (1 + 2.0 ** -7), off


@pytest.mark.parametrize('filters', [1, 2])
def test_sums_of_a_few_terms_are_not_formed_from_parts_by_choice(filters):
    """At a stride of two a pixel of dx meets one to four taps: parts, which would be faster, lose bits of such sums."""
    N, C, H, W = 16, 64, 97, 99
    geo = _ci(N, C, H, W, filters, 3, 3, 1, 1, 2, 2, 1, 1)
    g = torch.Generator(device='cuda').manual_seed(96)
    dy = torch.randn(N, filters, 49, 50, generator=g, device='cuda')
    w = torch.randn(filters, C, 3, 3, generator=g, device='cuda')
    out = []
    try:
        for option in 1, 0:
            native.set_option('conv_fp32_split', option)
            out.append(torch.empty(N, C, H, W, device='cuda'))
            _call('conv2d_backward_data_ecf81c91', ctypes.c_int(out[-1].numel()), _ptr(dy), _ptr(w), ctypes.c_int(0), *geo,
                  _ptr(out[-1]))
    finally:
        native.set_option('conv_fp32_split', 1)
    assert torch.equal(*out)


@pytest.fixture
def halves_always():
    native.set_option('conv_fp32_split', 3)
    yield
    native.set_option('conv_fp32_split', 1)


def _layer(shape, seed, scale=1.0):
    """x, w, dy of a layer, its geometry, the three products in 64 bits, and the terms of their sums."""
    N, C, H, W, D, kernel, pad, stride, dil = shape
    g = torch.Generator().manual_seed(seed)
    x, w = torch.randn(N, C, H, W, generator=g) * scale, torch.randn(D, C, *kernel, generator=g) / scale
    xr, wr = x.double().requires_grad_(True), w.double().requires_grad_(True)
    y_ref = F.conv2d(xr, wr, None, stride=stride, padding=pad, dilation=dil)
    dy = torch.randn(y_ref.shape, generator=g)
    y_ref.backward(dy.double())
    geo = _ci(N, C, H, W, D, kernel[0], kernel[1], pad[0], pad[1], stride[0], stride[1], dil[0], dil[1])
    terms = C * kernel[0] * kernel[1], D * kernel[0] * kernel[1], dy[:, 0].numel()
    return (x.cuda(), w.cuda(), dy.cuda()), geo, (y_ref.detach(), xr.grad, wr.grad), terms


@pytest.mark.parametrize('scale', [1.0, 2.0 ** -40, 2.0 ** 70])
@pytest.mark.parametrize('shape', [
    # N, C, H, W, D, kernel, pad, stride, dilation
    (1, 1, 1, 1, 1, (1, 1), (0, 0), (1, 1), (1, 1)),         # one multiply-add
    (3, 16, 5, 3, 64, (1, 1), (0, 0), (1, 1), (1, 1)),       # one step of K; 15 pixels an image
    (40, 17, 2, 2, 65, (2, 2), (1, 1), (1, 1), (1, 1)),      # rows and channels one past a tile and a block
    (2, 272, 9, 10, 128, (1, 1), (0, 0), (1, 1), (1, 1)),    # 17 steps: sums that move once, whole rows of tiles
    (2, 33, 19, 21, 193, (3, 2), (2, 0), (1, 1), (1, 1)),    # odd planes: the element-wise conversion
    (4, 128, 24, 28, 256, (3, 3), (1, 1), (1, 1), (1, 1)),   # 72 and more steps: sums that move every sixteen
    (3, 48, 23, 17, 257, (3, 3), (0, 1), (2, 2), (1, 1)),    # strides: taps that reach no pixel
    (2, 24, 30, 22, 40, (3, 2), (2, 1), (2, 1), (1, 2)),     # strides and dilation
])
def test_fp32_products_of_two_halves(shape, scale, halves_always):
    """Operands of 23 bits and a sign (2^-23 of a value at most), the tails' product left out (2^-22), and up to six fp32
    roundings for sixteen of K, each of 2^-24 of a sum no larger than the result's own scale: the latter add up as
    their squares.  Operands of any scale."""
    (x, w, dy), geo, want, terms = _layer(shape, 97, scale)
    _leave_nan_patterns_in_the_workspace()
    got = _three_products(geo, x, w, dy)
    for a, b, k, what in zip(got, want, terms, ('y', 'dx', 'dw')):
        error = ((a.cpu().double() - b).norm() / b.norm()).item()
        assert error <= 2.0 ** -24 * (1 + 2 + 2 + 4 + (6 * (k / 16 + 1)) ** 0.5), (what, error)
    start = [torch.randn(t.shape, generator=torch.Generator().manual_seed(98)).cuda() * t.abs().max() for t in (x, w)]
    again = _three_products(geo, x, w, dy, *start)
    assert torch.equal(again[0], got[0])
    assert torch.equal(again[1], start[0] + got[1]) and torch.equal(again[2], start[1] + got[2])


@pytest.mark.parametrize('odd', ['lone pixel', 'lone channel', 'small beside large', 'listed', 'one more', 'far larger', 'unseen', 'inf',
                                 'nan', 'overflow'])
def test_values_that_two_halves_do_not_stand_for(odd, halves_always):
    """Up to 128 values of a tensor that are out of the range of two halves are listed and added behind the product; a tensor with
    more is multiplied in three parts (the same bits as when they are asked for), one that is not finite by the fp32
    kernels."""
    shape = (2, 96, 80, 80, 64, (3, 3), (1, 1), (1, 1), (1, 1))     # x: 1.2 million elements, an eighth of them looked at
    (x, w, dy), geo, _, _ = _layer(shape, 99)
    dy[:, :, 10:30] = 0.0
    if odd == 'lone pixel':            # 64 channels of a pixel, and what lies beside them, 2^-30 of the rest
        x[1, :64, 7, 9] *= 2.0 ** -30
        dy[0, :, 40, 3] *= 2.0 ** -30
    elif odd == 'lone channel':
        x[:, 5] *= 2.0 ** -30
    elif odd == 'small beside large':
        x[1, 3, 7, 9] *= 2.0 ** -60
        dy[0, 1, 40, 3] = 1e-40
    elif odd in ('listed', 'one more'):
        x.view(-1)[:9000 * (128 + (odd == 'one more')):9000] *= 2.0 ** -40
    elif odd == 'far larger':          # than all others: a thousand of them lie below 2^-27 of it
        x.view(-1)[5024] = 1e5
    elif odd == 'unseen':              # (the line of elements 4992 to 5023 is not looked at)
        x.view(-1)[5000] = 1e5
    elif odd == 'overflow':
        x.abs_().mul_(2.0 ** 124), w.abs_().mul_(2.0 ** 20), dy.abs_().mul_(2.0 ** 60)   # (of one sign: whatever the order)
    else:
        x[1, 3, 7, 9] = float(odd)
    got = _three_products(geo, x, w, dy)
    native.set_option('conv_fp32_split', 2)
    parts = _three_products(geo, x, w, dy)
    native.set_option('conv_fp32_split', 0)
    want = _three_products(geo, x, w, dy)
    for a, b, what in zip(got, want, ('y', 'dx', 'dw')):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf()), what
        fine = b.isfinite()
        assert (a[fine].double() - b[fine].double()).norm() <= 2e-6 * b[fine].double().norm(), what
    same = [torch.equal(a.nan_to_num(), b.nan_to_num()) for a, b in zip(got, parts)]
    # which products left the halves
    assert same == {'lone pixel': [False, False, False], 'lone channel': [True, False, True],
                    'small beside large': [False, False, False], 'listed': [False, False, False], 'one more': [True, False, True],
                    'far larger': [True, False, True], 'unseen': [False, False, False], 'inf': [True, False, True], 'nan': [True, False, True],
                    'overflow': [True, False, True]}[odd]


def _made_of_small_values(shape, which, scale, few, seed):
    """x, w, dy of which `which` holds small values (scale times the rest; scale 0: subnormals) that make up whole results:
    what would meet larger values beside them is zero in the other operand.  few: in a few places, else wherever there
    are any of that kind."""
    N, C, H, W, D, kernel, pad, stride, dil = shape
    g = torch.Generator().manual_seed(seed)
    x, w = torch.randn(N, C, H, W, generator=g), torch.randn(D, C, *kernel, generator=g)
    dy = torch.randn(F.conv2d(x, w, None, stride=stride, padding=pad, dilation=dil).shape, generator=g)

    def small(t):
        return t.sign() * 2.0 ** -133 if scale == 0 else t * scale

    def small_above(t, c):
        """Channel c of t: small values in the rows above the eighth, larger ones from the twelfth on."""
        kept = torch.zeros_like(t[:, c])
        where = (slice(None), slice(3, 5), slice(4, 6)) if few else (slice(None), slice(0, 8))
        kept[where] = small(t[:, c][where])
        kept[:, 12:] = t[:, c, 12:]
        t[:, c] = kept
    if which == 'all':       # one value in twenty is not zero, and a few of those are small: they meet each other, too
        for t in x, w, dy:
            t.mul_(torch.rand(t.shape, generator=g) < 0.05)
            flat = t.view(-1)
            places = flat.nonzero().flatten()
            places = places[torch.randperm(len(places), generator=g)[:40 if few else len(places) // 3]]
            flat[places] = small(flat[places])
    elif which == 'x':
        small_above(x, 5)
        w[:3, [c for c in range(C) if c != 5]] = 0.0   # filters that read this channel alone
        dy[:, :3, 3:] = 0.0                            # and whose gradients do not meet its larger values
    elif which == 'w':
        index = (slice(1, 2), slice(7, 9)) if few else (slice(0, 2),)
        w[index] = small(w[index])
        x[:, [c for c in range(C) if c not in (7, 8)], :8] = 0.0   # where nothing but these channels is not zero
        dy[:, [d for d in range(D) if d != 1], :8] = 0.0           # and nothing but this filter's gradient
    else:
        small_above(dy, 2)
        w[[d for d in range(D) if d != 2], 1] = 0.0    # a channel that this filter alone reads
        x[:, :2, 8:] = 0.0                             # and whose values do not meet the gradient's larger ones
    return x, w, dy


@pytest.mark.parametrize('few', [True, False])
@pytest.mark.parametrize('scale', [2.0 ** 30, 2.0 ** -24, 2.0 ** -40, 0.0])
@pytest.mark.parametrize('which', ['x', 'w', 'dy', 'all'])
@pytest.mark.parametrize('shape', [
    (2, 64, 16, 19, 64, (3, 3), (1, 1), (1, 1), (1, 1)),
    (3, 33, 21, 18, 65, (3, 2), (2, 1), (2, 1), (1, 2)),         # strides, dilation, odd counts
    (2, 96, 80, 80, 64, (3, 3), (1, 1), (1, 1), (1, 1)),         # more than a million elements
])
def test_results_that_small_values_alone_make_up(shape, which, scale, few, halves_always):
    """A value that is small for its tensor makes up a result where the larger ones beside it meet zeros.  Element by element
    against 64 bits: four and a half units of the magnitudes that are added (2^-23 of a value for either operand's last bit,
    2^-22 for the product of the tails, 2^-24 for the result; the roundings within sums are far below that of so many
    terms, but for a few values that are larger than all others: there every later one of up to six for sixteen
    terms is 2^-24 of the whole).  Subnormal results
    besides: half of 2^-149 for every product that is not zero (the fp32 kernels, which take tensors with many of
    them, round each) and for the result."""
    x, w, dy = _made_of_small_values(shape, which, scale, few, 107)
    N, C, H, W, D, kernel, pad, stride, dil = shape
    geo = _ci(N, C, H, W, D, kernel[0], kernel[1], pad[0], pad[1], stride[0], stride[1], dil[0], dil[1])
    want, sizes, products = [], [], []
    for out, f in (want, lambda t: t.double()), (sizes, lambda t: t.double().abs()), (products, lambda t: (t != 0).double()):
        xr, wr = f(x).requires_grad_(True), f(w).requires_grad_(True)
        y = F.conv2d(xr, wr, None, stride=stride, padding=pad, dilation=dil)
        y.backward(f(dy))
        out += [y.detach(), xr.grad, wr.grad]
    _leave_nan_patterns_in_the_workspace()
    got = _three_products(geo, x.cuda(), w.cuda(), dy.cuda())
    terms = C * kernel[0] * kernel[1], D * kernel[0] * kernel[1], dy[:, 0].numel()
    for a, b, size, count, k, what in zip(got, want, sizes, products, terms, ('y', 'dx', 'dw')):
        units = 2.0 ** -21 + 2.0 ** -24 + (2.0 ** -24 * 6 * (k / 16 + 1) if scale > 1 else 0.0)
        off = (a.cpu().double() - b).abs() - (units * size + 2.0 ** -150 * (count + 1))
        assert (off <= 0).all(), (what, float((off / size.clamp_min(1e-300)).max()), int((off > 0).sum()))


@pytest.mark.parametrize('shape', [
    (4, 64, 24, 28, 256, (3, 3), (1, 1), (1, 1), (1, 1)),        # 576 terms, and pieces of K
    (16, 64, 56, 56, 128, (3, 3), (1, 1), (1, 1), (1, 1)),
    (2, 256, 60, 61, 130, (5, 5), (2, 2), (1, 1), (1, 1)),
])
def test_sums_formed_by_choice_are_no_further_off_than_those_of_three_parts_or_fp32(shape):
    (x, w, dy), geo, want, _ = _layer(shape, 100)
    errors = {}
    try:
        for option in 1, 2, 0:
            native.set_option('conv_fp32_split', option)
            errors[option] = [((a.cpu().double() - b).norm() / b.norm()).item()
                              for a, b in zip(_three_products(geo, x, w, dy), want)]
    finally:
        native.set_option('conv_fp32_split', 1)
    for chosen, parts, fp32, what in zip(errors[1], errors[2], errors[0], ('y', 'dx', 'dw')):
        assert chosen <= 1.02 * max(parts, fp32), (what, chosen, parts, fp32)

def test_sums_that_three_parts_cut_shorter_are_left_to_them():
    """A weight gradient of few pixels, which is cut along K: shorter sums in three parts than in halves, and nearer."""
    (x, w, dy), geo, want, _ = _layer((8, 512, 14, 14, 512) + ((3, 3), (1, 1), (1, 1), (1, 1)), 100)
    errors = {}
    try:
        for option in 1, 2:
            native.set_option('conv_fp32_split', option)
            errors[option] = ((_three_products(geo, x, w, dy)[2].cpu().double() - want[2]).norm() / want[2].norm()).item()
    finally:
        native.set_option('conv_fp32_split', 1)
    assert errors[1] <= 1.02 * errors[2]


def test_halves_in_a_recorded_graph(halves_always):
    """What is known of the operands is found anew by every replay: halves, three parts, halves with a few listed values."""
    shape = (2, 64, 24, 28, 128, (3, 3), (1, 1), (1, 1), (1, 1))
    (x, w, dy), geo, _, _ = _layer(shape, 101)
    usual, odd, few = x.clone(), x.clone(), x.clone()
    few[1, 3, 7:9, 9] *= 2.0 ** -30
    odd[1, :, 7, 9] *= 2.0 ** -30
    odd[0, 5] *= 2.0 ** -30
    lib, stream = native.library(), torch.cuda.Stream()
    y, dx, dw = torch.empty_like(dy), torch.empty_like(x), torch.empty_like(w)

    def call(on=None):
        native.begin_call(on, [])
        lib.conv2d_forward_c6a7aa85(ctypes.c_int(0), ctypes.c_int(y.numel()), _ptr(x), _ptr(w), _ptr(w), ctypes.c_int(0),
                                    *geo, _ptr(y))
        lib.mobula_hip_conv2d_backward(ctypes.c_int(0), _ptr(dy), _ptr(x), _ptr(w), *geo, _ptr(dx), _ptr(dw))
        native.end_call('conv2d')
    try:
        want = []
        for values in usual, odd, few:
            x.copy_(values)
            call()
            torch.cuda.synchronize()
            want.append([t.clone() for t in (y, dx, dw)])
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            call(on=torch.cuda.current_stream().cuda_stream)
        for which in (0, 1, 2, 0, 0, 2, 1):
            x.copy_((usual, odd, few)[which])
            for t in (y, dx, dw):
                t.fill_(float('nan'))
            graph.replay()
            torch.cuda.synchronize()
            for a, b in zip((y, dx, dw), want[which]):
                assert torch.equal(a, b)
        del graph
    finally:
        native.unpin_workspace()
