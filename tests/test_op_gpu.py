"""GPU tests of the Python surface: `mobula.op.ROIAlign` through the torch and
NumPy glues and `mobula.func.*` directly, checked against the CPU oracle."""
import numpy as np
import pytest

torch = pytest.importorskip('torch')

from mobulaop_amd import native, workloads  # noqa: E402
from mobulaop_amd.testing import assert_parity  # noqa: E402
from oracle import roialign as oracle  # noqa: E402

pytestmark = pytest.mark.gpu
FWD_TOL, BWD_TOL = 1e-5, 1e-4


@pytest.fixture(autouse=True)
def _announce(request):
    print('\n[case] {}'.format(request.node.nodeid), flush=True)


def _small():
    w = workloads.make_workload('cfg2', scale_down=32)
    want_y = oracle.forward(w['data'], w['rois'], w['pooled_size'], w['spatial_scale'],
                            w['sampling_ratio'])
    want_dx = oracle.backward(w['dy'], w['rois'], w['data'].shape, w['spatial_scale'],
                              w['sampling_ratio'], impl='ordered')
    return w, want_y, want_dx


def test_reference_example_through_torch(mobula):
    # examples/RunROIAlign.py:12-26 with torch tensors on the GPU
    x = torch.arange(2 * 3 * 4 * 4, dtype=torch.float32, device='cuda').reshape(2, 3, 4, 4)
    x.requires_grad_(True)
    rois = torch.tensor([[0, 1, 1, 3, 3]], dtype=torch.float32, device='cuda')
    out = mobula.op.ROIAlign(data=x, rois=rois, pooled_size=(2, 2), spatial_scale=1.0,
                             sampling_ratio=1)
    out.backward(torch.ones_like(out))
    want = torch.tensor([[7.5, 8.5], [11.5, 12.5]], device='cuda')
    for c in range(3):
        assert torch.equal(out[0, c].detach(), want + 16 * c)
    k = torch.tensor([[.25, .5, .25], [.5, 1, .5], [.25, .5, .25]], device='cuda')
    assert torch.equal(x.grad[0, 0, 1:4, 1:4], k) and float(x.grad[1].abs().sum()) == 0


def test_torch_autograd_path(mobula):
    w, want_y, want_dx = _small()
    x = torch.from_numpy(w['data']).cuda().requires_grad_(True)
    rois = torch.from_numpy(w['rois']).cuda().requires_grad_(True)
    y = mobula.op.ROIAlign(x, rois, pooled_size=w['pooled_size'],
                           spatial_scale=w['spatial_scale'], sampling_ratio=w['sampling_ratio'])
    assert y.requires_grad and y.shape == want_y.shape
    y.backward(torch.from_numpy(w['dy']).cuda())
    assert_parity(y, want_y, FWD_TOL, 'y')
    assert_parity(x.grad, want_dx, BWD_TOL, 'dx')
    assert float(rois.grad.abs().max()) == 0      # no gradient to the boxes
    # a second backward accumulates into .grad exactly once
    y2 = mobula.op.ROIAlign(x, rois, pooled_size=w['pooled_size'],
                            spatial_scale=w['spatial_scale'], sampling_ratio=w['sampling_ratio'])
    y2.backward(torch.from_numpy(w['dy']).cuda())
    assert_parity(x.grad, 2 * want_dx, BWD_TOL, 'dx twice')


def test_numpy_path_stages_through_the_gpu(mobula):
    w, want_y, want_dx = _small()
    op = mobula.op.ROIAlign[np.ndarray](pooled_size=w['pooled_size'],
                                        spatial_scale=w['spatial_scale'],
                                        sampling_ratio=w['sampling_ratio'])
    y = op(w['data'], w['rois'])
    assert isinstance(y, np.ndarray)
    assert_parity(y, want_y, FWD_TOL, 'y')
    dx, drois = op.backward(w['dy'])
    assert_parity(dx, want_dx, BWD_TOL, 'dx')
    assert not drois.any()
    # req = add accumulates into the caller's gradient, req = null leaves it alone
    base = np.ones_like(w['data'])
    op.backward(w['dy'], in_grad=[base, np.zeros_like(w['rois'])], req=['add', 'null'])
    assert_parity(base, want_dx + 1, BWD_TOL, 'dx add')


def test_direct_function_calls_kwargs_and_strided_tensors(mobula):
    w, want_y, want_dx = _small()
    N, C, H, W = w['data'].shape
    PH, PW = w['pooled_size']
    x = torch.from_numpy(w['data']).cuda()
    rois = torch.from_numpy(w['rois']).cuda()
    # output written through a non-contiguous view: copied back after the call
    backing = torch.zeros(want_y.shape[0], C, PH, 2 * PW, device='cuda')
    y_view = backing[..., ::2]
    assert not y_view.is_contiguous()
    mobula.func.roi_align_forward(
        nthreads=y_view.numel(), bottom_data=x, spatial_scale=w['spatial_scale'], channels=C,
        height=H, width=W, pooled_height=PH, pooled_width=PW, sampling_ratio=w['sampling_ratio'],
        bottom_rois=rois, top_data=y_view)
    assert_parity(backing[..., ::2], want_y, FWD_TOL, 'strided y')
    assert float(backing[..., 1::2].abs().sum()) == 0
    # strided input
    x_t = torch.from_numpy(np.ascontiguousarray(w['data'].transpose(0, 1, 3, 2))).cuda().transpose(2, 3)
    assert not x_t.is_contiguous()
    y = torch.empty(want_y.shape, device='cuda')
    mobula.func.roi_align_forward(y.numel(), x_t, w['spatial_scale'], C, H, W, PH, PW,
                                  w['sampling_ratio'], rois, y)
    assert_parity(y, want_y, FWD_TOL, 'strided x')
    dx = torch.zeros(N, C, H, W, device='cuda')
    mobula.func.roi_align_backward(y.numel(), torch.from_numpy(w['dy']).cuda(), w['spatial_scale'],
                                   C, H, W, PH, PW, w['sampling_ratio'], dx, rois)
    assert_parity(dx, want_dx, BWD_TOL, 'dx')


def test_errors_surface_as_python_exceptions(mobula):
    x = torch.rand(1, 2, 4, 4, device='cuda')
    rois = torch.zeros(2, 5, device='cuda')
    y = torch.empty(3, 2, 2, 2, device='cuda')  # claims 3 ROIs, rois has 2
    with pytest.raises(RuntimeError):
        mobula.func.roi_align_forward(y.numel(), x, 1.0, 2, 4, 4, 2, 2, 2, rois, y)
    with pytest.raises(AssertionError):          # host and device tensor in one call
        mobula.func.roi_align_forward(8, x, 1.0, 2, 4, 4, 2, 2, 2, rois.cpu().numpy(), y)


def test_runs_on_the_callers_stream(mobula):
    w, want_y, _ = _small()
    x = torch.from_numpy(w['data']).cuda()
    rois = torch.from_numpy(w['rois']).cuda()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = mobula.op.ROIAlign(x, rois, pooled_size=w['pooled_size'],
                               spatial_scale=w['spatial_scale'],
                               sampling_ratio=w['sampling_ratio'])
        doubled = y * 2          # ordered after the kernel on the same stream
    side.synchronize()
    assert_parity(doubled, 2 * want_y, FWD_TOL, 'stream')


def test_channels_last_tensors_take_the_channels_last_path(mobula):
    # same numbers as with NCHW tensors; outputs and gradients come back channels-last
    torch.manual_seed(5)
    x = torch.randn(2, 32, 20, 24, device='cuda')
    rois = torch.tensor([[0, 1, 2, 60, 50], [1, 10, 10, 90, 70], [1, -5, 3, 20, 100]], device='cuda',
                        dtype=torch.float32)
    kw = dict(pooled_size=(7, 7), spatial_scale=0.25, sampling_ratio=2)
    xa = x.clone().requires_grad_(True)
    ya = mobula.op.ROIAlign(xa, rois, **kw)
    dy = torch.randn_like(ya)
    ya.backward(dy)
    xb = x.clone().to(memory_format=torch.channels_last).requires_grad_(True)
    yb = mobula.op.ROIAlign(xb, rois, **kw)
    assert yb.is_contiguous(memory_format=torch.channels_last) and not yb.is_contiguous()
    yb.backward(dy)
    assert xb.grad.is_contiguous(memory_format=torch.channels_last)
    assert float((ya - yb).detach().abs().max()) <= 1e-5 * float(ya.detach().abs().max())
    assert float((xa.grad - xb.grad).abs().max()) <= 1e-4 * float(xa.grad.abs().max())


@pytest.mark.parametrize('low,tol', [(torch.float16, 2e-3), (torch.bfloat16, 8e-3)])
def test_half_precision_training_step(mobula, low, tol):
    # 16-bit map and gradients through the operator: both passes run in the library
    # (bfloat16 carries 8 significant bits: 4e-3 per rounding)
    torch.manual_seed(6)
    x32 = torch.randn(2, 64, 20, 24, device='cuda')
    rois = torch.tensor([[0, 1, 2, 60, 50], [1, 10, 10, 90, 70], [1, -5, 3, 20, 100]], device='cuda',
                        dtype=torch.float32)
    kw = dict(pooled_size=(7, 7), spatial_scale=0.25, sampling_ratio=2)
    xh = x32.to(low).requires_grad_(True)
    yh = mobula.op.ROIAlign(xh, rois, **kw)
    assert yh.dtype == low
    dy = torch.randn_like(yh)
    yh.backward(dy)
    assert xh.grad.dtype == low
    xf = x32.to(low).float().requires_grad_(True)
    yf = mobula.op.ROIAlign(xf, rois, **kw)
    yf.backward(dy.float())
    assert float((yh.detach().float() - yf.detach()).abs().max()) <= tol * float(yf.detach().abs().max())
    assert float((xh.grad.float() - xf.grad).abs().max()) <= tol * float(xf.grad.abs().max())
    # channels-last 16-bit maps: the forward reads them where they lie
    xc = x32.to(low).contiguous(memory_format=torch.channels_last)
    xc.requires_grad_(True)
    yc = mobula.op.ROIAlign(xc, rois, **kw)
    assert float((yc.detach().float() - yf.detach()).abs().max()) <= tol * float(yf.detach().abs().max())
    yc.backward(dy.contiguous(memory_format=torch.channels_last))
    assert xc.grad.dtype == low and xc.grad.is_contiguous(memory_format=torch.channels_last)
    assert float((xc.grad.float() - xf.grad).abs().max()) <= tol * float(xf.grad.abs().max())


def test_double_tensors_through_the_operator(mobula):
    """float64 data and boxes resolve to the double instantiation; autograd gets dx."""
    rng = np.random.default_rng(9)
    xh = rng.standard_normal((2, 3, 12, 14))
    rh = np.array([[0, 2.5, 3.5, 30.25, 28.0], [1, -4, 0, 20, 44], [1, 8, 8, 8, 8]], dtype=np.float64)
    dyh = rng.standard_normal((3, 3, 4, 4))
    x = torch.from_numpy(xh).cuda().requires_grad_(True)
    rois = torch.from_numpy(rh).cuda()
    y = mobula.op.ROIAlign(x, rois, pooled_size=(4, 4), spatial_scale=0.25, sampling_ratio=0)
    assert y.dtype == torch.float64
    np.testing.assert_array_equal(y.detach().cpu().numpy(), oracle.forward_f64(xh, rh, (4, 4), 0.25, 0))
    y.backward(torch.from_numpy(dyh).cuda())
    np.testing.assert_allclose(x.grad.cpu().numpy(), oracle.backward_f64(dyh, rh, xh.shape, 0.25, 0),
                               rtol=0, atol=1e-13)
    # host arrays take the same symbols (device id -1: staged through the GPU)
    out = np.zeros((3, 3, 4, 4))
    mobula.func.roi_align_forward(out.size, xh, 0.25, 3, 12, 14, 4, 4, 0, rh, out)
    np.testing.assert_array_equal(out, oracle.forward_f64(xh, rh, (4, 4), 0.25, 0))


@pytest.mark.parametrize('form', ['plain', 'channels_last', 'transposed', 'channels_last_odd', 'one_bin'])
def test_direct_calls_agree_with_the_operator_class(mobula, form):
    """Calls on torch GPU tensors go straight to the library; the operator class gives the same values,
    formats and gradients (also for strided maps, expanded gradients and boxes that want one)."""
    torch.manual_seed(7)
    C, pooled = (6, (3, 5)) if form == 'channels_last_odd' else (8, (1, 1) if form == 'one_bin' else (3, 5))
    x = torch.randn(2, C, 12, 9, device='cuda')
    if form.startswith('channels_last') or form == 'one_bin':
        x = x.contiguous(memory_format=torch.channels_last)
    elif form == 'transposed':
        x = x.transpose(2, 3)
    rois = torch.tensor([[0, 1, 2, 30, 20], [1, -4, 3, 25, 40], [1, 8, 8, 9, 9]], device='cuda', dtype=torch.float32)
    rois.requires_grad_(True)
    kw = dict(pooled_size=pooled, spatial_scale=0.25, sampling_ratio=2)
    handle, results = mobula.op.ROIAlign, []
    handle(x, rois, **kw)
    direct = handle.direct
    assert direct is not None
    for call in (direct, None):
        handle.direct = call
        xi = x.detach().requires_grad_(True)
        y = handle(data=xi, rois=rois, **kw)
        results.append((y,) + torch.autograd.grad((2 * y).sum(), (xi, rois)))
    handle.direct = direct
    for a, b in zip(*results):
        assert a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.parametrize('context', ['grad', 'vmap', 'vmap_of_another', 'forward_ad', 'trace', 'fake', 'mode'])
def test_direct_calls_leave_transformed_calls_to_the_operator_class(mobula, context):
    """torch.func, tracing, forward mode and dispatch modes have to see the autograd function."""
    from torch.autograd import forward_ad
    from torch.utils.flop_counter import FlopCounterMode
    direct = native.torch_direct().ROIAlign
    x = torch.randn(1, 4, 8, 9, device='cuda')
    rois = torch.tensor([[0, 1, 2, 30, 20]], device='cuda', dtype=torch.float32)
    kw = dict(pooled_size=(2, 2), spatial_scale=0.25, sampling_ratio=2)
    seen = []

    def call(a):
        seen.append(direct(a, rois, **kw))
        return a.sum()

    def call_on_captured(a):
        seen.append(direct(x, rois, **kw))
        return a.sum()
    if context == 'grad':
        torch.func.grad(call)(x)
    elif context == 'vmap':
        torch.func.vmap(call)(x[None])
    elif context == 'vmap_of_another':
        torch.func.vmap(call_on_captured)(x)
    elif context == 'forward_ad':
        with forward_ad.dual_level():
            call(forward_ad.make_dual(x, torch.ones_like(x)))
    elif context == 'trace':
        torch.jit.trace(call, (x,), check_trace=False)
    elif context == 'fake':
        from torch._subclasses.fake_tensor import FakeTensorMode
        with FakeTensorMode() as mode:
            call(mode.from_tensor(x))
    else:
        with FlopCounterMode(display=False):
            call(x)
    assert seen == [NotImplemented]


def test_memory_kept_after_host_arrays_is_counted_and_given_back(mobula):
    """The device copies of host arrays outlive a call: they are part of what the library says it holds."""
    native.release_workspace()
    assert native.workspace_bytes() == 0
    x = np.ones((2, 64, 90, 91), dtype=np.float32)
    y = np.empty((3, 64, 2, 2), dtype=np.float32)
    rois = np.zeros((3, 5), dtype=np.float32)
    mobula.func.roi_align_forward(y.size, x, 1.0, 64, 90, 91, 2, 2, 2, rois, y)
    held = native.workspace_bytes()
    assert held >= x.nbytes + y.nbytes + rois.nbytes
    assert native.release_workspace() == held
    assert native.workspace_bytes() == 0 and native.release_workspace() == 0


@pytest.mark.parametrize('kind', ['forward_pre', 'forward', 'full_backward_pre', 'full_backward'])
def test_hooks_on_all_modules_see_direct_calls(mobula, kind):
    """The operator class's call is a module's: with such a hook registered it keeps the call."""
    from torch.nn.modules import module
    x = torch.randn(1, 4, 8, 9, device='cuda', requires_grad=True)
    rois = torch.tensor([[0, 1, 2, 30, 20]], device='cuda', dtype=torch.float32)
    kw = dict(pooled_size=(2, 2), spatial_scale=0.25, sampling_ratio=2)
    for _ in range(2):
        mobula.op.ROIAlign(x, rois, **kw)
    seen = []
    hook = getattr(module, 'register_module_{}_hook'.format(kind))(lambda m, *a: seen.append(type(m).__name__))
    try:
        mobula.op.ROIAlign(x, rois, **kw).sum().backward()
    finally:
        hook.remove()
    assert seen == ['_ROIAlign_TORCH_NN_MODULE']
    assert isinstance(native.torch_direct().ROIAlign(x, rois, **kw), torch.Tensor)   # (and not without one)


def test_direct_backward_refuses_batched_gradients(mobula):
    x = torch.randn(1, 4, 8, 9, device='cuda', requires_grad=True)
    rois = torch.tensor([[0, 1, 2, 30, 20]], device='cuda', dtype=torch.float32)
    y = native.torch_direct().ROIAlign(x, rois, (2, 2), 0.25, 2)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(y, x, torch.ones((3,) + y.shape, device='cuda'), is_grads_batched=True)


def test_adaptive_backward_does_not_wait_for_a_busy_stream(mobula):
    """Nothing of a dense grid's backward is awaited by the host: the call returns with the stream still at work, and gives
    what it gives on an idle one."""
    x = torch.randn(1, 4, 24, 25, device='cuda', requires_grad=True)
    rois = torch.tensor([[0, 1, 2, 80, 90]], device='cuda', dtype=torch.float32)
    a = torch.randn(4096, 4096, device='cuda')
    kw = dict(pooled_size=(2, 2), spatial_scale=0.25, sampling_ratio=0)
    (want,) = torch.autograd.grad(mobula.op.ROIAlign(x, rois, **kw).sum(), x)
    y = mobula.op.ROIAlign(x, rois, **kw).sum()
    for _ in range(30):
        a = (a @ a) * 1e-3
    (got,) = torch.autograd.grad(y, x)
    assert not torch.cuda.current_stream().query()   # (some forty milliseconds of products)
    assert torch.equal(got, want)


@pytest.mark.parametrize('bias,image_grad', [(True, True), (False, True), (True, False)])
def test_direct_convolution_agrees_with_the_operator_class(mobula, bias, image_grad):
    mobula.op.load('Convolution')
    torch.manual_seed(8)
    x = torch.randn(2, 5, 9, 7, device='cuda').contiguous(memory_format=torch.channels_last)
    w = torch.randn(6, 5, 3, 2, device='cuda', requires_grad=True)
    b = torch.randn(6, device='cuda', requires_grad=True)
    x.requires_grad_(image_grad)
    inputs = [x, w] + ([b] if bias else [])
    wanted = [t for t in inputs if t.requires_grad]
    handle, results = mobula.op.Conv2D, []
    kw = dict(channels=6, kernel_size=(3, 2), strides=(2, 1), padding=(1, 0), dilation=(1, 2))
    handle(*inputs, **kw)
    direct = handle.direct
    assert direct is not None
    for call in (direct, None):
        handle.direct = call
        y = handle(*inputs, **kw)
        results.append((y,) + torch.autograd.grad(y, wanted, torch.ones_like(y).expand_as(y)))
    handle.direct = direct
    for a, b in zip(*results):
        assert a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.parametrize('shape', [(1, 3, 8, 9), (2, 64, 90, 91), (3, 256, 100, 120)])   # one copy; a few pieces; rounds of the ring
def test_host_arrays_of_several_sizes_and_from_several_threads(mobula, shape):
    """Arrays in host memory go through pinned slots in pieces: every element arrives, also when threads
    use the ring at once and after its memory was given back."""
    import threading
    rng = np.random.default_rng(3)
    N, C, H, W = shape
    rois = np.array([[n % N, 3 * n % 40, 5, 3 * n % 40 + 30.5, 60] for n in range(100)], dtype=np.float32)
    kw = dict(pooled_size=(7, 7), spatial_scale=0.5, sampling_ratio=2)
    x = rng.random(shape, dtype=np.float32)
    dy = rng.standard_normal((100, C, 7, 7), dtype=np.float32)
    xt = torch.from_numpy(x).cuda().requires_grad_(True)
    yt = mobula.op.ROIAlign(xt, torch.from_numpy(rois).cuda(), **kw)
    yt.backward(torch.from_numpy(dy).cuda())
    wrong = []

    def work():
        op = mobula.op.ROIAlign[np.ndarray](**kw)
        for _ in range(2):
            y = op(x, rois)
            dx, _ = op.backward(dy)
            if not (np.array_equal(y, yt.detach().cpu().numpy()) and np.array_equal(dx, xt.grad.cpu().numpy())):
                wrong.append(1)
            native.release_workspace()
    threads = [threading.Thread(target=work) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize('wanted', ['x', 'weight', 'bias'])
def test_convolution_gradients_copy_only_what_they_read(mobula, wanted):
    """x and weight in another order than dense are copied for the gradients that read them: x for the weight's, the weight for x's,
    neither for the bias's."""
    mobula.op.load('Convolution')
    x = torch.randn(4, 64, 64, 64, device='cuda').to(memory_format=torch.channels_last)         # 4 MB
    weight = torch.randn(512, 64, 9, 9, device='cuda').to(memory_format=torch.channels_last)    # 10 MB
    inputs = dict(x=x, weight=weight, bias=torch.randn(512, device='cuda'))
    inputs[wanted].requires_grad_(True)
    y = mobula.op.Conv2D(*inputs.values(), channels=512, kernel_size=(9, 9), strides=(4, 4), padding=(4, 4))
    dy = torch.randn_like(y)
    y.backward(dy)   # (the workspace is there now)
    y = mobula.op.Conv2D(*inputs.values(), channels=512, kernel_size=(9, 9), strides=(4, 4), padding=(4, 4))
    torch.cuda.synchronize()
    inputs[wanted].grad = None
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    y.backward(dy)
    size = {k: 4 * t.numel() for k, t in inputs.items()}
    # the gradient, once dense and once in its input's order, and the other operand
    least = {'x': 2 * size['x'] + size['weight'], 'weight': 2 * size['weight'] + size['x'], 'bias': size['bias']}[wanted]
    assert torch.cuda.max_memory_allocated() - before <= least + (1 << 20)
