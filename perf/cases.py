"""The work whose speed counts: calls of the two operators as a program makes them.

`listed()` names twelve of them, `draw(rng)` gives more of the same ranges.  A case is
a dict of plain values; `prepare` makes the tensors a program has in hand before the
call (feature map, boxes, incoming gradient; images, weights), `run` is one pass
through `mobula.op.ROIAlign` / `mobula.op.Conv2D`, forward and, where the case trains,
backward."""
import math

import numpy as np
import torch

import mobulaop_amd as mobula
from mobulaop_amd import native

mobula.op.load('ROIAlign')
mobula.op.load('Convolution')

_DTYPES = {'float32': torch.float32, 'float16': torch.float16, 'bfloat16': torch.bfloat16}
# option "conv_compute" of the launcher library
_PRODUCTS = {'fp32': 0, 'bf16': 1, 'bf16x3': 2}

# What one pass may cost at most (the largest listed cases stand a little above or at these).
_MOST_BYTES = 3.5e9
_MOST_FLOPS = 3.5e11


def _roialign(name, images, channels, height, width, rois, pooled, sampling, stride, boxes, dtype='float32',
              layout='nchw', arrays='torch', train=True):
    case = dict(op='ROIAlign', arrays=arrays, dtype=dtype, layout=layout, train=train, images=images,
                channels=channels, height=height, width=width, rois=rois, pooled_h=pooled[0], pooled_w=pooled[1],
                sampling=sampling, stride=stride, boxes=boxes)
    return dict(case, name=name) if name else case


def _conv(name, images, channels, height, width, filters, kernel, pad, stride, products, bias, image_grad=True):
    case = dict(op='Conv2D', products=products, images=images, channels=channels, height=height, width=width,
                filters=filters, kernel_h=kernel[0], kernel_w=kernel[1], pad_h=pad[0], pad_w=pad[1], stride=stride,
                bias=bias, image_grad=image_grad)
    return dict(case, name=name) if name else case


def listed():
    return [
        # A handful of boxes on a small map (one image, late in a cascade): what a call costs at least.
        _roialign('few_boxes', 1, 64, 32, 32, 8, (7, 7), 2, 8, 'uniform'),
        # A detection head over a coarse level: BASELINE configuration 1 with tensors on the GPU.
        _roialign('small_map', 2, 256, 64, 64, 512, (7, 7), 2, 8, 'uniform'),
        # The same configuration as it is stated: NumPy arrays in host memory, forward and backward.
        _roialign('host_arrays', 2, 256, 64, 64, 512, (7, 7), 2, 8, 'uniform', arrays='numpy'),
        # The finest level of a feature pyramid, training: configuration 2, the headline.
        _roialign('fine_map', 4, 256, 200, 336, 4000, (7, 7), 2, 4, 'log_uniform'),
        # The same level in mixed-precision training of a channels-last model.
        _roialign('fine_map_bf16_channels_last', 4, 256, 200, 336, 4000, (7, 7), 2, 4, 'log_uniform',
                  dtype='bfloat16', layout='channels_last'),
        # A mask head: larger pooled maps, clustered boxes, some of them degenerate: configuration 3.
        _roialign('mask_head', 8, 256, 128, 128, 8192, (14, 14), 2, 8, 'clustered'),
        # Inference in half precision with the adaptive sampling grid: configuration 4.
        _roialign('inference_fp16', 4, 512, 100, 100, 6000, (7, 7), 0, 16, 'uniform', dtype='float16', train=False),
        # Nothing a multiple of anything: class score maps of an odd-sized image, adaptive grid, training.
        _roialign('ragged', 3, 81, 75, 113, 301, (5, 9), 0, 8, 'log_uniform'),
        # An inner 3x3 layer in full precision, forward and both gradients: configuration 5.
        _conv('conv_fp32', 32, 256, 56, 56, 256, (3, 3), (1, 1), 1, 'fp32', False),
        # The same layer with operands rounded to bf16.
        _conv('conv_bf16', 32, 256, 56, 56, 256, (3, 3), (1, 1), 1, 'bf16', False),
        # A smaller layer of odd sizes with split operands (nearly fp32 results), with a bias.
        _conv('conv_bf16x3_ragged', 5, 96, 45, 67, 130, (3, 3), (1, 1), 1, 'bf16x3', True),
        # The first layer of a network: three channels, a large strided kernel; the image needs no gradient.
        _conv('conv_first_layer', 8, 3, 224, 224, 64, (7, 7), (3, 3), 2, 'fp32', True, image_grad=False),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _channels(rng, low, high):
    """Channel counts are mostly round numbers; one in four is not."""
    c = _log_int(rng, low, high)
    step = rng.choice((1, 8, 32, 32)) if c >= 32 else rng.choice((1, 1, 8))
    return max(step, c // step * step)


def _draw_roialign(rng):
    while True:
        host = rng.random() < 0.15
        dtype = 'float32' if host else rng.choice(('float32', 'float32', 'float16', 'bfloat16'))
        side = rng.choice((7, 7, 7, 14, 14, 28, 0))   # 0: some other, not even square
        pooled = (side, side) if side else (rng.randint(1, 12), rng.randint(1, 12))
        case = _roialign(
            None, rng.randint(1, 8), _channels(rng, 16, 512), _log_int(rng, 16, 256), _log_int(rng, 16, 336),
            _log_int(rng, 4, 600 if host else 8192), pooled, rng.choice((2, 2, 2, 0, 0, 1, 3)),
            rng.choice((4, 8, 16, 32)), rng.choice(('uniform', 'log_uniform', 'clustered')), dtype=dtype,
            layout='nchw' if host else rng.choice(('nchw', 'nchw', 'channels_last')),
            arrays='numpy' if host else 'torch', train=rng.random() < 0.75)
        if work(case)['bytes'] <= (1.5e8 if host else _MOST_BYTES):
            return case


def _draw_conv(rng):
    while True:
        k = rng.choice((1, 3, 3, 3, 5, 7))
        height = _log_int(rng, 7, 224)
        channels = 3 if rng.random() < 0.15 else _channels(rng, 16, 512)
        case = _conv(
            None, rng.randint(1, 32), channels, height, max(7, int(height * rng.uniform(0.7, 1.4))),
            _channels(rng, 16, 512), (k, k), (k // 2, k // 2), rng.choice((1, 1, 1, 2)),
            rng.choice(('fp32', 'fp32', 'bf16', 'bf16', 'bf16x3')), rng.random() < 0.5, image_grad=channels > 3)
        w = work(case)
        if w['bytes'] <= 1.5e9 and w['flops'] <= _MOST_FLOPS:
            return case


def draw(rng):
    return _draw_roialign(rng) if rng.random() < 0.65 else _draw_conv(rng)


def _boxes(case, rng):
    """[R,5] rows (image, x1, y1, x2, y2) in pixels of an image `stride` times the map."""
    R, N = case['rois'], case['images']
    W, H = case['width'] * case['stride'], case['height'] * case['stride']
    image = rng.integers(0, N, R)
    if case['boxes'] == 'uniform':      # two corners anywhere in the image
        p = np.sort(rng.uniform(0, 1, (R, 2, 2)), axis=1)
        x1, y1, x2, y2 = p[:, 0, 0] * W, p[:, 0, 1] * H, p[:, 1, 0] * W, p[:, 1, 1] * H
    else:
        low = 16.0 if case['boxes'] == 'log_uniform' else 32.0
        w = np.exp(rng.uniform(np.log(low), np.log(max(low + 1, min(512.0, W))), R))
        h = np.exp(rng.uniform(np.log(low), np.log(max(low + 1, min(512.0, H))), R))
        if case['boxes'] == 'log_uniform':   # proposals of every size, inside the image
            w, h = np.minimum(w, W), np.minimum(h, H)
            cx, cy = rng.uniform(w / 2, W - w / 2), rng.uniform(h / 2, H - h / 2)
        else:                                # proposals around the objects of an image
            centre = rng.uniform(0, 1, (N, 16, 2)) * (W, H)
            c = centre[image, rng.integers(0, 16, R)] + rng.normal(0, 32.0, (R, 2))
            cx, cy = c[:, 0], c[:, 1]
        x1, y1, x2, y2 = cx - w / 2, cy - h / 2, cx + w / 2, cy + h / 2
        if case['boxes'] == 'clustered':     # one in ten off the image, without extent, or below a pixel
            odd = rng.permutation(R)[:R // 10]
            off, flat, tiny = np.array_split(odd, 3)
            x1[off] += 0.6 * W
            x2[off] += 0.6 * W
            x2[flat] = x1[flat]
            x2[tiny], y2[tiny] = x1[tiny] + 0.5, y1[tiny] + 0.3
    return np.stack([image, x1, y1, x2, y2], axis=1).astype(np.float32)


def _roialign_op_args(case):
    return dict(pooled_size=(case['pooled_h'], case['pooled_w']), spatial_scale=1.0 / case['stride'],
                sampling_ratio=case['sampling'])


def _prepare_roialign(case, seed):
    rng = np.random.default_rng(seed)
    shape = (case['images'], case['channels'], case['height'], case['width'])
    pooled = (case['rois'], case['channels'], case['pooled_h'], case['pooled_w'])
    rois = _boxes(case, rng)
    if case['arrays'] == 'numpy':
        op = mobula.op.ROIAlign[np.ndarray](**_roialign_op_args(case))
        dy = rng.standard_normal(pooled, dtype=np.float32) if case['train'] else None
        return dict(case=case, op=op, x=rng.random(shape, dtype=np.float32), rois=rois, dy=dy)
    g = torch.Generator(device='cuda').manual_seed(seed)
    fmt = torch.channels_last if case['layout'] == 'channels_last' else torch.contiguous_format
    dtype = _DTYPES[case['dtype']]
    # activations: after a rectifier in training, of either sign at inference
    make = torch.rand if case['train'] else torch.randn
    x = make(shape, generator=g, device='cuda').to(dtype).contiguous(memory_format=fmt)
    dy = None
    if case['train']:
        x.requires_grad_(True)
        dy = torch.randn(pooled, generator=g, device='cuda').to(dtype).contiguous(memory_format=fmt)
    return dict(case=case, x=x, rois=torch.from_numpy(rois).cuda(), dy=dy)


def _out_size(case):
    return ((case['height'] + 2 * case['pad_h'] - case['kernel_h']) // case['stride'] + 1,
            (case['width'] + 2 * case['pad_w'] - case['kernel_w']) // case['stride'] + 1)


def _prepare_conv(case, seed):
    native.set_option('conv_compute', _PRODUCTS[case['products']])
    g = torch.Generator(device='cuda').manual_seed(seed)
    N, C, D, K = case['images'], case['channels'], case['filters'], (case['kernel_h'], case['kernel_w'])
    x = torch.randn((N, C, case['height'], case['width']), generator=g, device='cuda')
    x.requires_grad_(case['image_grad'])
    weight = torch.randn((D, C) + K, generator=g, device='cuda') * math.sqrt(2.0 / (C * K[0] * K[1]))
    bias = torch.randn(D, generator=g, device='cuda').requires_grad_(True) if case['bias'] else None
    dy = torch.randn((N, D) + _out_size(case), generator=g, device='cuda')
    return dict(case=case, x=x, weight=weight.requires_grad_(True), bias=bias, dy=dy)


def prepare(case, seed):
    return (_prepare_roialign if case['op'] == 'ROIAlign' else _prepare_conv)(case, seed)


def _run_roialign(s):
    case, x, rois, dy = s['case'], s['x'], s['rois'], s['dy']
    if case['arrays'] == 'numpy':
        y = s['op'](x, rois)
        return [y] + (list(s['op'].backward(dy)) if case['train'] else [])
    if not case['train']:
        with torch.no_grad():
            return [mobula.op.ROIAlign(x, rois, **_roialign_op_args(case))]
    x.grad = None
    y = mobula.op.ROIAlign(x, rois, **_roialign_op_args(case))
    y.backward(dy)
    return [y.detach(), x.grad]


def _run_conv(s):
    case = s['case']
    inputs = [s['x'], s['weight']] + ([s['bias']] if case['bias'] else [])
    for t in inputs:
        t.grad = None
    y = mobula.op.Conv2D(*inputs, channels=case['filters'], kernel_size=(case['kernel_h'], case['kernel_w']),
                         strides=(case['stride'], case['stride']), padding=(case['pad_h'], case['pad_w']))
    y.backward(s['dy'])
    return [y.detach()] + [t.grad for t in inputs if t.requires_grad]


def run(state):
    return _run_roialign(state) if state['case']['op'] == 'ROIAlign' else _run_conv(state)


def work(case):
    if case['op'] == 'ROIAlign':
        e = 4 if case['dtype'] == 'float32' else 2
        bins = case['rois'] * case['channels'] * case['pooled_h'] * case['pooled_w']
        one_pass = e * case['images'] * case['channels'] * case['height'] * case['width'] + 20 * case['rois'] + e * bins
        passes = 2 if case['train'] else 1
        # a bin needs one bilinear sample at least: four corners, a multiply-add each
        return {'bytes': passes * one_pass, 'flops': passes * 8 * bins}
    OH, OW = _out_size(case)
    x = case['images'] * case['channels'] * case['height'] * case['width']
    y = case['images'] * case['filters'] * OH * OW
    weight = case['filters'] * case['channels'] * case['kernel_h'] * case['kernel_w']
    product = 2.0 * y * case['channels'] * case['kernel_h'] * case['kernel_w']
    # read x, weight, dy; write y, dW and, where it is asked for, dx (bf16x3: priced as one product)
    return {'bytes': 4 * (x + weight + y + y + weight + (x if case['image_grad'] else 0) +
                          (2 * case['filters'] if case['bias'] else 0)),
            'flops': product * (3 if case['image_grad'] else 2)}


def tolerance(case):
    if case['op'] == 'ROIAlign':
        # sums in fp32 in every case; 16-bit results are rounded once
        return {'rel': {'float32': 1e-5, 'float16': 1e-3, 'bfloat16': 8e-3}[case['dtype']]}
    # operands are rounded the same way by every implementation, sums are fp32; the
    # split mode leaves 16 significant bits per operand
    return {'rel': 2e-5 if case['products'] == 'bf16x3' else 1e-5}
