"""The plan of a strided data gradient's columns (csrc/conv_geometry.h), on the CPU."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, '..', 'mobulaop_amd', 'csrc')


@pytest.fixture(scope='module')
def plan(tmp_path_factory):
    path = str(tmp_path_factory.mktemp('conv_phases') / 'phases.so')
    subprocess.run(['g++', '-O1', '-std=c++17', '-shared', '-fPIC', '-Wall', '-I' + CSRC, '-o', path,
                    os.path.join(HERE, 'conv_phases.cpp')], check=True)
    lib = ctypes.CDLL(path)

    def call(N, H, W, D, k, pad, stride, dil, parts, channels=8):
        OH, OW = ((s + 2 * p - ((f - 1) * d + 1)) // t + 1 for s, p, f, d, t in zip((H, W), pad, k, dil, stride))
        geometry = (ctypes.c_int * 15)(N, channels, H, W, D, *k, OH, OW, *pad, *stride, *dil)
        out = (ctypes.c_int * 200)()
        step = 32 if parts == 1 else 16
        image_bytes = 2 * OH * OW * ((D + step - 1) // step * step)
        lib.phases(geometry, ctypes.c_longlong(image_bytes), parts, out)
        return out[0], tuple(out[1:5]), out[5], out[6], [tuple(out[7 + 11 * f:18 + 11 * f]) for f in range(out[0])], image_bytes
    return call


@pytest.mark.parametrize('parts', [1, 2, 3])
@pytest.mark.parametrize('hw', [(14, 14), (9, 30), (5, 3)])
@pytest.mark.parametrize('k,pad,dil,stride', [((3, 3), (1, 1), (1, 1), (2, 2)), ((3, 4), (2, 1), (2, 3), (2, 4)), ((5, 2), (2, 0), (1, 2), (3, 1))])
def test_without_phases_every_tap_is_walked(plan, hw, k, pad, dil, stride, parts):
    """Numbers of images on both sides of the one up to which offsets of the phases' tiles stay below 2^31: beyond it the
    kernel walks all taps of every pixel, one after the other."""
    if any(s + 2 * p < (f - 1) * d + 1 for s, p, f, d in zip(hw, pad, k, dil)):
        pytest.skip('the window does not fit')
    D = 512
    _, _, _, least, _, image_bytes = plan(1, *hw, D, k, pad, stride, dil, parts)
    bound = ((1 << 31) - 1) // image_bytes       # images that fit
    most = (bound - 255 // least - 2) // parts if parts > 1 else 1
    seen = set()
    for N in range(max(most - 3, 1), most + 4):
        if parts == 1:   # (no bound on the images, but on an image's size: as many filters as pass it)
            D = (1 << 31) // (image_bytes // 512 * (255 // least + 2)) // 32 * 32 + 32 * (N - most)
        phases, by, columns, got_least, _, bytes_ = plan(N, *hw, D, k, pad, stride, dil, parts)
        seen.add(phases)
        fits = (255 // least + 2 + (parts * N if parts > 1 else 0)) * bytes_ < 1 << 31
        assert (phases > 0) == fits, (N, D)
        if phases == 0:
            assert by == (1, 1) + dil and columns == N * hw[0] * hw[1] and got_least == hw[0] * hw[1]
    assert len(seen) == 2


@pytest.mark.parametrize('hw,k,pad,dil,stride', [
    ((14, 13), (3, 3), (1, 1), (1, 1), (2, 2)), ((17, 31), (5, 4), (2, 0), (1, 1), (2, 1)), ((21, 20), (3, 3), (2, 1), (2, 1), (2, 4)),
    ((19, 23), (3, 4), (1, 2), (2, 3), (3, 2)), ((3, 2), (2, 2), (1, 0), (1, 1), (4, 2)), ((40, 37), (7, 7), (3, 3), (1, 1), (4, 4)),
    ((30, 30), (6, 5), (2, 2), (1, 1), (5, 4)), ((12, 12), (1, 1), (0, 0), (1, 1), (2, 2)), ((15, 12), (3, 3), (2, 2), (4, 6), (4, 3))])
def test_phases_meet_their_taps(plan, hw, k, pad, dil, stride):
    """Every pixel of every image has one column, phases are whole tiles, and the taps and the pixels of dy that a phase walks
    are those that the definition gives."""
    N = 3
    phases, by, columns, _, all_phases, _ = plan(N, *hw, 20, k, pad, stride, dil, 2)
    if phases == 0:
        assert by == (1, 1) + dil
        return
    pixels, at, before = set(), 0, 1 << 30
    for first, rows, cols, y, x, kh, kw, nkh, nkw, oy, ox in all_phases:
        assert first == at and first % 256 == 0 and nkh * nkw <= before
        at, before = (first + N * rows * cols + 255) // 256 * 256, nkh * nkw
        taps = {(kh + t * by[0], kw + u * by[1], oy - t * by[2], ox - u * by[3]) for t in range(nkh) for u in range(nkw)}
        for i in range(rows):
            for j in range(cols):
                h, w = y + i * stride[0], x + j * stride[1]
                assert h < hw[0] and w < hw[1] and (h, w) not in pixels
                pixels.add((h, w))
                want = {(a, b, (h + pad[0] - a * dil[0]) // stride[0], (w + pad[1] - b * dil[1]) // stride[1])
                        for a in range(k[0]) for b in range(k[1])
                        if (h + pad[0] - a * dil[0]) % stride[0] == 0 and (w + pad[1] - b * dil[1]) % stride[1] == 0}
                assert {(a, b, i + r, j + c) for a, b, r, c in taps} == want
    assert len(pixels) == hw[0] * hw[1] and columns == at
