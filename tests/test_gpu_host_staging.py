"""Host-fed frames through pinned staging (nf3d_engine_get_frame): pageable planes of any stride,
with and without a crop, give the bits of page-locked ones; nothing outside the processed region
is written; strides shorter than a row and null planes are refused."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _get(eng, n, planes, strides, dst, dst_stride):
    import neo_fft3d_amd as nf
    refs = (nf.FrameRef * len(planes))(*[nf.FrameRef(k, p, s) for k, (p, s) in enumerate(zip(planes, strides))])
    err = ctypes.create_string_buffer(256)
    return nf.lib().nf3d_engine_get_frame(eng.h, n, refs, len(planes), dst, dst_stride, err, 256), err.value.decode()


@pytest.mark.parametrize("w,h,bits,pad,crop", [(320, 200, 8, 0, 0), (331, 203, 8, 37, 0), (256, 128, 16, 0, 0),
                                               (517, 311, 16, 10, 4), (2048, 400, 8, 64, 2)])
def test_pageable_equals_pinned(w, h, bits, pad, crop):
    import torch

    import neo_fft3d_amd as nf
    dt = np.uint8 if bits == 8 else np.uint16
    rng = np.random.default_rng(w + h)
    stride = w * dt().itemsize + pad
    src = [rng.integers(0, 256, (h, stride), dtype=np.uint8) for _ in range(4)]
    prm = nf.default_params(2.0, bt=3, bw=16, bh=16, l=crop, t=crop, r=crop, b=crop)
    fmt = nf.make_format("gray", bits)
    a, b = (nf.Engine(prm, fmt, w, h, 4, 0) for _ in range(2))
    pinned = [torch.from_numpy(s).pin_memory() for s in src]
    for n in range(4):
        out = np.full((h, stride), 171, np.uint8)
        want = torch.full((h, stride), 171, dtype=torch.uint8).pin_memory()
        assert _get(a, n, [s.ctypes.data for s in src], [stride] * 4, out.ctypes.data, stride)[0] == 0
        assert _get(b, n, [s.data_ptr() for s in pinned], [stride] * 4, want.data_ptr(), stride)[0] == 0
        assert np.array_equal(out, want.numpy()), n
        edge = np.ones((h, stride), bool)
        bps = dt().itemsize
        edge[crop:h - crop, crop * bps:(w - crop) * bps] = False
        assert (out[edge] == 171).all()


def test_refused():
    import neo_fft3d_amd as nf
    w, h = 128, 96
    eng = nf.Engine(nf.default_params(2.0, bt=1, bw=16, bh=16), nf.make_format("gray", 8), w, h, 1, 0)
    src, dst = np.zeros((h, w), np.uint8), np.zeros((h, w), np.uint8)
    assert _get(eng, 0, [src.ctypes.data], [w - 1], dst.ctypes.data, w)[0] == -1
    assert _get(eng, 0, [src.ctypes.data], [-w], dst.ctypes.data, w)[0] == -1
    assert _get(eng, 0, [src.ctypes.data], [w], dst.ctypes.data, w - 1)[0] == -1
    assert _get(eng, 0, [src.ctypes.data], [w], None, w)[0] == -1
    assert _get(eng, 0, [None], [w], dst.ctypes.data, w)[0] == -1
    assert _get(eng, 0, [src.ctypes.data], [w], dst.ctypes.data, w)[0] == 0
