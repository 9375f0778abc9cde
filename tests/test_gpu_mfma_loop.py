"""The matrix-core form in the frame loop gives the bits of the per-frame kernel: every block size,
temporal mode and sample size, at one to a full tile's blocks past a multiple of the tile, with
edge bands (first and last block row and column), crops and interlaced fields."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,o", [(32, 16), (32, 10), (48, 16), (48, 24), (64, 16), (64, 32)])
@pytest.mark.parametrize("kw", [dict(bt=3, sharpen=0.3), dict(bt=0), dict(bt=1, sharpen=0.5), dict(bt=5, dehalo=0.5),
                                dict(bt=2, interlaced=1), dict(bt=4, l=2, t=4, r=6, b=8)])
def test_loop_equals_per_frame(n, o, kw):
    import torch

    import neo_fft3d_amd as nf
    rng = np.random.default_rng(n + o)
    F = 7
    for k, bits in ((2, 8), (3, 16), (5, 10), (8, 8)):  # blocks past the plane's first tiles
        w, h = (n - o) * k + o + 3, (n - o) * 3 + 2 * n
        h += h % 2
        img = rng.normal(120, 25, (F, h, w)).clip(0, 255) * ((1 << bits) - 1) / 255
        src = torch.from_numpy(img.astype(np.uint8 if bits == 8 else np.int16)).cuda()
        prm, fmt = nf.default_params(2.0, bw=n, bh=n, ow=o, oh=o, **kw), nf.make_format("gray", bits)
        try:
            a, b = (nf.Engine(prm, fmt, w, h, F, 0) for _ in range(2))
        except nf.Nf3dError as e:
            assert "too small" in str(e)
            continue
        a.set_dft(1)
        b.set_dft(1)
        stride = src.stride(1) * src.element_size()
        got, want = torch.zeros_like(src), torch.zeros_like(src)
        torch.cuda.synchronize()
        a.run_device(0, F, [f.data_ptr() for f in src], stride, [f.data_ptr() for f in got], stride)
        a.sync()
        refs = (nf.FrameRef * F)(*[nf.FrameRef(i, f.data_ptr(), stride) for i, f in enumerate(src)])
        err = ctypes.create_string_buffer(256)
        for i in range(F):
            assert nf.lib().nf3d_engine_get_frame_device(b.h, i, refs, F, ctypes.c_void_p(want[i].data_ptr()), stride,
                                                         None, err, 256) == 0, err.value
        b.sync()
        assert torch.equal(got.to(torch.int32), want.to(torch.int32)), (k, bits)
