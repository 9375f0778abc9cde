"""The frame loop's gather and overlap-add at every kind of row and column range: with sigma 0 every
gain is one, so whatever the overlaps, the tile's width (one to four passes of 64 columns), the
plane's edges and the sample size, the filter returns its input (integers exactly, floats within
the transform's error of 1e-5)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(8, 8), (16, 16), (24, 24), (32, 32), (48, 48), (64, 64), (32, 16), (16, 32)]


@pytest.mark.parametrize("bw,bh", SHAPES)
@pytest.mark.parametrize("frac", [0.0, 0.06, 0.21, 0.33, 0.5])
def test_sigma_zero_returns_the_input(bw, bh, frac):
    import torch

    from neo_fft3d_amd import Engine, default_params, make_format
    rng = np.random.default_rng(bw * bh)
    ow, oh = int(round(bw * frac)), int(round(bh * (0.5 - frac)))
    for w, h, bits, bt, il in ((300, 202, 8, 3, 0), (523, 190, 16, 1, 1), (261, 203, 32, 2, 0)):
        flt = bits == 32
        top = 1.0 if flt else (1 << bits) - 1
        img = rng.uniform(0, top, (4, h, w))
        src = torch.from_numpy(img.astype(np.float32 if flt else np.uint8 if bits == 8 else np.uint16).view(
            np.float32 if flt else np.uint8 if bits == 8 else np.int16)).cuda()
        dst = torch.zeros_like(src)
        eng = Engine(default_params(0.0, bt=bt, bw=bw, bh=bh, ow=ow, oh=oh, interlaced=il), make_format("gray", bits, flt),
                     w, h, 4, 0)
        stride = src.stride(1) * src.element_size()
        torch.cuda.synchronize()
        eng.run_device(0, 4, [f.data_ptr() for f in src], stride, [f.data_ptr() for f in dst], stride)
        eng.sync()
        if flt:
            assert float((dst - src).abs().max()) < 1e-5, (w, h, bits)
        else:
            assert torch.equal(dst, src), (w, h, bits)
