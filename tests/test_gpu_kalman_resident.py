"""Kalman launches that keep the state in registers over their frames give the bits of one-frame
launches, which keep it in memory: every block shape, sharpen case and launch length from two
frames to sixteen and one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bw,bh", [(8, 8), (16, 16), (24, 24), (32, 32), (48, 48), (64, 64), (32, 16), (16, 32)])
@pytest.mark.parametrize("kw", [{}, {"sharpen": 0.5}, {"dehalo": 0.5, "sigma4": 6.0}])
def test_launch_length_does_not_matter(bw, bh, kw):
    import torch

    from neo_fft3d_amd import Engine, default_params, make_format
    rng = np.random.default_rng(bw + bh)
    w, h, F = 333, 207, 18
    src = torch.from_numpy((rng.normal(120, 6, (F, h, w)) + rng.normal(0, 40, (1, h, w))).clip(0, 255).astype(np.uint8)).cuda()
    stride, outs = src.stride(1), []
    prm, fmt = default_params(3.0, bt=0, bw=bw, bh=bh, **kw), make_format("gray", 8)
    torch.cuda.synchronize()
    for steps in ([1] * F, [F], [1, 2, 3, 4, 5, 3]):
        eng, dst, n = Engine(prm, fmt, w, h, F, 0), torch.zeros_like(src), 0
        for k in steps:
            eng.run_device(n, k, [f.data_ptr() for f in src], stride, [f.data_ptr() for f in dst], stride)
            n += k
        eng.sync()
        outs.append(dst)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
