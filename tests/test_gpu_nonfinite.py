"""Samples of a float plane that are no number, infinite or near the largest float reach only the
pixels of the blocks that hold them, in the frames whose windows do: every other pixel keeps the
bits of the clip without them (window, seams and overlap-add of the frame loop)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf"), 3e38])
@pytest.mark.parametrize("bt", [-1, 0, 1, 2, 3, 5])
@pytest.mark.parametrize("b,ow", [(48, 16), (32, 16), (16, 4), (8, 2), (64, 0)])
def test_stays_in_its_blocks(b, ow, bt, value):
    import torch

    from neo_fft3d_amd import Engine, default_params, make_format, run_device_batch
    w, h, F, at = 531, 307, 13, 6
    g = torch.Generator(device="cuda")
    g.manual_seed(b + bt)
    clean = torch.rand((F, h, w), generator=g, device="cuda")
    dirty = clean.clone()
    points = [(b + 70, b + 90), (h - b - 75, w - b - 90), (b + 71, w - b - 91)]
    for y, x in points:
        dirty[at, y, x] = value
    out = []
    for src in (clean, dirty):
        dst = torch.zeros_like(src)
        e = Engine(default_params(3.0, bt=bt, bw=b, bh=b, ow=ow, oh=ow, sharpen=0.4), make_format("gray", 32, True), w, h, F, 0)
        torch.cuda.synchronize()
        run_device_batch([(e, 0, F, [f.data_ptr() for f in src], w * 4, [f.data_ptr() for f in dst], w * 4)], 0)
        e.sync()
        out.append(dst)
    same = out[0].view(torch.int32) == out[1].view(torch.int32)
    reach = torch.zeros((F, h, w), dtype=torch.bool, device="cuda")
    first, last = (at, at) if bt in (-1, 1) else (at, F - 1) if bt == 0 else (at - (bt - 1) // 2, at + bt // 2)
    for y, x in points:
        reach[first:last + 1, y - b + 1:y + b, x - b + 1:x + b] = True
    assert bool((same | reach).all())
    assert not bool(same.all())
