"""Engines that shared a batch call and then run by themselves, on streams of their own, and the
batch's first engine destroyed while the others go on: the bits of engines that never met."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bt", [0, 3])
@pytest.mark.parametrize("sizes", [[(333, 207), (166, 103), (166, 103)], [(1280, 720), (64, 48), (320, 240)]])
def test_apart(bt, sizes):
    import torch

    from neo_fft3d_amd import Engine, default_params, make_format, run_device_batch
    F, b, ow = 40, 16, 4
    rng = np.random.default_rng(bt)
    prm, fmt = default_params(3.0, bt=bt, bw=b, bh=b, ow=ow, oh=ow), make_format("gray", 8)
    src = [torch.from_numpy(rng.integers(0, 256, (F, h, w), dtype=np.uint8)).cuda() for w, h in sizes]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(4)]

    def engines():
        return [Engine(prm, fmt, w, h, F, 0) for w, h in sizes]

    def item(e, k, dst, first, count):
        return (e, first, count, [f.data_ptr() for f in src[k]], src[k].stride(1), [f.data_ptr() for f in dst[k]],
                dst[k].stride(1))

    steps = [(0, 12), (12, 9), (21, 1), (22, 18)]  # together, apart, together, apart
    want, dst = ([torch.zeros_like(s) for s in src] for _ in range(2))
    torch.cuda.synchronize()
    for k, e in enumerate(engines()):
        for n, c in steps:
            run_device_batch([item(e, k, want, n, c)], streams[3].cuda_stream)
    es = engines()
    for j, (n, c) in enumerate(steps):
        if j % 2 == 0:
            run_device_batch([item(e, k, dst, n, c) for k, e in enumerate(es)], streams[3].cuda_stream)
            continue
        for k, e in enumerate(es):
            run_device_batch([item(e, k, dst, n, c)], streams[k].cuda_stream)
        if j == 3:
            es[0].sync()
            es[0].close()
    for e in es[1:]:
        e.sync()
    torch.cuda.synchronize()
    for w, d in zip(want, dst):
        assert torch.equal(w, d)
