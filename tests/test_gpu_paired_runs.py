"""Wiener-3D ranges of few tiles run two runs of frames side by side, each in a spectra ring of its
own: the bits of one-frame calls (which have no second run), whatever the number of pairs, the split
of the clip into calls, the number of planes, and in graphs, bound to the ring or not.  (The frames at
the clip's ends come in one call with a whole window: a call of such frames alone is the per-frame
kernel's, whose transforms round differently.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def setup(sizes, F, bt, b, ow, dft, seed):
    import torch

    from neo_fft3d_amd import Engine, default_params, make_format
    rng = np.random.default_rng(seed)
    prm, fmt = default_params(3.0, bt=bt, bw=b, bh=b, ow=ow, oh=ow, sharpen=0.4), make_format("gray", 8)
    src = [torch.from_numpy((rng.normal(120, 6, (F, h, w)) + rng.normal(0, 40, (1, h, w))).clip(0, 255)
                            .astype(np.uint8)).cuda() for w, h in sizes]
    torch.cuda.synchronize()

    def engines():
        es = [Engine(prm, fmt, w, h, F, 0) for w, h in sizes]
        for e in es:
            if dft:
                e.set_dft(1)
        return es

    def items(es, dst, first, count):
        return [(e, first, count, [f.data_ptr() for f in s], s.stride(1), [f.data_ptr() for f in d], d.stride(1))
                for e, s, d in zip(es, src, dst)]
    return src, engines, items


def singles(F, bt):
    lo, hi = bt // 2 + 1, (bt - 1) // 2 + 1
    return [lo] + [1] * (F - lo - hi) + [hi]


def run(src, engines, items, steps):
    import torch

    from neo_fft3d_amd import run_device_batch
    es, dst, n = engines(), [torch.zeros_like(s) for s in src], 0
    torch.cuda.synchronize()
    for k in steps:
        run_device_batch(items(es, dst, n, k), 0)
        n += k
    for e in es:
        e.sync()
    torch.cuda.synchronize()
    return dst


@pytest.mark.parametrize("bt", [2, 3, 4, 5])
@pytest.mark.parametrize("b,ow,dft", [(32, 10, 0), (48, 16, 0), (64, 16, 0), (16, 4, 0), (48, 16, 1)])
def test_splits_and_pairs(bt, b, ow, dft):
    import torch
    F = 72
    for sizes in ([(333, 207), (166, 103), (166, 103)], [(333, 207)]):
        s = setup(sizes, F, bt, b, ow, dft, seed=bt + b)
        want = run(*s, singles(F, bt))
        # one pair; two and three pairs; calls that go on from the ring, pairs and single runs in turn
        for steps in ([20], [42], [F], [9, 1, 12, 7, 33, 10], [5, 16, 40, 11]):
            print(bt, b, dft, len(sizes), steps, flush=True)
            got = run(*s, steps)
            for w, g in zip(want, got):
                n = sum(steps)
                assert torch.equal(w[:n], g[:n])


@pytest.mark.parametrize("ring", [False, True])
@pytest.mark.parametrize("count", [14, 40])
def test_graphs(ring, count):
    import torch

    from neo_fft3d_amd import Graph, run_device_batch
    F = 64
    s = setup([(333, 207), (166, 103), (166, 103)], F, 3, 32, 10, 0, seed=count)
    want = run(*s, singles(F, 3))
    src, engines, items = s
    es, dst = engines(), [torch.zeros_like(x) for x in src]
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    run_device_batch(items(es, dst, 0, 10), stream.cuda_stream)
    stream.synchronize()
    g = Graph(items(es, dst, 10, count), stream.cuda_stream, ring=ring)
    for replay in range(1 if ring else 3):
        with torch.cuda.stream(stream):
            for d in dst:
                d[10:].zero_()
            float(torch.randn(1 << 20, device="cuda").sum())
        g.launch(stream.cuda_stream)
        stream.synchronize()
        for w, d in zip(want, dst):
            assert torch.equal(w[10:10 + count], d[10:10 + count]), replay
    run_device_batch(items(es, dst, 10 + count, F - 10 - count), stream.cuda_stream)
    stream.synchronize()
    for w, d in zip(want, dst):
        assert torch.equal(w, d)
    g.close()
