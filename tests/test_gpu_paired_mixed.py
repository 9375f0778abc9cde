"""Batches of Wiener-3D ranges that do not all run in pairs: an engine whose range is too short for a
second run beside one that has it, engines of another block shape or transform form (groups on
streams of their own) -- the bits of each engine's range in a call of its own, in graphs too where one
group is captured."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (width, height, block, overlap, bt, dft, first frame, frames)
BATCHES = [
    [(333, 207, 32, 10, 3, 0, 0, 40), (166, 103, 32, 10, 3, 0, 0, 7)],
    [(166, 103, 32, 10, 3, 0, 3, 5), (333, 207, 32, 10, 3, 0, 0, 22), (200, 120, 32, 10, 3, 0, 1, 9)],
    [(333, 207, 48, 16, 3, 0, 0, 40), (333, 207, 16, 4, 3, 0, 0, 12), (166, 103, 48, 16, 3, 0, 2, 6)],
    [(333, 207, 32, 10, 5, 0, 0, 19), (333, 207, 32, 10, 2, 0, 0, 31), (333, 207, 32, 10, 3, 1, 5, 33)],
]


NO_GRAPH = pytest.mark.skip(reason="a captured batch of two block shapes with pairs in its branches ended in a "
                            "segmentation fault in the launch of its graph; the cause is not known, such batches no "
                            "longer pair under capture (tests/test_host_calls.py: captured_pairs)")


@pytest.mark.parametrize("batch,graph", [(0, False), (0, True), (1, False), (1, True), (2, False),
                                         pytest.param(2, True, marks=NO_GRAPH), (3, False),
                                         pytest.param(3, True, marks=NO_GRAPH)])
def test_mixed(batch, graph):
    import torch

    from neo_fft3d_amd import Engine, Graph, default_params, make_format, run_device_batch
    F = 44
    rng = np.random.default_rng(batch)
    fmt, stream = make_format("gray", 8), torch.cuda.Stream()
    src = [torch.from_numpy(rng.integers(0, 256, (F, c[1], c[0]), dtype=np.uint8)).cuda() for c in BATCHES[batch]]
    want, dst = ([torch.zeros_like(s) for s in src] for _ in range(2))

    def engines():
        es = [Engine(default_params(3.0, bt=bt, bw=b, bh=b, ow=ow, oh=ow, sharpen=0.3), fmt, w, h, F, 0)
              for w, h, b, ow, bt, dft, _, _ in BATCHES[batch]]
        for e, c in zip(es, BATCHES[batch]):
            if c[5]:
                e.set_dft(1)
        return es

    def items(es, out):
        return [(e, c[6], c[7], [f.data_ptr() for f in s], s.stride(1), [f.data_ptr() for f in d], d.stride(1))
                for e, c, s, d in zip(es, BATCHES[batch], src, out)]
    torch.cuda.synchronize()
    es = engines()
    for it in items(es, want):
        run_device_batch([it], stream.cuda_stream)
    es = engines()
    if graph:
        g = Graph(items(es, dst), stream.cuda_stream)
        for _ in range(3):
            with torch.cuda.stream(stream):
                for d in dst:
                    d.zero_()
            g.launch(stream.cuda_stream)
            stream.synchronize()
            for w, d in zip(want, dst):
                assert torch.equal(w, d)
        g.close()
    else:
        run_device_batch(items(es, dst), stream.cuda_stream)
        stream.synchronize()
    for w, d in zip(want, dst):
        assert torch.equal(w, d)
