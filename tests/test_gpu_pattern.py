"""The per-region pattern search (k_pattern_sums, k_pattern_set, k_pattern_regions) bit for bit
against the reference's sequential float sums (src/helper.cpp:57-130) taken on the engine's own
spectra, at every block shape (terms per block below, at and past the kernels' chunks) and at
regions from one block to the whole grid.  Without degrid the terms are |X|^2 times the pattern
window in float, so numpy's float32 gives the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bw,bh", [(8, 8), (16, 16), (24, 24), (32, 32), (48, 48), (64, 64), (32, 16), (16, 32)])
@pytest.mark.parametrize("rx,ry", [(1, 1), (3, 2), (1000, 1000)])
def test_region_psd_bits(bw, bh, rx, ry):
    import torch

    from neo_fft3d_amd import Engine, default_params, make_format
    from neo_fft3d_amd.learned import engine_spectra, region_labels
    w, h = 331, 283
    rng = np.random.default_rng(bw * 100 + bh)
    yy, xx = np.mgrid[0:h, 0:w]
    plane = rng.normal(0.5, 0.02, (h, w)) * (1 + 0.5 * np.sin(xx / 17.0) * np.cos(yy / 23.0))
    src = torch.from_numpy(plane.astype(np.float32)).cuda()
    eng = Engine(default_params(2.0, bw=bw, bh=bh, degrid=0.0), make_format("gray", 32, True), w, h, 1, 0)
    g = eng.geometry()
    nox, noy, ow = g["nox"], g["noy"], g["outwidth"]
    spec = torch.empty((noy, nox, bh * ow, 2), dtype=torch.float32, device="cuda")
    out = torch.empty((noy, nox, bh * ow), dtype=torch.float32, device="cuda")
    engine_spectra(eng, src.data_ptr(), w * 4, spec.data_ptr())
    region_labels(eng, src.data_ptr(), w * 4, rx, ry, out.data_ptr())
    c, got = spec.cpu().numpy(), out.cpu().numpy()
    f = np.float32
    fh = np.minimum(np.arange(bh), bh - np.arange(bh)).astype(f) * f(2) / f(bh)
    fw = np.arange(ow).astype(f) * f(2) / f(bw)
    f2 = (fh * fh)[:, None] + (fw * fw)[None, :]
    pwin = (f2 / (f2 + f(0.1) * f(0.1))).astype(f).reshape(-1)
    term = (c[..., 0] * c[..., 0] + c[..., 1] * c[..., 1]) * pwin
    s = np.zeros((noy, nox), f)
    for k in range(bh * ow):
        s = s + term[..., k]

    def first_min(y0, y1, x0, x1):
        best, at = f(1e15), None
        for y in range(max(y0, 2), min(y1, noy - 2)):
            for x in range(max(x0, 2), min(x1, nox - 2)):
                if s[y, x] < best:
                    best, at = s[y, x], (y, x)
        return at

    whole = first_min(0, noy, 0, nox) or (0, 0)
    for y0 in range(0, noy, ry):
        for x0 in range(0, nox, rx):
            at = first_min(y0, y0 + ry, x0, x0 + rx) or whole
            region = got[y0:y0 + ry, x0:x0 + rx]
            assert np.array_equal(region, np.broadcast_to(term[at], region.shape)), (x0, y0, at)
