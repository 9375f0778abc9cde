"""Block transforms on the matrix cores at ragged counts and addresses.

A workgroup transforms four blocks and moves each through LDS in 16-byte
pieces, the last of which only some lanes have: counts that leave a workgroup
partly empty, one block alone, buffers at an 8-byte instead of a 256-byte
address, and guard values on both sides of the output.  The bar is the FP64
DFT within 2e-6 of the largest magnitude, and the same bits at both addresses.
"""
import ctypes

import numpy as np
import pytest

from test_gpu_mfma_dft import env, windowed_blocks  # noqa: F401  (module fixture)

pytestmark = pytest.mark.gpu

PAD, GUARD = 64, -12345.0


def transform(torch, lib, host, count, nb, n, inverse, scale, shift):
    d_in = torch.zeros(host.size + shift, dtype=torch.float32, device="cuda")
    d_in[shift:] = torch.from_numpy(host.reshape(-1)).cuda()
    d_out = torch.full((count + 2 * PAD + shift,), GUARD, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    rc = lib.nf3d_dft2d_mfma(ctypes.c_void_p(d_in.data_ptr() + 4 * shift),
                             ctypes.c_void_p(d_out.data_ptr() + 4 * (PAD + shift)), nb, n, int(inverse),
                             ctypes.c_float(scale), None)
    assert rc == 0
    torch.cuda.synchronize()
    got = d_out.cpu().numpy()
    assert (got[:PAD + shift] == GUARD).all() and (got[PAD + shift + count:] == GUARD).all()
    return got[PAD + shift:PAD + shift + count]


@pytest.mark.parametrize("n", [32, 48, 64])
@pytest.mark.parametrize("nb", [1, 2, 3, 5])
def test_ragged_counts_and_addresses(env, n, nb):  # noqa: F811
    torch, lib = env
    h = n // 2 + 1
    x = windowed_blocks(nb, 1023.0, seed=nb, n=n)
    Z = np.fft.rfft2(x.astype(np.float64))
    Zf = np.stack([Z.real, Z.imag], axis=-1).astype(np.float32)

    fwd = [transform(torch, lib, x, nb * n * h * 2, nb, n, False, 1.0, shift) for shift in (0, 2)]
    assert np.array_equal(fwd[0], fwd[1])
    got = fwd[0].reshape(nb, n, h, 2)
    assert np.abs(got[..., 0] + 1j * got[..., 1] - Z).max() <= 2e-6 * np.abs(Z).max()

    inv = [transform(torch, lib, Zf, nb * n * n, nb, n, True, 1.0 / 32, shift) for shift in (0, 2)]
    assert np.array_equal(inv[0], inv[1])
    want = np.fft.irfft2(Zf[..., 0].astype(np.float64) + 1j * Zf[..., 1].astype(np.float64), s=(n, n)) * float(n * n)
    assert np.abs(inv[0].reshape(nb, n, n) - want).max() <= 2e-6 * np.abs(want).max()
