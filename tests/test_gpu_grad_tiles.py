"""Gradients at ragged widths and batches, and from weights that an update just wrote.

A weight gradient's operands have the batch row as their inner index, outer
widths that leave a tile of 32 or 64 partly empty (multiples of 8), row counts
that are no multiple of 4 or of a step of 64, and a row count that splits K
unevenly; the forward products read the transposed weights, which an Adam step
has to bring up to date.  Bars as for the other gradients: 3e-2 of each
piece's norm against the oracle with BF16 operands, loss within 1e-4.
"""
import numpy as np
import pytest

from test_gpu_learned import make, mo, piece_errors, rand_params, torch, upload_bf16  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,rows", [((8, 8, 8), 1), ((40, 24, 56), 33), ((72, 40, 104), 66), ((200, 64, 200), 1027),
                                       ((104, 8, 2088), 1030)])
def test_ragged_gradients_before_and_after_an_update(torch, dims, rows):  # noqa: F811
    rng = np.random.default_rng(rows)
    params = rand_params(*dims, seed=rows)
    x = rng.standard_normal((rows, dims[0]))
    t = (rng.exponential(1.0, (rows, dims[2])) * np.exp(rng.standard_normal((1, dims[2])))).astype(np.float32)
    m = make(*dims, rows, params)
    xb, tt = upload_bf16(torch, x), torch.from_numpy(t).cuda()
    for step in range(2):
        loss = m.grad(xb.data_ptr(), tt.data_ptr(), rows)
        got = m.get_grads().astype(np.float64)
        now = mo.unpack(m.get_params(), *dims)
        want = mo.backward(now, x, t.astype(np.float64), bf16=True)
        want_loss = mo.whittle_loss(mo.forward(now, x, bf16=True)["y"], t.astype(np.float64))
        errs = piece_errors(got, want, dims)
        print(f"{dims} x {rows}, step {step}: {errs}, loss {loss} vs {want_loss}", flush=True)
        assert max(errs.values()) <= 3e-2
        assert abs(loss - want_loss) <= 1e-4 * abs(want_loss) + 1e-6
        m.adam(1e-2)
