"""F32 and BF16 products at few input rows (one wave per weight row,
iq_dense_f32.hip), bitwise to the stated lane order: row lengths at the edges
of its passes of 32, 16 and 8 steps, and tall matrices at one to five rows."""
import numpy as np
import pytest
import torch

from conftest import assert_bitexact, bits
from inferq_amd import qgemm as Q
from test_gpu_float_matrices import _matrix, lane_order_product

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,m", [(5, c, 1 + i % 8) for i, c in enumerate(
    (1, 63, 64, 65, 511, 512, 513, 1000, 1023, 1024, 1025, 1535, 1536, 1537, 1984, 2047, 2048, 2049, 3000, 3583, 4160))] +
    [(8193, 512, 1), (8193, 200, 2), (2049, 1111, 2), (8193, 300, 3), (4097, 2049, 2), (2731, 1600, 3), (2733, 1025, 3), (2049, 700, 4), (1640, 513, 5)])
@pytest.mark.parametrize("dtype", [Q.IQ_F32, Q.IQ_BF16])
def test_few_rows_follow_the_lane_order(gpu, dtype, rows, cols, m):
    mat, wf = _matrix(gpu, dtype, rows, cols, rows + cols + m)
    x = np.random.default_rng(m).standard_normal((m, cols), dtype=np.float32)
    out = torch.full((m + 1, rows), 7.0, device=gpu)
    mat.forward_into(torch.from_numpy(x).to(gpu), out[:m])
    assert torch.all(out[m] == 7.0)
    step = 500
    want = np.concatenate([lane_order_product(x, wf[i:i + step]) for i in range(0, rows, step)], 1)
    assert_bitexact(out[:m].cpu().numpy(), want, f"[{rows} x {cols}] at {m} rows")


@pytest.mark.parametrize("rows,m", [(64, 4), (8193, 2)])
def test_values_past_the_end_stay_out(gpu, rows, m):
    """The last value of a row, which the steps past its end load again, is infinite or NaN in some rows."""
    cols = 333
    mat, wf = _matrix(gpu, Q.IQ_F32, rows, cols, 4)
    x = np.random.default_rng(4).standard_normal((m, cols), dtype=np.float32)
    x[0, 332], x[1, 332] = np.inf, np.nan
    got = mat.forward(torch.from_numpy(x).to(gpu)).cpu().numpy()
    with np.errstate(invalid="ignore"):
        want = lane_order_product(x, wf)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.array_equal(bits(got)[ok], bits(want)[ok])
