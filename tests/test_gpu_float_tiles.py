"""F32 and BF16 products of many pairs (the register tiles of
iq_dense_f32.hip), bitwise to the stated lane order at the edges of their
tiles and stages: each dispatch variant, ragged rows, columns and widths."""
import numpy as np
import pytest
import torch

from conftest import assert_bitexact, bits
from inferq_amd import qgemm as Q
from test_gpu_float_matrices import _matrix, lane_order_product

pytestmark = pytest.mark.gpu


# pairs, 4 x 4 tiles of long and of short stages, 8 x 4 tiles
@pytest.mark.parametrize("rows,cols,m", [(64, 512, 128), (64, 511, 129), (65, 513, 127), (33, 1, 300), (256, 2048, 40),
                                         (9, 1000, 1100), (61, 255, 700), (72, 64, 690), (203, 300, 650), (241, 257, 605)])
@pytest.mark.parametrize("dtype", [Q.IQ_F32, Q.IQ_BF16])
def test_tiles_follow_the_lane_order(gpu, dtype, rows, cols, m):
    mat, wf = _matrix(gpu, dtype, rows, cols, rows + cols + m)
    x = np.random.default_rng(m).standard_normal((m, cols), dtype=np.float32)
    got = mat.forward(torch.from_numpy(x).to(gpu)).cpu().numpy()
    step = 100
    want = np.concatenate([lane_order_product(x[i:i + step], wf) for i in range(0, m, step)])
    assert_bitexact(got, want, f"[{rows} x {cols}] at {m} rows")


def test_tiles_keep_nonfinite_values(gpu):
    rows, cols, m = 64, 333, 200
    mat, wf = _matrix(gpu, Q.IQ_F32, rows, cols, 4)
    x = np.random.default_rng(4).standard_normal((m, cols), dtype=np.float32)
    x[3, 332], x[5, 0], x[7, 100], x[9] = np.inf, -np.inf, np.nan, 0.0
    got = mat.forward(torch.from_numpy(x).to(gpu)).cpu().numpy()
    with np.errstate(invalid="ignore"):
        want = lane_order_product(x, wf)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.array_equal(bits(got)[ok], bits(want)[ok])
