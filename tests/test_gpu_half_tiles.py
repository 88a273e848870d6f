"""K-quant products on the f16 MFMA row tiles (iq_mfma_half.h), bitwise to the
oracle at the edges of their 16 / 32 x 64 tiles, on blocks of extreme bytes,
and across the passes of a call wider than one pass's workspace."""
import numpy as np
import pytest
import torch

from conftest import assert_bitexact
from inferq_amd import qgemm as Q
from inferq_amd import synth as S

pytestmark = pytest.mark.gpu


# few weight rows run on 16-row tiles, many (or wide calls) on 32-row tiles
@pytest.mark.parametrize("rows,cols,m", [(1, 256, 64), (63, 512, 65), (65, 768, 79), (130, 256, 97), (8256, 512, 64),
                                         (8200, 256, 95), (4100, 512, 161)])
@pytest.mark.parametrize("dtype", [S.Q4_K, S.Q5_K, S.Q6_K])
def test_tile_edges_bitwise(gpu, oracle, dtype, rows, cols, m):
    if dtype == S.Q6_K and cols % 512:
        cols *= 2  # an even block count keeps rows dword-aligned
    rng = np.random.default_rng([dtype, rows, cols, m])
    w = S.random_matrix(dtype, rows, cols, rng)
    x = S.normal((m, cols), rng)
    x[0] = 0.0
    got = Q.QuantizedMatrix.upload(w, dtype, rows, cols).forward(torch.from_numpy(x).to(gpu)).cpu().numpy()
    assert_bitexact(got, oracle.matmul(dtype, w, rows, cols, x), f"[{rows} x {cols}] at {m} rows")


@pytest.mark.parametrize("fill", [0xFF, 0x80, 0x7F, 0x00])
@pytest.mark.parametrize("dtype", [S.Q4_K, S.Q5_K, S.Q6_K])
def test_extreme_integers_bitwise(gpu, oracle, dtype, fill):
    """Every payload byte at an extreme (scales 63, -1, -128, 127; quants 0 or largest) against rows of +-128."""
    rows, cols, m = 8256, 512, 70
    w = S.random_matrix(dtype, rows, cols, np.random.default_rng(fill)).reshape(-1, S.BLOCK_BYTES[dtype])
    w[:, (slice(0, 208) if dtype == S.Q6_K else slice(4, None))] = fill
    x = np.full((m, cols), -3.0, np.float32)
    x[1::3] = 3.0
    x[2::3, ::2] = 3.0
    got = Q.QuantizedMatrix.upload(w.reshape(-1), dtype, rows, cols).forward(torch.from_numpy(x).to(gpu)).cpu().numpy()
    assert_bitexact(got, oracle.matmul(dtype, w.reshape(-1), rows, cols, x), f"bytes {fill:#x}")


@pytest.mark.parametrize("dtype", [S.Q4_K, S.Q5_K, S.Q6_K])
def test_passes_match_narrow_calls(gpu, dtype):
    """A call of more than 16 MiB of f16 activations gives each row what a call of 64 rows gives it, in one pass and
    through the allocation-free entry, whose 16 MiB it must not outgrow."""
    from inferq_amd._lib import check, lib

    rows, cols, m = 40, 8192, 1100  # 16 MiB hold 956 rows: two passes of 550
    rng = np.random.default_rng(dtype)
    mat = Q.QuantizedMatrix.upload(S.random_matrix(dtype, rows, cols, rng), dtype, rows, cols)
    x = torch.from_numpy(S.normal((m, cols), rng)).to(gpu)
    got = mat.forward(x)
    want = torch.cat([mat.forward(x[i:i + 64].contiguous()) for i in range(0, 1024, 64)] +
                     [mat.forward(x[1024:].contiguous())])
    assert torch.equal(got.view(torch.int32), want.view(torch.int32))
    y = torch.empty_like(got)
    torch.cuda.synchronize()
    check(lib().iq_matmul_noalloc(mat.handle, x.data_ptr(), m, y.data_ptr(), None))
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int32), got.view(torch.int32))


@pytest.mark.parametrize("rows,m", [(70, 64), (8256, 70)])
@pytest.mark.parametrize("dtype", [S.Q4_K, S.Q5_K, S.Q6_K])
def test_nonfinite_values_as_the_lane_kernel(gpu, dtype, rows, m):
    """Infinities and NaN in rows and in block scales: NaN where the lane kernel has NaN, its bits elsewhere."""
    from inferq_amd import _lib

    cols = 512
    rng = np.random.default_rng([dtype, m])
    w = S.random_matrix(dtype, rows, cols, rng).reshape(rows, 2, -1)
    d = 208 if dtype == S.Q6_K else 0
    w[3, 1, d:d + 2] = np.array([0x7C00], np.uint16).view(np.uint8)  # inf
    w[7, 0, d:d + 2] = np.array([0x7E00], np.uint16).view(np.uint8)  # NaN
    if dtype != S.Q6_K:
        w[9, 0, 2:4] = np.array([0xFC00], np.uint16).view(np.uint8)  # -inf, of the mins
    x = S.normal((m, cols), rng)
    x[2, 5], x[4, 300], x[6, 200] = np.inf, -np.inf, np.nan
    mat = Q.QuantizedMatrix.upload(w.reshape(-1), dtype, rows, cols)
    xd = torch.from_numpy(x).to(gpu)
    got, ref = (mat.forward_via(xd, p).cpu().numpy() for p in (_lib.PATH_AUTO, _lib.PATH_LANES))
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ref)
    assert np.array_equal(got[ok].view(np.uint32), ref[ok].view(np.uint32))
