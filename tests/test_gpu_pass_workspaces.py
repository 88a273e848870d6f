"""Wide K-quant products in workspaces of different sizes (one pass, or several
where the workspace holds fewer rows): the same bits, nothing written past the
workspace, and capture in a workspace that holds what the call needs."""
import ctypes

import numpy as np
import pytest
import torch

from conftest import assert_bitexact
from inferq_amd import qgemm as Q
from inferq_amd import synth as S
from inferq_amd._lib import check, lib

pytestmark = pytest.mark.gpu

ROWS, COLS, M = 40, 8192, 1100  # one pass: 19.3 MB


def _case(gpu, dtype):
    rng = np.random.default_rng(dtype)
    mat = Q.QuantizedMatrix.upload(S.random_matrix(dtype, ROWS, COLS, rng), dtype, ROWS, COLS)
    x = torch.from_numpy(S.normal((M, COLS), rng)).to(gpu)
    want = torch.cat([mat.forward(x[i:i + 50].contiguous()) for i in range(0, M, 50)]).cpu().numpy()
    return mat, x, want


@pytest.mark.parametrize("dtype", [S.Q4_K, S.Q5_K, S.Q6_K])
def test_given_workspace_sizes(gpu, dtype):
    mat, x, want = _case(gpu, dtype)
    least = lib().iq_matmul_workspace_size(mat.handle, M)
    one = M * COLS // 256 * 548 + 1024
    assert least < one
    for size in (least, one - 4, one, 3 * one):
        ws = torch.full((size + 256,), 0x5A, dtype=torch.uint8, device=gpu)
        y = torch.empty(M, ROWS, device=gpu)
        check(lib().iq_matmul_ws(mat.handle, x.data_ptr(), M, y.data_ptr(), ws.data_ptr(), size,
                                 ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        assert_bitexact(y.cpu().numpy(), want, f"{size} bytes")
        assert torch.all(ws[size:] == 0x5A)


def test_capture_in_a_workspace_of_the_least_size(gpu):
    """The stream's workspace, sized by calls of another matrix, holds what the call needs but not one pass of it."""
    mat, x, want = _case(gpu, S.Q6_K)
    other = Q.QuantizedMatrix.upload(S.random_matrix(S.Q8_0, 64, COLS, np.random.default_rng(1)), S.Q8_0, 64, COLS)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        Q.release_workspace()
        other.reserve(M)
    x_buf, y = torch.zeros_like(x), torch.empty(M, ROWS, device=gpu)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        mat.forward_into(x_buf, y)
    x_buf.copy_(x)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert_bitexact(y.cpu().numpy(), want, "replay")
        assert_bitexact(mat.forward(x).cpu().numpy(), want, "eager")
