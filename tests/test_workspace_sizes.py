"""Workspace sizes on the CPU: what serves calls of m input rows serves every
narrower call too, so the size never falls as m grows (kernel plans change
with m: splits over K, the passes of a wide call)."""
import ctypes

import pytest

import inferq_amd
from inferq_amd import _lib
from inferq_amd import synth as S


@pytest.mark.parametrize("cols", [2048, 4096, 5120, 8192])
@pytest.mark.parametrize("rows", [64, 512, 2048, 8192])
@pytest.mark.parametrize("dtype", [S.Q4_K, S.Q5_K, S.Q6_K, S.Q8_0])
def test_size_does_not_fall_with_rows(dtype, rows, cols):
    L = inferq_amd.lib()
    h = ctypes.c_void_p()
    # a view is never dereferenced by a size query
    assert L.iq_weights_view(1 << 20, S.matrix_bytes(dtype, rows, cols), dtype, rows, cols, ctypes.byref(h)) == _lib.IQ_OK
    sizes = [L.iq_matmul_workspace_size(h, m) for m in range(1, 9001)]
    L.iq_weights_free(h)
    falls = [(m + 1, a, b) for m, (a, b) in enumerate(zip(sizes, sizes[1:]), 1) if b < a]
    assert not falls, f"{len(falls)} falls, the first at {falls[0]}"
