"""Workspaces sized for wide calls serve narrower ones, whose kernels may need
more (other plans): products captured after a wider reserve, and MoE calls
after a wider reserve of a handle whose shared expert runs apart."""
import numpy as np
import pytest
import torch

from conftest import assert_bitexact
from inferq_amd import _lib
from inferq_amd import moe as MOE
from inferq_amd import qgemm as Q
from inferq_amd import synth as S

pytestmark = pytest.mark.gpu


# one pass of 1900 rows needs more than the two of 2048; eight splits over K of 200 rows more than the four of 256
@pytest.mark.parametrize("dtype,cols,wide,m,path", [(S.Q6_K, 4096, 2048, 1900, _lib.PATH_AUTO),
                                                    (S.Q4_K, 2048, 256, 200, _lib.PATH_PREFILL_TILES)])
def test_capture_after_a_wider_reserve(gpu, dtype, cols, wide, m, path):
    rows = 512
    rng = np.random.default_rng([dtype, m])
    mat = Q.QuantizedMatrix.upload(S.random_matrix(dtype, rows, cols, rng), dtype, rows, cols)
    xs = [torch.from_numpy(S.normal((m, cols), rng)).to(gpu) for _ in range(2)]
    expected = [mat.forward_via(x, path).cpu().numpy() for x in xs]
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        Q.release_workspace()  # torch hands streams out again
        mat.reserve(wide)
    x_buf, y_buf = torch.zeros(m, cols, device=gpu), torch.empty(m, rows, device=gpu)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        mat.forward_into(x_buf, y_buf, path)
    for rep in range(2):
        for i, x in enumerate(xs):
            x_buf.copy_(x)
            graph.replay()
            torch.cuda.synchronize()
            assert_bitexact(y_buf.cpu().numpy(), expected[i], f"replay {rep}.{i}")
            assert_bitexact(mat.forward_via(xs[1 - i], path).cpu().numpy(), expected[1 - i], "eager between replays")


@pytest.mark.parametrize("hidden,inter,routed,shared,wide,m", [(4096, 256, S.Q4_K, S.Q6_K, 2048, 1900),
                                                               (2048, 512, S.Q6_K, S.Q4_K, 256, 200)])
def test_moe_call_after_a_wider_reserve(gpu, hidden, inter, routed, shared, wide, m):
    rng = np.random.default_rng([hidden, m])
    layer = S.random_moe_layer(hidden, inter, 4, routed, routed, rng)
    for name, r, c in (("shared_gate", inter, hidden), ("shared_up", inter, hidden), ("shared_down", hidden, inter)):
        layer[name] = S.random_matrix(shared, r, c, rng)
    t = {k: torch.from_numpy(v).to(gpu) for k, v in layer.items() if isinstance(v, np.ndarray)}
    x = torch.from_numpy(S.normal((m, hidden), rng)).to(gpu)
    lg = torch.from_numpy(S.normal((m, 4), rng)).to(gpu)

    def run(reserve):
        moe = MOE.QuantizedMoeLayer(hidden, inter, 4, 2, routed, routed, t["gate"], t["up"], t["down"], t["shared_gate"],
                                    t["shared_up"], t["shared_down"], t["selector"], shared_gate_dtype=shared,
                                    shared_down_dtype=shared)
        moe.reserve(reserve)
        out = torch.empty_like(x)
        moe.forward_into(x, lg, out)
        return out.cpu().numpy()

    assert_bitexact(run(wide), run(m), f"{m} tokens after a reserve of {wide}")
