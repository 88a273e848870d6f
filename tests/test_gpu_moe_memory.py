"""Device memory of a MoE handle: f16 copies of the activations only where the
grouped products read them (Q4_K and Q5_K experts)."""
import gc

import pytest
import torch

from inferq_amd import moe as MOE
from inferq_amd import synth as S

pytestmark = pytest.mark.gpu


def test_q6k_and_q80_handles_hold_no_f16_activations(gpu):
    hidden, inter, experts, top_k, tokens = 4096, 1024, 4, 4, 1024

    def held(dtype):
        g, d = S.matrix_bytes(dtype, experts * inter, hidden), S.matrix_bytes(dtype, experts * hidden, inter)
        buf = torch.zeros(max(g, d), dtype=torch.uint8, device=gpu)
        moe = MOE.QuantizedMoeLayer(hidden, inter, experts, top_k, dtype, dtype, buf[:g], buf[:g], buf[:d])
        gc.collect()
        torch.cuda.synchronize()
        before = torch.cuda.mem_get_info()[0]
        moe.reserve(tokens)
        return before - torch.cuda.mem_get_info()[0]

    # two bytes per value of x and of the SwiGLU rows of routed and shared experts; allocations are rounded
    copies = 2 * tokens * hidden + 2 * tokens * (top_k + 1) * inter
    slack = 4 << 20
    q4 = held(S.Q4_K)
    for dtype in (S.Q6_K, S.Q8_0):
        assert held(dtype) <= q4 - copies + slack
