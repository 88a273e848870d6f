"""Grouped MoE calls as wide as one set of launches goes (the grouping kernel's
LDS at its largest), bit for bit what narrower calls give each token."""
import numpy as np
import pytest
import torch

from conftest import assert_bitexact
from inferq_amd import moe as MOE
from inferq_amd import synth as S

pytestmark = pytest.mark.gpu


# experts x 32-token words at their limit (8192): 256 x 32 and 512 x 16; and a slice of 4096 tokens, one route each
@pytest.mark.parametrize("experts,top_k,tokens", [(256, 4, 1024), (512, 8, 512), (24, 1, 4096)])
def test_widest_slice_equals_narrow_calls(gpu, experts, top_k, tokens):
    hidden = inter = 256
    rng = np.random.default_rng(experts)
    layer = S.random_moe_layer(hidden, inter, experts, S.Q4_K, S.Q6_K, rng)
    t = {k: torch.from_numpy(v).to(gpu) for k, v in layer.items() if isinstance(v, np.ndarray)}
    moe = MOE.QuantizedMoeLayer(hidden, inter, experts, top_k, S.Q4_K, S.Q6_K, t["gate"], t["up"], t["down"],
                                t["shared_gate"], t["shared_up"], t["shared_down"], t["selector"],
                                router=torch.from_numpy(S.normal((experts, hidden), rng)).to(gpu))
    assert moe.slice_tokens() == tokens
    x, res = (torch.from_numpy(S.normal((tokens, hidden), rng)).to(gpu) for _ in range(2))

    def run(step):
        out = torch.empty_like(x)
        experts_out = torch.empty(tokens, top_k, dtype=torch.int32, device=gpu)
        weights = torch.empty(tokens, top_k, device=gpu)
        for i in range(0, tokens, step):
            s = slice(i, i + step)
            moe.forward_x_into(x[s], out[s], res[s], experts_out[s], weights[s])
        return out.cpu().numpy(), experts_out.cpu().numpy(), weights.cpu().numpy()

    wide, narrow = run(tokens), run(8)
    assert np.array_equal(wide[1], narrow[1])
    assert_bitexact(wide[2], narrow[2], "weights")
    assert_bitexact(wide[0], narrow[0], "outputs")
