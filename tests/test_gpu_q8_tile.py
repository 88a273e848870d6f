"""Q8_0 products at many input rows (iq_q8_tile.hip: the reference's eight
chains on f16 MFMA), bitwise to the oracle at the edges of its 32 x 64 tiles
and 4-block stages, and to the lane kernel on rows with no finite scale."""
import numpy as np
import pytest

from conftest import assert_bitexact, bits

pytestmark = pytest.mark.gpu


def _mat(rows, cols, rng):
    from inferq_amd import qgemm as Q, synth as S

    w = S.random_matrix(S.Q8_0, rows, cols, rng)
    return w, Q.QuantizedMatrix.upload(w, S.Q8_0, rows, cols)


# widths of 1, 3 and 5 stages of 128 that no GEMV takes (9..63 rows stay on the tile), and whole model widths
@pytest.mark.parametrize("rows,cols", [(1, 128), (63, 384), (64, 640), (65, 384), (130, 128), (512, 2048), (200, 4096)])
@pytest.mark.parametrize("m", [9, 16, 17, 31, 32, 33, 64, 97])
def test_tile_edges_bitwise(gpu, oracle, rows, cols, m):
    import torch

    from inferq_amd import synth as S

    rng = np.random.default_rng([rows, cols, m])
    w, mat = _mat(rows, cols, rng)
    x = S.normal((m, cols), rng)
    x[0] = 0.0
    x[m - 1] *= np.float32(1e-20)
    got = mat.forward(torch.from_numpy(x).to(gpu)).cpu().numpy()
    assert_bitexact(got, oracle.matmul(S.Q8_0, w, rows, cols, x), f"[{rows} x {cols}] at {m} rows")


# 3..8 rows: either side of the rule's lines (the GEMV takes the other), ragged row counts, one to four steps of 1024
@pytest.mark.parametrize("rows,cols,m", [(8681, 1024, 3), (8680, 1024, 3), (6511, 1024, 4), (3256, 1024, 8),
                                         (2443, 2048, 8), (3907, 2048, 5), (2051, 3072, 8), (1862, 4096, 7),
                                         (1629, 4096, 8), (1628, 4096, 8), (16384, 1024, 3), (16385, 1024, 3),
                                         (16385, 1024, 6), (65537, 1024, 8), (2000, 5120, 8)])
def test_few_rows_bitwise(gpu, oracle, rows, cols, m):
    import torch

    from inferq_amd import synth as S

    rng = np.random.default_rng([rows, cols, m])
    w, mat = _mat(rows, cols, rng)
    x = S.normal((m, cols), rng)
    x[0] = 0.0
    x[m - 1] *= np.float32(1e-20)
    x[1, :32] = np.where(np.arange(32) % 2, np.float32(-3), np.float32(3))
    out = torch.full((m + 1, rows), 7.0, device=gpu)
    mat.forward_into(torch.from_numpy(x).to(gpu), out[:m])
    assert torch.all(out[m] == 7.0)
    assert_bitexact(out[:m].cpu().numpy(), oracle.matmul(S.Q8_0, w, rows, cols, x), f"[{rows} x {cols}] at {m} rows")


# the lines of the rules, the tile on one side and the GEMV on the other
@pytest.mark.parametrize("rows,cols,m", [(16383, 1024, 3), (16384, 1024, 4), (16384, 2048, 4), (16384, 2048, 5),
                                         (24575, 1024, 4), (24576, 1024, 5), (2048, 1024, 32), (2048, 1024, 33),
                                         (4096, 1024, 16), (4096, 1024, 17)])
def test_either_side_of_a_line_bitwise(gpu, oracle, rows, cols, m):
    import torch

    from inferq_amd import synth as S

    rng = np.random.default_rng([rows, cols, m])
    w, mat = _mat(rows, cols, rng)
    x = S.normal((m, cols), rng)
    got = mat.forward(torch.from_numpy(x).to(gpu)).cpu().numpy()
    assert_bitexact(got, oracle.matmul(S.Q8_0, w, rows, cols, x), f"[{rows} x {cols}] at {m} rows")


@pytest.mark.parametrize("fill", [0x80, 0x7F, 0xFF, 0x00])
def test_extreme_values_bitwise(gpu, oracle, fill):
    """Every weight byte -128, 127, -1 or 0 against rows that quantise to +-127."""
    import torch

    from inferq_amd import qgemm as Q, synth as S

    rows, cols, m = 70, 640, 40
    rng = np.random.default_rng(fill)
    w = S.random_matrix(S.Q8_0, rows, cols, rng).reshape(-1, 34)
    w[:, 2:] = fill
    x = np.where(rng.random((m, cols)) < 0.5, np.float32(-3), np.float32(3)).astype(np.float32)
    x[0], x[1] = 3.0, -3.0
    mat = Q.QuantizedMatrix.upload(w.reshape(-1), S.Q8_0, rows, cols)
    got = mat.forward(torch.from_numpy(x).to(gpu)).cpu().numpy()
    assert_bitexact(got, oracle.matmul(S.Q8_0, w.reshape(-1), rows, cols, x), f"bytes {fill:#x}")


@pytest.mark.parametrize("rows,cols,m", [(66, 384, 35), (3260, 1024, 8)])
def test_nonfinite_scales_as_the_lane_kernel(gpu, rows, cols, m):
    """Infinities and NaN in rows and in weight scales: NaN where the lane kernel has NaN, its bits elsewhere."""
    import torch

    from inferq_amd import _lib, qgemm as Q, synth as S

    rng = np.random.default_rng(5)
    w = S.random_matrix(S.Q8_0, rows, cols, rng).reshape(rows, -1, 34)
    w[3, 2, 0:2] = np.array([0x7C00], np.uint16).view(np.uint8)  # inf
    w[7, 0, 0:2] = np.array([0x7E00], np.uint16).view(np.uint8)  # NaN
    x = S.normal((m, cols), rng)
    x[2, 5], x[4, 100], x[6, 200] = np.inf, -np.inf, np.nan
    mat = Q.QuantizedMatrix.upload(w.reshape(-1), S.Q8_0, rows, cols)
    xd = torch.from_numpy(x).to(gpu)
    got, ref = (mat.forward_via(xd, p).cpu().numpy() for p in (_lib.PATH_AUTO, _lib.PATH_LANES))
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ref)
    assert np.array_equal(bits(got)[ok], bits(ref)[ok])


# past 48 tokens the shared expert runs on the many-row tiles, gate and up in one launch, SwiGLU inside down's
# quantisation; hidden 1280: from 64 tokens only, its products apart below
@pytest.mark.parametrize("tokens", [49, 64, 97])
@pytest.mark.parametrize("hidden,inter", [(512, 256), (1280, 512)])
def test_q8_shared_expert_wide_equals_narrow(gpu, tokens, hidden, inter):
    """Each token of a wide call gets, bit for bit, what calls of 8 tokens (the few-token kernels) give it and, with a
    gate of exactly one half, what the lane kernel's products with SwiGLU in between add to the routed sum."""
    import torch

    from inferq_amd import _lib, moe as M, qgemm as Q, synth as S

    rng = np.random.default_rng([tokens, hidden])
    gate = down = S.Q4_K
    layer = S.random_moe_layer(hidden, inter, 8, gate, down, rng)
    shared = {"shared_gate": (inter, hidden), "shared_up": (inter, hidden), "shared_down": (hidden, inter)}
    for name, (r, c) in shared.items():
        layer[name] = S.random_matrix(S.Q8_0, r, c, rng)
    t = {k: torch.from_numpy(v).to(gpu) for k, v in layer.items() if isinstance(v, np.ndarray)}
    x = torch.from_numpy(S.normal((tokens, hidden), rng)).to(gpu)
    lg = torch.from_numpy(S.normal((tokens, 8), rng)).to(gpu)

    def run(selector, step=tokens):
        args = () if selector is None else (t["shared_gate"], t["shared_up"], t["shared_down"], selector)
        m = M.QuantizedMoeLayer(hidden, inter, 8, 2, gate, down, t["gate"], t["up"], t["down"], *args,
                                shared_gate_dtype=S.Q8_0, shared_down_dtype=S.Q8_0)
        out = torch.empty_like(x)
        for i in range(0, tokens, step):
            m.forward_into(x[i:i + step].contiguous(), lg[i:i + step].contiguous(), out[i:i + step])
        return out.cpu().numpy()

    assert_bitexact(run(t["selector"]), run(t["selector"], 8), f"{tokens} tokens against 8")

    mats = {k: Q.QuantizedMatrix.view(t[k], S.Q8_0, r, c) for k, (r, c) in shared.items()}
    g, u = (mats[k].forward_via(x, _lib.PATH_LANES).cpu().numpy() for k in ("shared_gate", "shared_up"))
    one = np.float32(1)
    with np.errstate(over="ignore"):
        act = g / (one + np.exp(-g.astype(np.float64)).astype(np.float32)) * u
    y = mats["shared_down"].forward_via(torch.from_numpy(act).to(gpu), _lib.PATH_LANES).cpu().numpy()
    half = run(torch.zeros_like(t["selector"]))
    assert_bitexact(half, run(None) + y * np.float32(0.5), f"{tokens} tokens against the lane kernel")


# widths of one and several 256-value groups a wave, the widest (2048) and one past it, which runs as single products
@pytest.mark.parametrize("hidden,inter", [(256, 256), (768, 1280), (2048, 512), (512, 2048), (2304, 256)])
def test_q8_shared_expert_few_tokens(gpu, hidden, inter):
    """1, 5 and 48 tokens (two launches for the shared expert, combination and residual included) and 49 (its products
    apart) give each token what a call of 70 tokens gives it, bit for bit, with a residual added."""
    import torch

    from inferq_amd import moe as M, synth as S

    rng = np.random.default_rng([hidden, inter])
    layer = S.random_moe_layer(hidden, inter, 8, S.Q4_K, S.Q6_K, rng)
    for name, r, c in (("shared_gate", inter, hidden), ("shared_up", inter, hidden), ("shared_down", hidden, inter)):
        layer[name] = S.random_matrix(S.Q8_0, r, c, rng)
    t = {k: torch.from_numpy(v).to(gpu) for k, v in layer.items() if isinstance(v, np.ndarray)}
    m = M.QuantizedMoeLayer(hidden, inter, 8, 2, S.Q4_K, S.Q6_K, t["gate"], t["up"], t["down"], t["shared_gate"],
                            t["shared_up"], t["shared_down"], t["selector"], shared_gate_dtype=S.Q8_0,
                            shared_down_dtype=S.Q8_0, router=torch.from_numpy(S.normal((8, hidden), rng)).to(gpu))
    x, res = (torch.from_numpy(S.normal((70, hidden), rng)).to(gpu) for _ in range(2))
    x[3] = 0.0
    wide = torch.empty_like(x)
    m.forward_x_into(x, wide, res)
    for n in (1, 5, 48, 49):
        for r in (res, None):
            got = torch.full((n + 1, hidden), 7.0, device=gpu)
            m.forward_x_into(x[70 - n:].contiguous(), got[:n], None if r is None else r[70 - n:].contiguous())
            assert torch.all(got[n] == 7.0)
            if r is not None:
                assert_bitexact(got[:n].cpu().numpy(), wide[70 - n:].cpu().numpy(), f"{n} tokens")
            else:
                assert torch.allclose(got[:n] + res[70 - n:], wide[70 - n:], rtol=0, atol=0)  # res + v, one addition
