"""A forward of few rows, whose launches touch the weights of the block after them: the same bits as the blocks called one by one,
which know of no block after theirs, fused and separate projections, weights of sizes that no share of the lines divides."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("separate", [False, True])
@pytest.mark.parametrize("T,C", [(1, 128), (33, 256), (100, 768), (130, 1024), (100, 192)])
def test_forward_is_its_blocks(T, C, separate):
    from lighthouse_amd import ops

    g = torch.Generator(device="cuda").manual_seed(T + C)
    draw = lambda *s: torch.randn(s, device="cuda", generator=g) / s[0] ** 0.5

    def block():
        weights = {"w_o": (C, C), "w_fc": (C, 4 * C), "w_proj": (4 * C, C)}
        weights.update({"w_q": (C, C), "w_k": (C, C), "w_v": (C, C)} if separate else {"w_qkv": (C, 3 * C)})
        p = {k: draw(*s).bfloat16() for k, s in weights.items()}
        for k, n in (("b_o", C), ("b_fc", 4 * C), ("b_proj", C)) + (() if separate else (("b_qkv", 3 * C),)):
            p[k] = draw(n) if separate else draw(n).bfloat16()
        for k in ("ln1", "ln2"):
            p[k + "_g"], p[k + "_b"] = 1.0 + 0.1 * draw(C), 0.1 * draw(C)
        return p

    layers, x = [block() for _ in range(3)], draw(1, T, C)
    options = {"causal": not separate, "activation": "relu" if separate else "gelu_tanh"}
    lnf_g, lnf_b, lm_w = 1.0 + 0.1 * draw(C), 0.1 * draw(C), draw(C, 264).bfloat16()
    got = ops.nanogpt_forward(x, layers, lnf_g, lnf_b, lm_w, None, C // 64, **options)
    for p in layers:
        x = ops.nanogpt_block(x, p, C // 64, **options)
    want = ops.gemm(ops.layer_norm(x.view(T, C), lnf_g, lnf_b, out_dtype=torch.bfloat16), lm_w, out_dtype=torch.float32)
    assert torch.equal(got.view(T, 264), want)
