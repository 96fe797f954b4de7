"""LayerNorm and its projections in one launch (few rows): row and column edges of the tiles, every row width, fused and
separate projections, against the oracle, which has the kernels' rounding points.  Which of the sizes take that launch, and on
which of its tiles, is asserted where no GPU is needed (test_host_dispatch.py)."""

import numpy as np
import pytest
import torch

from oracle import lh_oracle as orc
from tests.conftest import assert_close

pytestmark = pytest.mark.gpu

# The result is the residual stream plus four products whose operands carry up to two roundings to the matmul type each, and
# whose sums add up in another order than the oracle's: 8 units of the type's rounding (2^-9, 2^-12) of the largest value.
TOLERANCE = {"bf16": 8 * 2.0**-9, "f16": 8 * 2.0**-12}


# A row is a multiple of 128 columns there, and up to 1024; the other widths (64, 192, 320, 704, 960) and many rows run the
# LayerNorm and the projections one after the other.
SIZES = [(1, 64), (15, 64), (17, 128), (33, 192), (100, 256), (250, 256), (700, 256), (31, 320), (100, 512), (16, 704), (101, 768),
         (3, 960), (65, 1024), (128, 1024)]
# Every width on each of the tiles of 16 x 32, 16 x 64 and 32 x 64, with those above: 128 (odd) columns are 4 (odd) steps of K,
# which eight waves share unevenly.
SIZES += [(340, 128), (1060, 128), (340, 256), (15, 384), (130, 384), (230, 384), (3, 512), (165, 512), (31, 640), (70, 640), (130, 640),
          (16, 768), (60, 768), (115, 768), (2, 896), (50, 896), (100, 896), (17, 1024)]


@pytest.mark.parametrize("mode,separate", [("bf16", False), ("f16", True)])
@pytest.mark.parametrize("T,C", SIZES)
def test_normed_products(T, C, mode, separate):
    from lighthouse_amd import ops

    rng = np.random.default_rng(T * C)
    dt = {"bf16": torch.bfloat16, "f16": torch.float16}[mode]
    draw = lambda *s: (rng.standard_normal(s) / np.sqrt(s[0])).astype(np.float32)
    weights = {"w_o": draw(C, C), "w_fc": draw(C, 4 * C), "w_proj": draw(4 * C, C)}
    weights.update({k: draw(C, C) for k in ("w_q", "w_k", "w_v")} if separate else {"w_qkv": draw(C, 3 * C)})
    p = {k: orc.round_to(v, mode) for k, v in weights.items()}
    for k, n in (("b_o", C), ("b_fc", 4 * C), ("b_proj", C)) + (() if separate else (("b_qkv", 3 * C),)):
        p[k] = rng.uniform(-0.5, 0.5, n).astype(np.float32)
        if not separate:
            p[k] = orc.round_to(p[k], mode)
    for k in ("ln1", "ln2"):
        p[k + "_g"], p[k + "_b"] = rng.uniform(0.5, 1.5, C).astype(np.float32), rng.uniform(-0.5, 0.5, C).astype(np.float32)
    # (rows of very different mean and spread: a row normalised by another's would show)
    x = (rng.standard_normal((1, T, C)) * rng.uniform(0.1, 2.0, (1, T, 1)) + rng.uniform(-2, 2, (1, T, 1))).astype(np.float32)
    dev = {k: torch.from_numpy(v).cuda().to(torch.float32 if k.startswith("ln") or (separate and k.startswith("b_")) else dt)
           for k, v in p.items()}
    got = ops.nanogpt_block(torch.from_numpy(x).cuda(), dev, C // 64, causal=not separate,
                            activation="relu" if separate else "gelu_tanh")
    want = orc.nanogpt_block(x, p, C // 64, mode=mode, causal=not separate, activation="relu" if separate else "gelu_tanh",
                             bias_f32=separate)
    assert_close(got.cpu().numpy(), want, TOLERANCE[mode], f"block {mode} T={T} C={C}")
