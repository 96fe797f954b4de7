"""A forward of few rows, whose launches touch the weights of the ones after them: the same bits as the blocks called one by one,
which know of no block after theirs, fused and separate projections, weights of sizes that no share of the lines divides.  Which
launches touch what is asserted where no GPU is needed."""

import ctypes
import multiprocessing
import re

import pytest
import torch

from tests import recorded_launches as rec

# T, C: do the first and the second product of the MLP touch what later launches read ("separate": separate q, k and v alone, fewer lines)?
SIZES = {(1, 128): (False, True), (100, 192): (False, True), (33, 256): (False, False), (300, 256): (False, True), (200, 384): (True, True),
         (16, 512): (True, False), (64, 512): (False, False), (100, 512): (True, False), (200, 512): (True, True), (33, 768): (True, False),
         (100, 768): (True, True), (160, 768): (False, "separate"), (200, 768): (False, True), (16, 1024): (True, False), (80, 1024): (True, True)}


@pytest.mark.gpu
@pytest.mark.parametrize("separate", [False, True])
@pytest.mark.parametrize("T,C", [size for size, touching in SIZES.items() if any(touching)])
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


def _launch(n):
    tile = re.search(r"gemm_(normed|small)_\w+ILi\dELi(\d)ELi(\d)E", n.name)
    if not tile:
        return n.name, None, 0, n.gemm.b, n.touched
    kind, mt, nt = tile.group(1), int(tile.group(2)), int(tile.group(3))
    tiles = -(-n.gemm.M // (16 * mt)) * -(-n.gemm.N // (16 * nt))
    return n.name, (kind, mt, nt), n.grid - -(-tiles // 8) * 8, n.gemm.b, n.touched


def _forward(so, sizes):
    """{(T, C, type, separate): (weights by name of each block, the launches: name, tile, workgroups behind the work's, B, ranges to touch)}"""
    r, lib, found = rec.Recorder(so), rec._lib, {}
    for T, C in sizes:
        for dtype, separate in ((lib.BF16, False), (lib.F16, True)):
            blocks = (lib.NanoGPTBlockParams * 3)()
            weights = []
            for k, p in enumerate(blocks):
                missing = ("w_qkv", "b_qkv") if separate else ("w_q", "w_k", "w_v")
                weights.append({name: (3 << 50) + ((32 * k + i) << 32) for i, (name, _) in enumerate(p._fields_) if name not in missing})
                for name, address in weights[-1].items():
                    setattr(p, name, address)
            opts = ctypes.byref(lib.NanoGPTBlockOpts(1, lib.ACT_GELU_TANH, dtype, 4 * C))
            need = r.lib.lh_hip_nanogpt_forward_workspace_bytes(1, T, C, 264, dtype, opts)
            rc, launches = r.calls("lh_hip_nanogpt_forward", 1 << 50, 2 << 50, blocks, 3, 5 << 50, 6 << 50, 7 << 50, None, 1, T, C, C // 64,
                                   264, 1e-5, dtype, opts, 8 << 50, need, None)
            assert rc == 0, r.lib.lh_hip_last_error()
            found[T, C, dtype, separate] = weights, [_launch(n) for n in launches]
    return found


def test_who_touches_what(tmp_path):
    """The first product of an MLP touches the second one's weights, the second those of the block after its own: whole ranges, in
    workgroups behind those of the work."""
    with multiprocessing.get_context("spawn").Pool(1) as pool:
        found = pool.apply(_forward, (rec.build(tmp_path), list(SIZES)))
    reached = set()
    for (T, C, dtype, separate), (weights, launches) in found.items():
        lines = {"w_qkv": 3 * C * C // 64, "w_fc": 4 * C * C // 64, "w_proj": 4 * C * C // 64} | dict.fromkeys(("w_q", "w_k", "w_v", "w_o"), C * C // 64)
        first, second = SIZES[T, C][0], SIZES[T, C][1] in (True, "separate" if separate else None)
        expected = []  # (block by block)
        for k in range(3):
            if first:
                expected.append(("normed", [(weights[k]["w_proj"], lines["w_proj"])]))
            if second and k < 2:
                expected.append(("small", [(weights[k + 1][n], lines[n]) for n in (("w_q", "w_k", "w_v") if separate else ("w_qkv", "w_o", "w_fc"))]))
        touching = [n for n in launches if n[4] and n[2]]
        assert [(n[1][0], n[4]) for n in touching] == expected, (T, C, separate)
        assert [n[2] for n in touching] == [sum(-(-c // 2048) for _, c in ranges) for _, ranges in expected]
        assert all(n[3] == weights[k]["w_proj"] for k, n in enumerate(n for n in touching if n[1][0] == "small"))
        reached |= {(dtype, *n[1]) for n in touching}
    for dtype in (rec._lib.BF16, rec._lib.F16):
        assert reached >= {(dtype, *tile) for tile in (("normed", 1, 2), ("normed", 1, 4), ("normed", 2, 4), ("small", 1, 2), ("small", 2, 2))}
