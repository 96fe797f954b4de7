"""The small-problem attention kernel: both tile counts, edges of tiles and key steps, strided views, large scores."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _view(Z, H, T, dtype, seed):
    """[Z, H, T, 64] normal values as a strided view of [Z, T + 40, H, 72]; everything around it holds NaN."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    buf = torch.full((Z, T + 40, H, 72), float("nan"), device="cuda", dtype=dtype)
    buf[:, :T, :, :64] = torch.randn(Z, T, H, 64, device="cuda", generator=g).to(dtype)
    return buf[:, :T, :, :64].transpose(1, 2)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype,eps", [(torch.bfloat16, 2.0**-8), (torch.float16, 2.0**-11)])
@pytest.mark.parametrize("gain", [1.0, 40.0])  # (40: the softmax is nearly one-hot, its maximum moves from step to step)
@pytest.mark.parametrize("Z,H,T", [(1, 1, 65), (1, 12, 100), (2, 2, 256),   # 16 rows; fewer steps than waves
                                   (1, 17, 255), (2, 12, 192),              # 16 rows, more workgroups than CUs
                                   (2, 3, 1000), (1, 14, 401),              # 32 rows
                                   (1, 8, 1500)])                           # causal only: two workgroups per CU
def test_small_attention(Z, H, T, gain, dtype, eps, causal):
    from lighthouse_amd import ops

    q, k, v = (_view(Z, H, T, dtype, seed) for seed in (1, 2, 3))
    q = q * gain
    out = torch.full((Z, H, T + 9, 64), 7.0, device="cuda", dtype=dtype)
    ops.attention(q, k, v, causal=causal, out=out[:, :, :T])
    assert bool((out[:, :, T:] == 7.0).all())
    s = q.double() @ k.double().transpose(-1, -2).contiguous() * 0.125
    if causal:
        s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device="cuda").triu(1), -float("inf"))
    p = s.softmax(-1)
    want = p @ v.double().contiguous()
    # P and the result are each rounded once, by eps at most (f16: P may also lose 2^-25 where it is subnormal); the f32
    # scores, up to `largest`, leave 2^-20 of their size in the exponent whatever the scaling.  Where the large kernel
    # is the faster one (non-causal 1500) it also rounds the scaled Q.
    largest = float(s[s > -float("inf")].abs().max())
    q_rounding = eps * largest if T == 1500 and not causal else 0.0
    bound = (2 * eps + 2.0**-20 * largest + 2 * q_rounding) * (p @ v.double().abs().contiguous()) + 2.0**-24 * T
    assert bool(((out[:, :, :T].double() - want).abs() <= bound).all())


@pytest.mark.parametrize("scale_in_f32", [False, True])
@pytest.mark.parametrize("stages", [3, 4])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype,eps", [(torch.bfloat16, 2.0**-8), (torch.float16, 2.0**-11)])
@pytest.mark.parametrize("Z,H,T", [(2, 3, 1000), (1, 2, 200), (1, 1, 300), (1, 2, 65), (2, 3, 512)])
def test_large_kernels_on_request(Z, H, T, dtype, eps, causal, stages, scale_in_f32):
    """Few query rows on the 128-row kernels, which these shapes run only on request: lengths that end inside a key
    tile, Q scaled and rounded or the scores scaled in f32."""
    from lighthouse_amd import ops

    q, k, v = (_view(Z, H, T, dtype, seed) for seed in (4, 5, 6))
    out = torch.full((Z, H, T + 9, 64), 7.0, device="cuda", dtype=dtype)
    ops.attention(q, k, v, causal=causal, out=out[:, :, :T], rows_per_wave=32, stages=stages, scale_in_f32=scale_in_f32)
    assert bool((out[:, :, T:] == 7.0).all())
    s = q.double() @ k.double().transpose(-1, -2).contiguous() * 0.125
    size = q.double().abs() @ k.double().abs().transpose(-1, -2).contiguous() * 0.125
    if causal:
        mask = torch.ones(T, T, dtype=torch.bool, device="cuda").triu(1)
        s, size = s.masked_fill(mask, -float("inf")), size.masked_fill(mask, 0.0)
    p = s.softmax(-1)
    want = p @ v.double().contiguous()
    # P and the result are rounded once, by eps at most (f16: P may also lose 2^-25 where it is subnormal).  A score is off
    # by 2^-20 of the sum of its terms' sizes (f32) plus, where the scaled Q is rounded, eps of it; P by e^(2 off) - 1.
    off = float(size.max()) * (2.0**-20 + (0.0 if scale_in_f32 else eps))
    bound = (2 * eps + 2.7183**(2 * off) - 1) * (p @ v.double().abs().contiguous()) + 2.0**-24 * T
    assert bool(((out[:, :, :T].double() - want).abs() <= bound).all())
