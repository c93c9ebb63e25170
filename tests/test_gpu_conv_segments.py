"""GPU: the vector forward of the causal conv at the edges of its token segments, at each segment length.

Against fp64. Bound: one rounding of the output plus fp32 arithmetic on five terms, 2^-18 of their magnitudes.
"""
import pytest
import torch
import torch.nn.functional as F

from sorernn_amd import causal_conv1d
from sorernn_amd.ops import qkv_causal_conv1d

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF_ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-24}


# 8 tokens a segment up to 4,099 x 4,096 (and for few channels at any length), then 16, 32 and 64
@pytest.mark.parametrize("b,t,c,docs", [
    (1, 1, 8, None), (2, 9, 264, None), (1, 257, 24, [1, 2, 7, 8, 9, 63, 65, 256]), (1, 4099, 4096, [8, 4098]),
    (1, 9001, 4096, [15, 16, 17, 6000]), (2, 9001, 4096, None), (1, 25007, 4096, [63, 64, 65, 24999]),
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_conv_forward_at_segment_edges(b, t, c, docs, dtype):
    gen = torch.Generator(DEV).manual_seed(t + c)
    bounds = [0, *(docs or []), t]
    n = len(bounds) - 1 if docs else b
    x = torch.randn(b, t, c, generator=gen, device=DEV).to(dtype)
    w = torch.rand(c, 4, generator=gen, device=DEV) - 0.5
    bias = 0.1 * torch.randn(c, generator=gen, device=DEV)
    init = torch.randn(n, c, 4, generator=gen, device=DEV).to(dtype)
    cu = torch.tensor(bounds) if docs else None
    y, fin = causal_conv1d(x, w, bias, initial_state=init, activation="silu", output_final_state=True,
                           cu_seqlens=None if cu is None else cu.to(DEV), cu_seqlens_cpu=cu)
    parts = [x[:, a:e] for a, e in zip(bounds[:-1], bounds[1:])] if docs else [x]
    at = 0
    for i, part in enumerate(parts):
        pre = init[i:i + 1] if docs else init
        full = torch.cat([pre.transpose(1, 2), part], 1)
        assert torch.equal(fin[i:i + 1] if docs else fin, full[:, -4:].transpose(1, 2))
        xs, e = full[:, 1:].double(), part.shape[1]
        z = sum(xs[:, j:j + e] * w[:, j].double() for j in range(4)) + bias.double()
        mag = sum((xs[:, j:j + e] * w[:, j].double()).abs() for j in range(4)) + bias.double().abs()
        r = F.silu(z)
        bound = HALF_ULP[dtype] * r.abs() * 1.01 + 2.0**-18 * 1.1 * mag + (2.0**-25 if dtype == torch.float16 else 0)
        err = (y[:, at:at + e].double() - r).abs()
        assert (err <= bound).all(), f"document {i}: {(err / bound).max().item():.2f} of the bound"
        at += e


@pytest.mark.parametrize("t", [1, 9, 4099, 9001, 25007])
def test_qkv_conv_at_segment_edges(t):
    """The one-pass q/k/v conv equals the plain conv at every segment length: the same formulas, of which either
    kernel may contract a multiply-add differently, so one ulp (|x| 2^-7) apart at most, and almost always equal."""
    gen = torch.Generator(DEV).manual_seed(t)
    x = torch.randn(1, t, 4096, generator=gen, device=DEV).bfloat16()
    w = torch.rand(4096, 4, generator=gen, device=DEV) - 0.5
    got = torch.cat(qkv_causal_conv1d(x, w, 1024, 2048, 128, l2norm=False), 2)
    ref = causal_conv1d(x, w, activation="silu")[0]
    assert ((got.float() - ref.float()).abs() <= 2.0**-7 * ref.float().abs().clamp_min(2.0**-14)).all()
    assert (got != ref).float().mean().item() <= 1e-2
