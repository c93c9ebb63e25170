"""GPU: the vector backward of the causal conv at the edges of its token segments and channel blocks.

Against fp64 autograd through the document-wise conv. Bounds: dx is one rounding of a sum of at most four
products, each of whose factors carries fp32 arithmetic (2^-18 of the terms' magnitudes); the fp32 weight
and bias gradients are bounded by 2^-18 of the sum of their terms' magnitudes.
"""
import pytest
import torch
import torch.nn.functional as F

from sorernn_amd import causal_conv1d

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF_ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-24}


def _ref(x, w, bias, init, bounds, act):
    outs = []
    for n, (a, e) in enumerate(zip(bounds[:-1], bounds[1:])):
        pre = init[n, :, 1:].T[None] if init is not None else x.new_zeros(1, 3, x.shape[2])
        xs = torch.cat([pre, x[:, a:e]], 1)
        outs.append(sum(xs[:, i:i + e - a] * w[:, i] for i in range(4)))
    y = torch.cat(outs, 1)
    y = y if bias is None else y + bias
    return F.silu(y) if act else y


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("t,c,docs", [
    (1, 4, None), (3, 260, None), (64, 256, [1, 2, 3, 16, 17]), (65, 1028, [15, 16, 18, 64]), (257, 512, None),
    (1031, 60, [62, 63, 64, 66, 128, 700, 1030]), (4099, 2048, [1000, 1001, 4095]), (9000, 4096, [4500]),
])
@pytest.mark.parametrize("full", [True, False])
def test_conv_backward_at_segment_edges(t, c, docs, dtype, full):
    gen = torch.Generator().manual_seed(t + c)
    bounds = [0, *(docs or []), t]
    n = len(bounds) - 1
    x, dy = (torch.randn(1, t, c, generator=gen).to(dtype) for _ in range(2))
    w = torch.rand(c, 4, generator=gen) - 0.5
    bias = 0.1 * torch.randn(c, generator=gen) if full else None
    init = torch.randn(n, c, 4, generator=gen).to(dtype) if full else None
    cu = torch.tensor(bounds) if docs else None
    lv = [v for v in (x, w, bias, init) if v is not None]
    dev = [v.to(DEV).requires_grad_(True) for v in lv]
    y, _ = causal_conv1d(dev[0], dev[1], dev[2] if full else None, initial_state=dev[3] if full else None,
                         activation="silu" if full else None, cu_seqlens=None if cu is None else cu.to(DEV), cu_seqlens_cpu=cu)
    got = torch.autograd.grad(y, dev, dy.to(DEV))
    ref_in = [v.to(DEV).double().requires_grad_(True) for v in lv]
    yr = _ref(ref_in[0], ref_in[1], ref_in[2] if full else None, ref_in[3] if full else None, bounds, full)
    ref = torch.autograd.grad(yr, ref_in, dy.to(DEV).double())
    # |dz| <= 1.1 |dy| (the largest slope of SiLU), |w| <= 0.5, at most four terms of each dx
    m = F.pad(dy.to(DEV).double().abs(), (0, 0, 0, 3))
    near = torch.stack([m[:, j:j + t] for j in range(4)]).amax(0)
    scale = [4 * 0.55 * near, 1.1 * (dy.double().abs().sum((0, 1))[:, None] * x.double().abs().amax((0, 1))[:, None]).to(DEV),
             1.1 * dy.double().abs().sum((0, 1)).to(DEV)]
    names = ["dx", "dweight", "dbias"]
    if init is not None:
        scale[1] = scale[1] + 1.1 * dy.double().abs().sum((0, 1)).to(DEV)[:, None] * init.double().abs().amax((0, 2)).to(DEV)[:, None]
    for name, a, r, sc in zip(names, got, ref, scale):
        bound = HALF_ULP[a.dtype] * r.abs() * 1.01 + 2.0**-18 * sc + (2.0**-25 if dtype == torch.float16 else 0)
        err = (a.double() - r).abs()
        assert (err <= bound).all(), f"{name}: {(err / bound).max().item():.2f} of the bound"
    if init is not None:  # added in fp32, then rounded to the state's type
        err, r = (got[3].double() - ref[3]).abs(), ref[3].abs()
        bound = HALF_ULP[dtype] * r * 1.01 + 2.0**-18 * 4 * 0.55 * dy.double().abs().max().item() + 2.0**-25
        assert (err <= bound).all(), f"dinit: {(err / bound).max().item():.2f} of the bound"


def test_conv_backward_does_not_leak_nan_across_documents():
    x, dy = torch.randn(1, 40, 64, device=DEV).bfloat16(), torch.randn(1, 40, 64, device=DEV).bfloat16()
    x[0, 20] = float("nan")
    dy[0, 21] = float("nan")
    cu = torch.tensor([0, 20, 30, 40])
    x.requires_grad_(True)
    y, _ = causal_conv1d(x, torch.rand(64, 4, device=DEV), activation="silu", cu_seqlens=cu.to(DEV), cu_seqlens_cpu=cu)
    (dx,) = torch.autograd.grad(y, x, dy)
    assert torch.isfinite(dx[0, :20]).all() and torch.isfinite(dx[0, 30:]).all() and not torch.isfinite(dx[0, 20]).any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_conv_parameter_gradients_of_saturated_activations(dtype):
    """The fp32 parameter gradients carry SiLU's slope in fp32, whatever type the activations have. Over 4,096 biases its
    errors (18 units in the mean square at -40 to -60, from expf's argument reduction) leave 0.3 units of their mean,
    the sums over equal terms at most one; 2 are allowed. A bias of the errors would stay whole."""
    dy, bias = torch.ones(1, 64, 4096, dtype=dtype, device=DEV), torch.linspace(-60, -40, 4096, device=DEV).requires_grad_(True)
    x = torch.zeros(1, 64, 4096, dtype=dtype, device=DEV).requires_grad_(True)
    y, _ = causal_conv1d(x, torch.ones(4096, 4, device=DEV), bias, activation="silu")
    (got,) = torch.autograd.grad(y, bias, dy)
    z = bias.detach().double().requires_grad_(True)
    (slope,) = torch.autograd.grad(F.silu(z).sum(), z)
    err = ((got.double() - 64 * slope) / (64 * slope)).mean().abs().item()
    assert err <= 2 * 2.0**-24, err * 2**24
