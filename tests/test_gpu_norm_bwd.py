"""GPU: the vector backward of the L2 norm and of the (gated) RMSNorm at the edges of its tiles.

Against fp64 autograd on the same inputs. The bound per element is one rounding of the result to its
type (half a unit in the last place) plus 2^-20 of the row's largest term for the fp32 arithmetic; the
fp32 parameter gradients, sums over all rows, are bounded by 2^-20 of the sum of their terms' magnitudes.
"""
import pytest
import torch
import torch.nn.functional as F

from sorernn_amd import l2norm, rms_norm_gated

pytestmark = pytest.mark.gpu
DEV = "cuda"
# relative to the value: 8, 11 and 24 significant bits (a value just above 2^k has units of 2^(k-7), 2^(k-10), 2^(k-23))
HALF_ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-24}


def _check(name, got, ref, row_scale):
    err = (got.double().cpu() - ref).abs()
    # subnormal fp16 results round to a fixed step of 2^-24
    bound = HALF_ULP[got.dtype] * ref.abs() * 1.01 + 2.0**-20 * row_scale + (2.0**-25 if got.dtype == torch.float16 else 0)
    assert (err <= bound).all(), f"{name}: {(err / bound).max().item():.2f} of the bound"


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("rows", [1, 3, 17, 64, 1025, 70001])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_norm_backwards_at_tile_edges(dtype, rows, d):
    gen = torch.Generator().manual_seed(rows + d)
    x, g, dy = (torch.randn(rows, d, generator=gen).to(dtype) for _ in range(3))
    w, b = torch.randn(d, generator=gen), 0.1 * torch.randn(d, generator=gen)
    xr = x.double().requires_grad_(True)
    xd = x.to(DEV).requires_grad_(True)
    (ref,) = torch.autograd.grad(F.normalize(xr, dim=-1), xr, dy.double())
    (got,) = torch.autograd.grad(l2norm(xd), xd, dy.to(DEV))
    _check("l2 dx", got, ref, (dy.double().abs().amax(-1, keepdim=True) / x.double().norm(dim=-1, keepdim=True)))
    for act, bias, gated in (("swish", None, True), (None, b, True), ("swish", b, False)):
        lv = [x, g, w] + ([b] if bias is not None else [])
        rf = [t.double().requires_grad_(True) for t in lv]
        rr = torch.rsqrt(rf[0].square().mean(-1, keepdim=True) + 1e-6)
        u = rf[0] * rr * rf[2] + (rf[3] if bias is not None else 0)
        y = u * (F.silu(rf[1]) if act else rf[1]) if gated else u
        dev = [t.to(DEV).requires_grad_(True) for t in lv]
        yd = rms_norm_gated(dev[0], dev[1] if gated else None, dev[2], dev[3] if bias is not None else None, activation=act)
        pick = [0] + ([1] if gated else []) + [2] + ([3] if bias is not None else [])
        refs = torch.autograd.grad(y, [rf[i] for i in pick], dy.double())
        gots = torch.autograd.grad(yd, [dev[i] for i in pick], dy.to(DEV))
        gate = (F.silu(rf[1]) if act else rf[1]).detach() if gated else torch.ones(1, dtype=torch.double)
        du = dy.double() * gate
        top = lambda t: t.abs().amax(-1, keepdim=True)  # noqa: E731
        n, rd = (rf[0] * rr).detach(), rr.detach()
        scale = {0: rd * top(du * rf[2].detach()) * (1 + top(n)) ** 2, 2: (du * n).abs().sum(0), 3: du.abs().sum(0)}
        # u = n w + b can cancel: its fp32 error is relative to the two terms, not to their sum
        u_terms = (n * rf[2].detach()).abs() + (b.double().abs() if bias is not None else 0)
        scale[1] = dy.double().abs() * u_terms * (1 + g.double().abs())
        for i, a, r in zip(pick, gots, refs):
            _check(f"rms {act} gated={gated} grad {i}", a, r, scale[i])


@pytest.mark.parametrize("size", [1e-3, 1e10, 1e15, 1e17])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rms_backward_of_large_and_small_rows(dtype, size):
    """r^3 leaves fp32's range long before the row's sum of squares does. dx = r (du w - n mean(du w n)): the bound is
    one rounding and 2^-20 of r's largest product, n and the mean of 128 products each of at most |n| <= 12."""
    gen = torch.Generator().manual_seed(5)
    x, dy = ((size if i == 0 else 1.0) * torch.randn(33, 128, generator=gen) for i in range(2))
    x, dy, w = x.to(dtype), dy.to(dtype), torch.randn(128, generator=gen)
    xr, wr = x.double().requires_grad_(True), w.double().requires_grad_(True)
    rr = torch.rsqrt(xr.square().mean(-1, keepdim=True) + 1e-6)
    ref = torch.autograd.grad(xr * rr * wr, [xr, wr], dy.double())
    xd, wd = x.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    got = torch.autograd.grad(rms_norm_gated(xd, None, wd), [xd, wd], dy.to(DEV))
    rd, n = rr.detach(), (xr * rr).detach()
    _check("dx", got[0], ref[0], rd * (dy.double() * w.double()).abs().amax(-1, keepdim=True) * (1 + n.abs().amax()) ** 2)
    _check("dweight", got[1], ref[1], (dy.double() * n).abs().sum(0))


@pytest.mark.parametrize("rows", [1, 31, 33, 1025])
@pytest.mark.parametrize("gated", [True, False])
def test_rms_backward_without_eps(rows, gated):
    """eps = 0: the rows that fill the last tile up take no part in the parameter gradients."""
    gen = torch.Generator().manual_seed(rows)
    x, g, dy = (torch.randn(rows, 128, generator=gen) for _ in range(3))
    w, b = torch.randn(128, generator=gen), torch.randn(128, generator=gen)
    ref_in = [t.double().requires_grad_(True) for t in (x, w, b)]
    u = ref_in[0] * torch.rsqrt(ref_in[0].square().mean(-1, keepdim=True)) * ref_in[1] + ref_in[2]
    act = F.silu(g.double()) if gated else torch.ones(1).double()
    ref = torch.autograd.grad(u * act, ref_in, dy.double())
    dev = [t.to(DEV).requires_grad_(True) for t in (x, w, b)]
    got = torch.autograd.grad(rms_norm_gated(dev[0], g.to(DEV) if gated else None, dev[1], dev[2], eps=0.0), dev, dy.to(DEV))
    n = (x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True))).abs()
    du = (dy.double() * act).abs()
    _check("dx", got[0], ref[0], n.amax() ** 2 * (du * w.double().abs()).amax(-1, keepdim=True)
           * torch.rsqrt(x.double().square().mean(-1, keepdim=True)))
    _check("dweight", got[1], ref[1], (du * n).sum(0))
    _check("dbias", got[2], ref[2], du.sum(0))


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_rms_parameter_gradients_of_saturated_gates(dtype):
    """The fp32 parameter gradients carry the gate's activation in fp32, whatever type the rows have: terms of one size
    over 128 gates. A gate's activation is off by up to 40 units (expf's argument reduction at -50), by a third of that in
    the mean square and either way: 14 / sqrt(128) units for the sum, 5 are allowed. A bias would add up to all of them."""
    g = (-50 + torch.arange(128) / 32).repeat(64)[:, None].expand(-1, 128).to(dtype).contiguous()
    dy = (0.5 * torch.exp(-48 - g.float())).to(dtype)
    x = torch.randn(g.shape, generator=torch.Generator().manual_seed(1)).to(dtype)
    b = torch.zeros(128, device=DEV, requires_grad=True)
    y = rms_norm_gated(x.to(DEV), g.to(DEV), torch.ones(128, device=DEV), b)
    (got,) = torch.autograd.grad(y, b, dy.to(DEV))
    ref = (dy.double() * F.silu(g.double())).sum(0)
    err = ((got.double().cpu() - ref) / ref).abs().max().item()
    assert err <= 5 * 2.0**-24, err * 2**24


def test_batched_gradients():
    """``is_grads_batched``: the device's backward thread runs under the caller's vmap, once per gradient."""
    gen = torch.Generator().manual_seed(3)
    x, dy = (torch.randn(33, 128, generator=gen).bfloat16().to(DEV).requires_grad_(True), torch.randn(3, 33, 128, generator=gen))
    dy, y = dy.bfloat16().to(DEV), l2norm(x)
    (got,) = torch.autograd.grad(y, x, dy, is_grads_batched=True, retain_graph=True)
    for i in range(3):
        assert torch.equal(got[i], torch.autograd.grad(y, x, dy[i], retain_graph=True)[0])
