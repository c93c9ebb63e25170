"""GPU: the recurrent kernels around their step sizes, against the fp64 oracle.

Lengths around the few-token kernel's 4 tokens and the 16-token steps, sequences of mixed lengths, value heads
sharing q/k heads, gates that decay to nothing, rows at odd element offsets, and a NaN that must not reach
earlier tokens, other heads or other sequences. fp32 bound: at most 2^-17 of the largest magnitude (T <= 70
tokens of K <= 128 products, fp32 sums); 16-bit outputs add half a unit in the last place.
"""
import pytest
import torch
import torch.nn.functional as F

from oracle import recurrent_gated_delta_rule
from sorernn_amd import fused_recurrent_gated_delta_rule

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF_ULP = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 2.0**-24}


def _inputs(b, t, h, hv, kd, vd, n, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    q, k = (F.normalize(torch.randn(b, t, h, kd, generator=gen), dim=-1).to(dtype) for _ in range(2))
    v = torch.randn(b, t, hv, vd, generator=gen).to(dtype)
    g = -F.softplus(torch.randn(b, t, hv, generator=gen)) * (torch.rand(b, t, hv, generator=gen) * 6 - 4).exp()
    g[torch.rand(b, t, hv, generator=gen) < 0.05] = -float("inf")  # a token that forgets everything
    g[torch.rand(b, t, hv, generator=gen) < 0.05] = -300.0
    beta = torch.randn(b, t, hv, generator=gen).sigmoid()
    return q, k, v, g, beta, torch.randn(n, hv, kd, vd, generator=gen)


def _check(o, st, o_ref, st_ref, dtype):
    err, top = (o.double().cpu() - o_ref).abs(), o_ref.abs().max().item()
    bound = 2.0**-17 * top + HALF_ULP[dtype] * o_ref.abs() * 1.01
    assert (err <= bound).all(), f"o: {(err / bound).max().item():.2f} of the bound"
    assert ((st.double().cpu() - st_ref).abs() <= 2.0**-17 * st_ref.abs().max()).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("t", [1, 3, 4, 5, 8, 15, 16, 17, 33, 70])
@pytest.mark.parametrize("b,h,hv,kd,vd", [(2, 2, 4, 128, 128), (1, 3, 3, 64, 128), (3, 1, 2, 128, 64), (1, 2, 2, 64, 64)])
def test_lengths_around_the_steps(b, h, hv, kd, vd, t, dtype):
    q, k, v, g, beta, h0 = _inputs(b, t, h, hv, kd, vd, b, dtype, 10 * t + b)
    o, st = fused_recurrent_gated_delta_rule(*(x.to(DEV) for x in (q, k, v, g, beta)), initial_state=h0.to(DEV),
                                             output_final_state=True)
    o_ref, st_ref = recurrent_gated_delta_rule(*(x.double() for x in (q, k, v, g, beta)), kd**-0.5, h0.double(), True)
    _check(o, st, o_ref.double(), st_ref.double(), dtype)


@pytest.mark.parametrize("lens", [[1, 2, 1, 4], [1, 40, 3, 16, 17, 1], [5, 5, 2, 1]])
def test_mixed_lengths_with_norm_and_gate_in_kernel(lens):
    t, n = sum(lens), len(lens)
    q, k, v, _, _, h0 = _inputs(1, t, 2, 4, 128, 128, n, torch.bfloat16, t)
    gen = torch.Generator().manual_seed(t)
    q, k = (3 * torch.randn(q.shape, generator=gen)).bfloat16(), (3 * torch.randn(k.shape, generator=gen)).bfloat16()
    k[0, t // 2] = 0  # a zero row: 0 / max(0, 1e-12)
    a, bl = (torch.randn(1, t, 4, generator=gen).bfloat16() for _ in range(2))
    a_log, dtb = torch.rand(4, generator=gen) * 2, torch.randn(4, generator=gen)
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()])
    o, st = fused_recurrent_gated_delta_rule(
        *(x.to(DEV) for x in (q, k, v, a, bl)), initial_state=h0.to(DEV), output_final_state=True, cu_seqlens=cu.to(DEV),
        cu_seqlens_cpu=cu, use_qk_l2norm_in_kernel=True, use_beta_sigmoid_in_kernel=True, use_gate_in_kernel=True,
        A_log=a_log.to(DEV), dt_bias=dtb.to(DEV))
    g = -a_log.double().exp() * F.softplus(a.double() + dtb.double())
    o_ref, st_ref = recurrent_gated_delta_rule(F.normalize(q.double(), dim=-1), F.normalize(k.double(), dim=-1), v.double(), g,
                                               bl.double().sigmoid(), 128**-0.5, h0.double(), True, cu_seqlens=cu)
    _check(o, st, o_ref.double(), st_ref.double(), torch.bfloat16)


@pytest.mark.parametrize("t", [3, 37])
def test_rows_at_odd_element_offsets(t):
    q, k, v, g, beta, h0 = _inputs(1, t, 2, 2, 128, 128, 1, torch.bfloat16, t)

    def odd(x):  # the same values, contiguous, one element into a larger allocation
        flat = torch.empty(x.numel() + 1, dtype=x.dtype, device=DEV)
        flat[1:] = x.flatten().to(DEV)
        return flat[1:].view(x.shape)

    o, st = fused_recurrent_gated_delta_rule(*(odd(x) for x in (q, k, v, g, beta)), initial_state=odd(h0), output_final_state=True)
    o_ref, st_ref = recurrent_gated_delta_rule(*(x.double() for x in (q, k, v, g, beta)), 128**-0.5, h0.double(), True)
    _check(o, st, o_ref.double(), st_ref.double(), torch.bfloat16)


@pytest.mark.parametrize("t,bad", [(4, 2), (40, 21), (16, 15)])
@pytest.mark.parametrize("where", ["q", "k", "v", "g", "beta"])
def test_nan_reaches_only_later_tokens_of_its_head(t, bad, where):
    x = dict(zip(("q", "k", "v", "g", "beta"), _inputs(2, t, 2, 2, 64, 64, 2, torch.float32, t)[:5]))
    x[where][0, bad, 1] = float("nan")
    o, st = fused_recurrent_gated_delta_rule(*(x[n].to(DEV) for n in ("q", "k", "v", "g", "beta")), output_final_state=True)
    assert torch.isfinite(o[0, :bad]).all() and torch.isfinite(o[:, :, 0]).all() and torch.isfinite(o[1]).all()
    assert torch.isfinite(st[1]).all() and torch.isfinite(st[0, 0]).all()
    assert not torch.isfinite(o[0, bad, 1]).any()
    if where == "q":
        assert torch.isfinite(o[0, bad + 1:]).all() and torch.isfinite(st).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("t", [3, 16, 23, 40])
@pytest.mark.parametrize("kd,vd", [(128, 128), (64, 64), (128, 64), (64, 128)])
def test_decays_above_one(kd, vd, t, dtype):
    """Nine log decays of 10, then nine of -10, of tiny states and values: the products of the decays leave fp32's range, the
    states stay in it. Error of a token: T sums of K terms, sqrt(K) T 2^-24 < 2^-15 of its state's largest column."""
    q, k, v, _, beta, h0 = _inputs(1, t, 2, 2, kd, vd, 1, dtype, t)
    g = torch.zeros(1, t, 2)
    g[:, 2:11], g[:, 11:20] = 10.0, -10.0
    v = 1e-10 * v
    o, st = fused_recurrent_gated_delta_rule(*(x.to(DEV) for x in (q, k, v, g, beta)), initial_state=1e-10 * h0.to(DEV),
                                             output_final_state=True)
    s, scale = 1e-10 * h0.double(), kd**-0.5
    for i in range(t):
        s = s * g[:, i].double().exp()[..., None, None]
        ki, qi = k[:, i].double(), q[:, i].double()
        d = beta[:, i].double()[..., None] * (v[:, i].double() - (s * ki[..., None]).sum(-2))
        s = s + ki[..., None] * d[..., None, :]
        ref, top = scale * (s * qi[..., None]).sum(-2), s.norm(dim=-2).amax(-1, keepdim=True)
        err, bound = (o[:, i].double().cpu() - ref).abs(), 2.0**-15 * scale * top + HALF_ULP[dtype] * ref.abs() * 1.01
        assert (err <= bound).all(), f"token {i}: {(err / bound).max().item():.2f} of the bound"
    assert ((st.double().cpu() - s).abs() <= 2.0**-15 * s.norm(dim=-2, keepdim=True).amax(-1, keepdim=True)).all()


@pytest.mark.parametrize("t", [4, 16, 40])
def test_decays_above_one_leave_a_zero_state(t):
    q, k, v, _, beta, _ = _inputs(2, t, 2, 2, 128, 128, 2, torch.bfloat16, t)
    v[:, 7:] = 0  # the state is zero from the -inf on
    g = torch.full((2, t, 2), 20.0)
    g[:, 7:8] = -float("inf")
    g[:, :7] = 0
    o, st = fused_recurrent_gated_delta_rule(*(x.to(DEV) for x in (q, k, v, g, beta)), output_final_state=True)
    assert torch.isfinite(o).all() and not o[:, 7:].any() and (t < 8 or not st.any())


@pytest.mark.parametrize("n,t", [(15, 4), (15, 5), (16, 6), (16, 7), (31, 6), (32, 8), (32, 9)])
def test_both_sides_of_the_few_token_lines(n, t):
    """16 heads of 128: the line lies at 4 tokens, at 6 from 16 sequences up and at 8 from 32 up."""
    q, k, v, g, beta, h0 = _inputs(n, t, 16, 16, 128, 128, n, torch.bfloat16, 100 * n + t)
    o, st = fused_recurrent_gated_delta_rule(*(x.to(DEV) for x in (q, k, v, g, beta)), initial_state=h0.to(DEV),
                                             output_final_state=True)
    o_ref, st_ref = recurrent_gated_delta_rule(*(x.double() for x in (q, k, v, g, beta)), 128**-0.5, h0.double(), True)
    _check(o, st, o_ref.double(), st_ref.double(), torch.bfloat16)


@pytest.mark.parametrize("long", [65, 193, 194])
def test_one_long_sequence_among_single_tokens(long):
    """64 packed sequences, 63 of one token: the mean length picks the kernel (193 + 63 is 4 tokens a sequence).
    The decays forget: a state holds the rounding of some dozen tokens, and the module's bound serves 194 as well."""
    lens = [1] * 40 + [long] + [1] * 23
    q, k, v, g, beta, h0 = _inputs(1, sum(lens), 2, 2, 128, 128, 64, torch.bfloat16, long)
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()])
    o, st = fused_recurrent_gated_delta_rule(*(x.to(DEV) for x in (q, k, v, g, beta)), initial_state=h0.to(DEV),
                                             output_final_state=True, cu_seqlens=cu.to(DEV), cu_seqlens_cpu=cu)
    o_ref, st_ref = recurrent_gated_delta_rule(*(x.double() for x in (q, k, v, g, beta)), 128**-0.5, h0.double(), True, cu_seqlens=cu)
    _check(o, st, o_ref.double(), st_ref.double(), torch.bfloat16)
