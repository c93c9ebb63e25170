"""GPU: q and k normalised in one launch are bitwise the two separate launches, at the edges of a block's rows,
for unaligned rows and for the head dims and types without a vector path; and the rule that picks that route."""
import pytest
import torch

from sorernn_amd import _lib, l2norm, ops
from sorernn_amd.ops import _l2norm_first, _l2norm_qk

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 1, 1, 128), (1, 63, 1, 128), (2, 129, 3, 64), (1, 1000, 16, 128), (1, 7, 3, 48)])
@pytest.mark.parametrize("offset", [0, 1])
def test_qk_l2norm_in_one_launch(shape, dtype, offset):
    gen = torch.Generator().manual_seed(sum(shape))

    def make():  # contiguous, `offset` elements into its allocation
        x = torch.randn(shape, generator=gen).to(dtype)
        flat = torch.empty(x.numel() + offset, dtype=dtype, device=DEV)
        flat[offset:] = x.flatten().to(DEV)
        return flat[offset:].view(shape)

    q, k = make(), make()
    qn, kn = _l2norm_qk(q, k)
    assert torch.equal(qn, l2norm(q)) and torch.equal(kn, l2norm(k))


def test_rule_follows_the_work():
    q = torch.empty(1, 1, 1, 128, device=DEV, dtype=torch.bfloat16)
    first = lambda b, t, hv: _l2norm_first(q, b, hv, 128, b * t)  # noqa: E731
    assert first(1, 1000, 16) and first(2, 4096, 16) and first(3, 4096, 16)
    assert not first(1, 100, 16) and not first(4, 4096, 16) and not first(53, 618, 16)
    with pytest.raises(ValueError):
        _lib.call("gdn_qk_l2norm_fwd", q.data_ptr(), None, q.data_ptr(), q.data_ptr(), 1, 128, 1, 1e-12, 0)


@pytest.mark.parametrize("b,t,h,hv,kd,vd", [(1, 1000, 16, 16, 128, 128), (2, 333, 3, 6, 64, 64), (1, 1, 1, 1, 128, 64),
                                            (3, 257, 2, 2, 64, 128), (1, 65, 4, 4, 128, 128)])
@pytest.mark.parametrize("offset", [0, 3])
@pytest.mark.parametrize("fused", [False, True])
def test_route_does_not_change_the_result(monkeypatch, b, t, h, hv, kd, vd, offset, fused):
    """Short of the long chains on a half-empty chip, the rows normalised ahead are the chunk kernels' own."""
    gen = torch.Generator().manual_seed(t)

    def make(d):  # contiguous, `offset` elements into its allocation; rows of very different sizes, one of zeros
        x = torch.randn(b, t, h, d, generator=gen) * (6 * torch.randn(b, t, h, 1, generator=gen)).exp()
        x[0, t // 2] = 0
        flat = torch.empty(x.numel() + offset, dtype=torch.bfloat16, device=DEV)
        flat[offset:] = x.bfloat16().flatten().to(DEV)
        return flat[offset:].view(b, t, h, d)

    q, k = make(kd), make(kd)
    v, gate = (torch.randn(b, t, hv, vd, generator=gen).bfloat16().to(DEV) for _ in range(2))
    g, beta = -torch.rand(b, t, hv, generator=gen).to(DEV), torch.rand(b, t, hv, generator=gen).to(DEV)
    outs, names, call = [], [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (names.append(name), call(name, *a))[1])
    for first in (False, True):
        monkeypatch.setattr(ops, "_l2norm_first", lambda *a, first=first: first)
        if fused:
            outs.append(ops.chunk_gated_delta_rule_gated_norm(q, k, v, g, beta, gate, torch.ones(vd, device=DEV),
                                                              output_final_state=True, use_qk_l2norm_in_kernel=True))
        else:
            outs.append(ops.chunk_gated_delta_rule(q, k, v, g, beta, output_final_state=True, use_qk_l2norm_in_kernel=True))
    assert names.count("gdn_qk_l2norm_chunk_fwd") == (offset == 0)
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    assert torch.isfinite(outs[0][0]).all()
