"""GPU: q and k normalised in one launch are bitwise the two separate launches, at the edges of a block's rows,
for unaligned rows and for the head dims and types without a vector path; and the rule that picks that route."""
import pytest
import torch

from sorernn_amd import _lib, l2norm
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
