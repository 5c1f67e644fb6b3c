"""Calls that find their launch arguments kept from an earlier call of the same shapes,
strides and options, against calls that build them."""
import pytest
import torch

from ascend_rsfa import flash_attention_forward as F
from oracle import attention as oracle

pytestmark = pytest.mark.gpu


def test_kept_plan_checks_addresses_and_options():
    q, k, v = (t.cuda() for t in oracle.make_inputs(2, 3, 200, 64, seed=1))
    want = {c: F.forward(q, k, v, c, 0.2) for c in (False, True)}
    for c in (False, True):
        o, lse = F.forward(q, k, v, c, 0.2, return_lse=True)  # the kept plan, with a logsumexp
        assert torch.equal(o, want[c])
        assert torch.equal(F.forward(q, k, v, c, 0.2, out=torch.empty_like(q)), want[c])
        # the same shape and strides two bytes past a 16-byte boundary
        flat = torch.empty(q.numel() + 1, dtype=q.dtype, device="cuda")
        shifted = flat[1:].view(q.shape).copy_(q)
        assert torch.equal(F.forward(shifted, k, v, c, 0.2), want[c])
        with pytest.raises(ValueError):
            F.forward(q, k, v[:, :, :199], c, 0.2)
        with pytest.raises(TypeError):
            F.forward(q, k, v.float(), c, 0.2)
        with pytest.raises(ValueError):
            F.forward(q, k, v.cpu(), c, 0.2)
    # split and fused calls of one shape keep different plans
    split = F.forward(q, k, v, True, 0.2, 128, 64, split=True)
    assert torch.allclose(split, F.forward(q, k, v, True, 0.2, 128, 64), atol=1e-3, rtol=1e-3)


@pytest.mark.parametrize("scale", [0.2, torch.tensor(0.2), 1, 1e300])
def test_scale_types(scale):
    q, k, v = (t.cuda() for t in oracle.make_inputs(1, 1, 64, 64, seed=2))
    q.zero_()  # scores 0: any finite scale gives the mean of V
    o = F.forward(q, k, v, False, scale)
    if float(scale) < 3e38:
        assert torch.allclose(o[0, 0], v[0, 0].float().mean(0).half().expand(64, 64), atol=2e-3)
