"""Calls that the attention module's own launches must leave to torch: where
torch refuses a call or has a subclass handle it, so does the module."""
import pytest
import torch
from torch.autograd import forward_ad

from magicube_amd import spattention

pytestmark = pytest.mark.gpu


def module(E=256, L=2752, bsz=2, bias=True):
    """A module, an input and mask arguments past the in-projection launch's
    128 tiles."""
    torch.manual_seed(E + L)
    mha = spattention.SpMultiheadAttention(E, E // 64, bias=bias).cuda().half().eval()
    cols, _, pairs, order, _ = spattention.static_random_mask_aligned(L // 8, L, 0.95, 16, seed=3)
    x = torch.randn(L, bsz, E, device="cuda").half()
    return mha, x, dict(need_weights=False, row_indices=order, row_offsets=pairs, column_indices=cols, vec_length=8)


@pytest.mark.parametrize("operand", ["input", "weight", "bias"])
def test_forward_mode_tangents_are_refused(operand):
    """torch's products into the plan's buffer refuse forward-mode AD; the
    module's own launch, which would drop the tangent, does not take its place."""
    mha, x, args = module()
    for p in mha.parameters():
        p.requires_grad_(False)
    with torch.no_grad(), forward_ad.dual_level():
        if operand == "input":
            x = forward_ad.make_dual(x, torch.ones_like(x))
        else:
            p = mha.in_proj_weight if operand == "weight" else mha.in_proj_bias
            dual = forward_ad.make_dual(p.detach(), torch.ones_like(p))
            name = "in_proj_weight" if operand == "weight" else "in_proj_bias"
            delattr(mha, name)
            setattr(mha, name, dual)
        with pytest.raises(NotImplementedError):
            mha(x, x, x, **args)
