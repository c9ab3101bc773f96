"""Calls that the attention module's own launches must leave to torch: where
torch refuses a call or has a subclass handle it, so does the module."""
import pytest
import torch
import torch.nn.functional as F
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


@pytest.mark.parametrize("residual", [False, True])
def test_layernorm_keeps_forward_mode_tangents(residual):
    """torch's LayerNorm, which has them, runs inside a forward-mode level."""
    ln = spattention.FusedLayerNorm(256).cuda().half()
    x, t, r = (torch.randn(40, 256, device="cuda").half() for _ in range(3))
    with torch.no_grad(), forward_ad.dual_level():
        d = forward_ad.make_dual(x, t)
        got = forward_ad.unpack_dual(ln(d, r) if residual else ln(d)).tangent
        exp = forward_ad.unpack_dual(F.layer_norm(d + r if residual else d, (256,), ln.weight, ln.bias, ln.eps)).tangent
    assert got is not None and torch.equal(got, exp)


class Recorded(torch.Tensor):
    """A tensor subclass that sees every torch function it passes through."""
    seen = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.seen.append(getattr(func, "__name__", str(func)))
        return super().__torch_function__(func, types, args, kwargs or {})


@pytest.mark.parametrize("operand", ["input", "weight"])
def test_subclass_operands_reach_torch(operand):
    """The in-projection of a tensor subclass is torch's addmm, which the subclass handles."""
    mha, x, args = module()
    if operand == "input":
        x = x.as_subclass(Recorded)
    else:
        w = mha.in_proj_weight.detach().as_subclass(Recorded)
        del mha.in_proj_weight
        mha.in_proj_weight = w
    Recorded.seen.clear()
    with torch.no_grad():
        mha(x, x, x, **args)
    assert "addmm" in Recorded.seen
