"""The quantizing in-projection at the edges of its tiles, against 64-bit products."""
import pytest
import torch

from magicube_amd import spattention

pytestmark = pytest.mark.gpu


def _close(got, exact):
    """Half an fp16 step for the store, and the fp32 sum of at most 1024 terms
    (here of magnitude below 8): 1024 * 2^-24 * 8."""
    step = torch.maximum(exact.abs(), torch.tensor(2.0 ** -14, device=exact.device)) * 2.0 ** -11
    return bool(((got.double() - exact).abs() <= step + 2.0 ** -11).all())


@pytest.mark.parametrize("L,bsz", [(1368, 3), (4096, 1), (600, 9)])
@pytest.mark.parametrize("pair", [(8, 8), (8, 4), (4, 4)])
def test_in_projection_quantizes_as_the_quantize_launch(L, bsz, pair):
    """Every K and V is trunc(clamp(36 y)) of an fp16 y within one step of the
    64-bit product, so the two quantized values differ by at most one where 36
    steps are below one."""
    E, H = 256, 4
    torch.manual_seed(L)
    mha = spattention.SpMultiheadAttention(E, H).cuda().half().eval()
    with torch.no_grad():
        mha.in_proj_bias.normal_(std=0.2)
    align = 32 if pair[1] == 4 else 16
    cols, _, pairs, order, _ = spattention.static_random_mask_aligned(L // 8, L, 0.9, align, seed=3)
    x = (torch.randn(L, bsz, E, device="cuda") * 0.7).half()
    print(f"in-projection L={L} bsz={bsz} pair={pair}", flush=True)
    with torch.no_grad():
        out, _ = mha(x, x, x, need_weights=False, row_indices=order, row_offsets=pairs, column_indices=cols,
                     vec_length=8, lhs_pre=pair[0], rhs_pre=pair[1])
        plan = next(iter(mha._plans.values()))
        assert plan.project(x.view(L * bsz, E), mha.in_proj_weight, mha.in_proj_bias)     # the launch under test ran
        y = (x.double() @ mha.in_proj_weight.double().T + mha.in_proj_bias.double()).view(L, bsz, 3, H, 64)
        torch.cuda.synchronize()
        assert _close(plan.qkv.view(L, bsz, 3, H, 64)[:, :, 0], y[:, :, 0])
        lo, hi = (-8, 7) if pair[1] == 4 else (-128, 127)
        wrong = total = 0
        for i, m in enumerate(plan.batch.mats):
            b, h = divmod(i, H)
            for part, buf, bits in ((1, m.kq, plan.rhs_pre), (2, m.vq, 8)):
                exp = (y[:, b, part, h].half().double() * 36.0).clamp(lo, hi).trunc().to(torch.int32)
                if bits == 4:
                    got = torch.stack([buf & 15, buf >> 4], dim=1).view(L, 64).to(torch.int32)
                    got = got - ((got >> 3) << 4)
                else:
                    got = buf.view(torch.int8).view(L, 64).to(torch.int32)
                d = (got - exp).abs()
                assert int(d.max()) <= 1
                wrong, total = wrong + int((d != 0).sum()), total + d.numel()
        # an fp16 y differs from the exact one's rounding at about 1 in 2000, a
        # truncation then at less than 1 in 10
        assert wrong <= total // 1000
    assert torch.isfinite(out).all()
