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


@pytest.mark.parametrize("E,L,bsz", [(128, 2752, 2), (128, 1848, 3), (256, 1368, 3), (256, 4096, 1)])
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("pair", [(8, 8), (8, 4), (4, 4)])
def test_module_attends_to_what_it_projected(E, L, bsz, bias, pair, monkeypatch):
    """The operands that one forward leaves behind are this input's (the input
    before it was another one), the output is the attention of these operands,
    and it is the layer's that torch's product and the quantize launch feed.
    There, an operand differs by a quantization step where the fp16 products
    round apart (at most 1 in 1000, checked above): a logit of 64 products of
    magnitude about 64 then moves by 64 / 10368, its P by less than 1 %, while
    operands of another matrix, input or moment would give another output altogether."""
    H = E // 64
    torch.manual_seed(E + L)
    mha = spattention.SpMultiheadAttention(E, H, bias=bias).cuda().half().eval()
    with torch.no_grad():
        # projections of std 1.8 for Q and K: attention that concentrates, so that P is not 0
        mha.in_proj_weight.normal_(std=E ** -0.5)
        mha.in_proj_weight[:2 * E] *= 1.8
        if bias:
            mha.in_proj_bias.normal_(std=0.1)
    # 4-bit Q and K (at the layer's scale of 36 within +-0.2) leave every row almost
    # uniform: P = trunc(32 p) is not 0 only in rows of fewer than 32 keys
    sparsity = 1.0 - 14 / L if pair[1] == 4 else 0.9
    cols, _, pairs, order, _ = spattention.static_random_mask_aligned(L // 8, L, sparsity, 32, seed=3)
    other, x = (torch.randn(L, bsz, E, device="cuda").half() for _ in range(2))
    args = dict(need_weights=False, row_indices=order, row_offsets=pairs, column_indices=cols, vec_length=8,
                lhs_pre=pair[0], rhs_pre=pair[1])
    ran = []
    project = spattention._Plan.project
    monkeypatch.setattr(spattention._Plan, "project", lambda *a: ran.append(project(*a)) or ran[-1])
    print(f"module E={E} L={L} bsz={bsz} bias={bias} pair={pair}", flush=True)
    with torch.no_grad():
        mha(other, other, other, **args)
        out, _ = mha(x, x, x, **args)
        assert ran == [True, True]
        plan = next(iter(mha._plans.values()))
        plan.batch.attend()
        assert torch.equal(out, torch.nn.functional.linear(plan.o, mha.out_proj.weight, mha.out_proj.bias))
        y = x.double() @ mha.in_proj_weight.double().T
        y = (y + mha.in_proj_bias.double() if bias else y).view(L, bsz, 3, H, 64)
        assert _close(plan.qkv.view(L, bsz, 3, H, 64)[:, :, 0], y[:, :, 0])
        lo, hi = (-8, 7) if pair[1] == 4 else (-128, 127)
        for i, m in enumerate(plan.batch.mats):
            b, h = divmod(i, H)
            for part, buf, bits in ((1, m.kq, plan.rhs_pre), (2, m.vq, 8)):
                exp = (y[:, b, part, h].half().double() * 36.0).clamp(lo, hi).trunc().to(torch.int32)
                if bits == 4:
                    got = torch.stack([buf & 15, buf >> 4], dim=1).view(L, 64).to(torch.int32)
                    got = got - ((got >> 3) << 4)
                else:
                    got = buf.view(torch.int8).view(L, 64).to(torch.int32)
                assert int((got - exp).abs().max()) <= 1
        monkeypatch.setattr(spattention._Plan, "project", lambda *a: False)
        ref, _ = mha(x, x, x, **args)
        scale = float(ref.float().norm())
        assert scale > 0 and float((out.float() - ref.float()).norm()) <= 0.05 * scale
