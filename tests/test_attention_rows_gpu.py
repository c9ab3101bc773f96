"""The fused attention kernel at the row lengths where its paths change: empty
and one-slot rows, off by one around 16 and 64 slots, around what its LDS copy
holds (384 slots at V = 8, 768 below), around what it keeps in all (512 and
896), and beyond.  O of the production kernel and S, P and P V of the debug
one equal the one-op-per-launch pipeline bit for bit."""
import numpy as np
import pytest
import torch

from magicube_amd import attention, formats, synthetic

pytestmark = pytest.mark.gpu

EDGES = {8: (383, 384, 385, 448, 449, 511, 512, 513, 577, 900),
         4: (767, 768, 769, 832, 833, 895, 896, 897, 961, 1030)}


@pytest.mark.parametrize("p_mode", [attention.P_ROW_SCALED, attention.P_REFERENCE, attention.P_REFERENCE_4BIT])
@pytest.mark.parametrize("qk_bits,v_bits", [(8, 8), (4, 8), (4, 4)])
@pytest.mark.parametrize("V", [8, 4, 2])
def test_row_lengths(V, qk_bits, v_bits, p_mode):
    counts = (0, 1, 15, 16, 17, 63, 64, 65, 127, 128, 129) + EDGES[8 if V == 8 else 4]
    L = max(1200 // V * V, len(counts) * V)
    counts = counts + (40,) * (L // V - len(counts))
    rng = np.random.default_rng(V + qk_bits)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    cols = np.concatenate([rng.permutation(L)[:n] for n in counts]).astype(np.int32)    # any order in a row
    mask = formats.VectorCSR(L // V, L, V, offsets, cols)
    q, k, v = (torch.from_numpy(x).cuda() for x in synthetic.attention_inputs(L, V))
    mats = [attention.AttentionMatrix(q * 2, k, v, mask)]
    # a reference scale above 127 needs the clamp
    for p_scale in ((127.0,) if p_mode == attention.P_ROW_SCALED else (32.0, 1000.0)):
        kw = dict(qk_bits=qk_bits, v_bits=v_bits, V=V, p_mode=p_mode, p_scale=p_scale, v_range4=v_bits == 4)
        b = attention.AttentionBatch(mats, debug=True, **kw)
        print(f"rows V={V} qk={qk_bits} v={v_bits} p_mode={p_mode} p_scale={p_scale}", flush=True)
        b.forward_plain()
        torch.cuda.synchronize()
        d = b.mats[0]
        plain = [d.work["p"].clone(), d.work["o_int"].clone(), d.o.clone()]
        b.forward()
        torch.cuda.synchronize()
        assert torch.equal(plain[0][:d.aligned_num * V], d.p_out[:d.aligned_num * V]), "P"
        assert torch.equal(plain[1], d.o_int), "P V"
        assert torch.equal(plain[2].view(torch.int32), d.o.view(torch.int32)), "O"
        fast = attention.AttentionBatch(mats, scales=[d.scales], **kw)
        out = fast.forward()[0]
        torch.cuda.synchronize()
        assert torch.equal(plain[2].view(torch.int32), out.view(torch.int32)), "O of the production kernel"
