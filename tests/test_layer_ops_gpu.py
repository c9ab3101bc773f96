"""The attention layer's ops (magicube_amd.sptrans) at the edges of their
kernels, bit for bit against the numpy restatements: ragged rows (empty, one
slot, one off a 16/32/64-slot group, longer than one staged chunk), widths
beside 64, divisors inside and outside the corrected-reciprocal range."""
import numpy as np
import pytest
import torch

from magicube_amd import formats, sptrans
from oracle import attention as oatt

pytestmark = pytest.mark.gpu

COUNTS = (0, 1, 15, 16, 17, 31, 33, 63, 64, 65, 127, 129, 0, 510, 514, 1030, 700, 3)
KEYS = 1100


def ragged_mask(align, seed, counts=COUNTS, keys=KEYS):
    rng = np.random.default_rng(seed)
    ro = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    cols = np.concatenate([np.sort(rng.permutation(keys)[:c]) for c in counts]).astype(np.int32)
    pairs, total = formats.align_rows(ro, align)
    aligned = formats.align_cols(ro, cols, pairs, total, shuffle=False)
    order = formats.sorted_rows(ro)
    return order, pairs, aligned


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def bits16(t):
    return t.cpu().numpy().view(np.uint16)


def packed(lanes, bits):
    return dev(formats.pack_lanes(lanes, bits).view(np.int32).reshape(lanes.shape[:-1] + (-1,)))


@pytest.mark.parametrize("pair", [(8, 8), (16, 8), (8, 4), (4, 4)])
@pytest.mark.parametrize("V", [8, 4, 2])
@pytest.mark.parametrize("n,divisor", [(64, 1152.0), (8, -3.7), (136, 2.0 ** 70), (520, 1e-3)])
def test_bspmm_edges(pair, V, n, divisor):
    lhs, rhs = pair
    batch = 2
    order, pairs, cols = ragged_mask(32 if rhs == 4 else 16, seed=V + n)
    rng = np.random.default_rng(n + lhs)
    # padding slots hold arbitrary lanes: no product may see them
    P = rng.integers(-(1 << (lhs - 1)), 1 << (lhs - 1), size=(batch, cols.size, V))
    v = rng.integers(-(1 << (rhs - 1)), 1 << (rhs - 1), size=(batch, KEYS, n))
    raw = np.stack([oatt.pack_p_reference(P[b], V, lhs) for b in range(batch)])
    fn = {(8, 8): sptrans.bspmm_8b, (16, 8): sptrans.bspmm_16b8b, (8, 4): sptrans.bspmm_8b4b,
          (4, 4): sptrans.bspmm_4b}[pair]
    print(f"bspmm {pair} V={V} n={n} divisor={divisor}", flush=True)
    out = fn(dev(order), dev(pairs), dev(cols), dev(raw.view(np.int32)), packed(v, rhs), V, lhs, rhs, divisor)
    torch.cuda.synchronize()
    with np.errstate(over="ignore"):
        exp = oatt.ref_bspmm(P, v, pairs, cols, V, divisor)
    assert np.array_equal(bits16(out), exp.view(np.uint16))
