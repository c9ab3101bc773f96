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


def scattered(pairs, cols, seed):
    """The same rows laid out in another order, with gaps before, between and after them."""
    rng = np.random.default_rng(seed)
    rows = pairs.size // 2
    where, at = np.zeros_like(pairs), 32
    out = np.full(2 * cols.size + 32 * (rows + 2), -1, np.int32)
    for i in rng.permutation(rows):
        n = int(pairs[2 * i + 1] - pairs[2 * i])
        where[2 * i:2 * i + 2] = at, at + n
        out[at:at + n] = cols[pairs[2 * i]:pairs[2 * i + 1]]
        at += (n + 31) // 32 * 32 + 32 * int(rng.integers(0, 2))
    return where, out[:at + 32]


@pytest.mark.parametrize("bits,k", [(8, 64), (4, 64), (8, 192), (4, 512), (8, 576)])
@pytest.mark.parametrize("V", [8, 4, 2])
@pytest.mark.parametrize("layout", ["aligned", "scattered"])
def test_bsddmm_edges(bits, k, V, layout):
    batch, divisor = 2, 1296.0 if k == 64 else 7.3
    order, pairs, cols = ragged_mask(32 if bits == 4 else 16, seed=V + k)
    if layout == "scattered":
        pairs, cols = scattered(pairs, cols, seed=k)
    rng = np.random.default_rng(k + V)
    lo, hi = -(1 << (bits - 1)), 1 << (bits - 1)
    lhs = rng.integers(lo, hi, size=(batch, len(COUNTS) * V, k))
    rhs = rng.integers(lo, hi, size=(batch, KEYS, k))
    # memory that the op must overwrite or zero
    torch.full((batch * cols.size * V,), float("nan"), dtype=torch.float16, device="cuda")
    fn = sptrans.bsddmm_8b if bits == 8 else sptrans.bsddmm_4b
    print(f"bsddmm bits={bits} k={k} V={V} {layout}", flush=True)
    got = fn(dev(order), dev(pairs), dev(cols), packed(lhs, bits), packed(rhs, bits), V, bits, divisor)
    torch.cuda.synchronize()
    exp = oatt.ref_bsddmm(lhs, rhs, pairs, cols, V, divisor)
    assert np.array_equal(bits16(got), exp.view(np.uint16))


@pytest.mark.parametrize("bits", [16, 8, 4])
@pytest.mark.parametrize("V", [8, 4, 2])
@pytest.mark.parametrize("layout", ["aligned", "scattered"])
def test_softmax_edges(bits, V, layout):
    """P against the restatement with the softmax's own exponentials: rows
    short, longer than the registers hold (1030 slots), and with sums outside
    the corrected reciprocal's range (rows v >= 1 far below their maximum's
    start at 0; an infinite or NaN logit)."""
    batch, scale = 2, {16: 32767.0, 8: 127.0, 4: 7.0}[bits]
    order, pairs, cols = ragged_mask(32, seed=V + bits)
    if layout == "scattered":
        pairs, cols = scattered(pairs, cols, seed=V)
    rng = np.random.default_rng(bits * V)
    logits = (rng.standard_normal((batch, cols.size, V)) * 16).astype(np.float16)
    low = pairs[2 * 9]                       # the row of 65 slots: exponentials near the smallest float
    logits[1, low:low + 65] = (-80 * 8 + rng.standard_normal((65, V))).astype(np.float16)
    real = np.zeros(cols.size, bool)
    for i in range(pairs.size // 2):
        real[pairs[2 * i]:pairs[2 * i + 1]] = True
    logits[:, ~real] = np.float16("nan")     # never read
    logits = logits.reshape(batch, -1)
    print(f"softmax bits={bits} V={V} {layout}", flush=True)
    attn = sptrans.q_bcsr_softmax(dev(order), dev(pairs), dev(logits), 0.125, scale, V, batch, bits)
    torch.cuda.synchronize()
    exp = oatt.ref_softmax_f16(logits, pairs, order, V, 0.125, scale, bits)
    raw = attn.cpu().numpy().view(np.uint8)
    for b in range(batch):
        got = oatt.unpack_p_reference(raw[b], cols.size, V, bits)
        # one step from rounding at a step's edge; 16-bit steps are as fine as
        # the exponential's own error (a few ulp of 2^-23 times 2^15)
        assert np.abs(got - exp[b]).max() <= 1
        assert (got != exp[b]).sum() <= max(4, got.size // 100)
        assert (got[~real] == 0).all()


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("rows", [(5, 64, 8), (3, 40, 24), (1, 7, 8), (2, 9, 40)])
def test_quantize_matches_the_restatement(bits, rows):
    """One tensor, contiguous or not, odd row counts, edges of a thread's and a block's share."""
    b, n, d = rows
    x = torch.randn((b, n * 61, d), device="cuda").half()
    for t in (x, x.transpose(0, 1), x[:, 1:]):
        if (d * bits) % 32:
            continue
        got = sptrans.bquantization(t, bits, 30.0)
        exp = oatt.quantize_ref(t.contiguous().cpu().numpy(), 30.0, bits, 0)
        lanes = formats.unpack_lanes(got.cpu().numpy().view(np.uint8), bits, exp.size, signed=True)
        assert np.array_equal(lanes.reshape(exp.shape), exp)


@pytest.mark.parametrize("alignment", [8, 16])
@pytest.mark.parametrize("layout", [0, 1])
def test_sddmm_output_has_no_stale_slots(alignment, layout):
    """A product into memory full of another value leaves 0 in every padding slot."""
    from magicube_amd import sddmm
    rng = np.random.default_rng(alignment)
    ro = np.concatenate([[0], np.cumsum(COUNTS)]).astype(np.int32)
    cols = np.concatenate([np.sort(rng.permutation(KEYS)[:c]) for c in COUNTS]).astype(np.int32)
    for V, counts in ((8, COUNTS), (2, COUNTS), (4, (0, 0))):
        csr = formats.VectorCSR(len(counts), KEYS, V, ro if counts is COUNTS else np.zeros(3, np.int32),
                                cols if counts is COUNTS else cols[:0])
        mask = sddmm.DeviceMask.upload(csr, alignment)
        lhs = rng.integers(-128, 128, size=(len(counts) * V, 64))
        rhs = rng.integers(-128, 128, size=(KEYS, 64))
        junk = torch.full((mask.output_size(),), 9, dtype=torch.int32, device="cuda")
        del junk        # the caching allocator hands this block to the output
        out = mask.sddmm(8, packed(lhs, 8), packed(rhs, 8), 64, layout=layout).cpu().numpy()
        slots = out.reshape(-1, V, 8).transpose(0, 2, 1).reshape(-1, V) if layout == 0 else out.reshape(-1, V)
        exp = np.zeros_like(slots)
        for i in range(len(counts)):
            s, e = int(mask.pairs[2 * i]), int(mask.pairs[2 * i + 1])
            exp[s:e] = rhs[mask.cols[s:e]] @ lhs[i * V:(i + 1) * V].T
        assert np.array_equal(slots, exp)
