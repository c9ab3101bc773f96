"""The layer's C entries on memory that the caller owns, filled beforehand and
with a guard past its end: every slot that an op promises is written (the rows'
products and the zeros between them), and nothing else is."""
import numpy as np
import pytest
import torch

from magicube_amd import _lib, attention, formats, sddmm, sptrans
from oracle import attention as oatt
from tests.test_layer_ops_gpu import COUNTS, KEYS, bits16, dev, packed, ragged_mask, scattered

pytestmark = pytest.mark.gpu

FILL, GUARD = 0xFF, 64          # 0xFFFF is a NaN in fp16


class Owned:
    """``size`` bytes of FILL followed by a guard."""

    def __init__(self, size):
        self.size = size
        self.buf = torch.full((size + GUARD,), FILL, dtype=torch.uint8, device="cuda")

    @property
    def ptr(self):
        return self.buf.data_ptr()

    def bytes(self):
        torch.cuda.synchronize()
        raw = self.buf.cpu().numpy()
        assert (raw[self.size:] == FILL).all(), "written past the end"
        return raw[:self.size]


def stream():
    return torch.cuda.current_stream().cuda_stream


def mask_of(layout, align, seed):
    order, pairs, cols = ragged_mask(align, seed)
    if layout == "scattered":
        pairs, cols = scattered(pairs, cols, seed)
    return order, pairs, cols


@pytest.mark.parametrize("layout", ["aligned", "scattered"])
@pytest.mark.parametrize("group", [8, 16, 32])
@pytest.mark.parametrize("slot_bits", [8, 16, 32, 64, 128])
def test_zero_gaps(layout, group, slot_bits):
    """Bytes outside every row's padded slots are 0; where rows lie in order,
    the rows' own bytes are not touched."""
    _, pairs, cols = mask_of(layout, 32, group)
    slots, batch = cols.size, 2
    stride = slots * slot_bits // 8
    out, ro = Owned(batch * stride), dev(pairs)
    _lib.check(_lib.lib().mc_attn_zero_gaps(batch, pairs.size // 2, ro.data_ptr(), slots, group, slot_bits, out.ptr,
                                            stride, stream()), "zero_gaps")
    owned = np.zeros(slots, bool)
    for s, e in pairs.reshape(-1, 2):
        owned[s:s + -(-(e - s) // group) * group] = True
    got = out.bytes().reshape(batch, slots, -1)
    assert not got[:, ~owned].any()
    if layout == "aligned":
        assert (got[:, owned] == FILL).all()


@pytest.mark.parametrize("layout", ["aligned", "scattered"])
@pytest.mark.parametrize("bits,k", [(8, 64), (4, 256), (8, 512)])
@pytest.mark.parametrize("V", [8, 4, 2])
def test_sddmm_f16(layout, bits, k, V):
    batch, divisor = 2, 324.0
    order, pairs, cols = mask_of(layout, 32 if bits == 4 else 16, V + k)
    rng = np.random.default_rng(k + V)
    lo, hi = -(1 << (bits - 1)), 1 << (bits - 1)
    lhs = rng.integers(lo, hi, size=(batch, len(COUNTS) * V, k))
    rhs = rng.integers(lo, hi, size=(batch, KEYS, k))
    ri, ro, ci, a, b = dev(order), dev(pairs), dev(cols), packed(lhs, bits), packed(rhs, bits)
    out = Owned(batch * cols.size * V * 2)
    _lib.check(_lib.lib().mc_sddmm_batched_f16(
        bits, batch, len(COUNTS), k, KEYS, ri.data_ptr(), ro.data_ptr(), ci.data_ptr(), cols.size, a.data_ptr(),
        lhs.shape[1] * k * bits // 8, b.data_ptr(), KEYS * k * bits // 8, divisor, out.ptr, cols.size * V, V,
        stream()), "sddmm_f16")
    exp = oatt.ref_bsddmm(lhs, rhs, pairs, cols, V, divisor)
    assert np.array_equal(out.bytes().view(np.uint16).reshape(batch, -1), exp.view(np.uint16))


@pytest.mark.parametrize("pair", [(8, 8), (16, 8), (8, 4), (4, 4)])
@pytest.mark.parametrize("V", [8, 4, 2])
@pytest.mark.parametrize("n", [64, 520])
def test_spmm_f16(pair, V, n):
    lhs, rhs = pair
    batch, divisor = 2, 1152.0
    order, pairs, cols = mask_of("scattered", 32, V + n)
    rng = np.random.default_rng(n + lhs)
    P = rng.integers(-(1 << (lhs - 1)), 1 << (lhs - 1), size=(batch, cols.size, V))
    v = rng.integers(-(1 << (rhs - 1)), 1 << (rhs - 1), size=(batch, KEYS, n))
    raw = np.stack([oatt.pack_p_reference(P[b], V, lhs) for b in range(batch)])
    ri, ro, ci, p, b = dev(order), dev(pairs), dev(cols), dev(raw.view(np.int32)), packed(v, rhs)
    m = len(COUNTS) * V
    out = Owned(batch * m * n * 2)
    _lib.check(_lib.lib().mc_spmm_batched_f16(
        lhs, rhs, batch, len(COUNTS), V, n, KEYS, ri.data_ptr(), ro.data_ptr(), ci.data_ptr(), p.data_ptr(),
        raw.shape[1], b.data_ptr(), KEYS * n * rhs // 8, divisor, out.ptr, m * n, stream()), "spmm_f16")
    exp = oatt.ref_bspmm(P, v, pairs, cols, V, divisor)
    assert np.array_equal(out.bytes().view(np.uint16).reshape(exp.shape), exp.view(np.uint16))


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("count", [8, 64, 4096, 4104, 100000])
def test_quantize_one(bits, count):
    x = torch.randn(count, device="cuda").half()
    out = Owned(count * bits // 8)
    _lib.check(_lib.lib().mc_attn_quantize(x.data_ptr(), count, 30.0, bits, attention.ROUND_TRUNC, out.ptr, stream()), "quantize")
    lanes = formats.unpack_lanes(out.bytes(), bits, count, signed=True)
    assert np.array_equal(lanes, oatt.quantize_ref(x.cpu().numpy(), 30.0, bits, 0).ravel())


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("row_len,stride,offset", [(96, 288, 0), (80, 84, 0), (48, 200, 4), (8, 24, 0), (40, 40, 1),
                                                   (64, 196, 0), (0, 0, 4), (0, 0, 0)])
def test_quantize_row_lengths(bits, row_len, stride, offset):
    """Jobs whose rows are no power of two, or start off 16 bytes."""
    rows = 701
    count = rows * row_len if row_len else 701 * 24 + (0 if bits == 4 else 3)
    x = torch.randn(rows * max(stride, 32) + offset, device="cuda").half()
    src = x[offset:].cpu().numpy()
    src = np.stack([src[i * stride:i * stride + row_len] for i in range(rows)]).ravel() if row_len else src[:count]
    out = Owned(count * bits // 8)
    job = attention._QuantJobC(x.data_ptr() + 2 * offset, count, 30.0, out.ptr, row_len, stride)
    jobs = torch.frombuffer(bytearray(bytes(job)), dtype=torch.uint8).cuda()
    _lib.check(_lib.lib().mc_attn_quantize_batched(jobs.data_ptr(), 1, bits, attention.ROUND_TRUNC, count, stream()),
               "quantize_batched")
    lanes = formats.unpack_lanes(out.bytes(), bits, count, signed=True)
    assert np.array_equal(lanes, oatt.quantize_ref(src, 30.0, bits, 0))


@pytest.fixture
def poisoned(monkeypatch):
    """torch.empty hands out memory full of FILL."""
    real = torch.empty

    def empty(*args, **kw):
        t = real(*args, **kw)
        if t.is_cuda and t.numel():
            t.view(torch.uint8).fill_(FILL)
        return t

    return lambda: monkeypatch.setattr(torch, "empty", empty)


@pytest.mark.parametrize("layout", ["aligned", "scattered"])
@pytest.mark.parametrize("V", [8, 4, 2])
@pytest.mark.parametrize("bits", [8, 4])
def test_ops_overwrite_what_they_allocate(layout, V, bits, poisoned):
    """bsddmm and the softmax leave 0 in every slot that no row owns."""
    batch = 2
    order, pairs, cols = mask_of(layout, 32, V)
    rng = np.random.default_rng(V)
    lo, hi = -(1 << (bits - 1)), 1 << (bits - 1)
    lhs = rng.integers(lo, hi, size=(batch, len(COUNTS) * V, 64))
    rhs = rng.integers(lo, hi, size=(batch, KEYS, 64))
    ri, ro, ci, a, b = dev(order), dev(pairs), dev(cols), packed(lhs, bits), packed(rhs, bits)
    poisoned()
    op = sptrans.bsddmm_8b if bits == 8 else sptrans.bsddmm_4b
    logits = op(ri, ro, ci, a, b, V, bits, 324.0)
    assert np.array_equal(bits16(logits), oatt.ref_bsddmm(lhs, rhs, pairs, cols, V, 324.0).view(np.uint16))
    real = np.zeros(cols.size, bool)
    for s, e in pairs.reshape(-1, 2):
        real[s:e] = True
    for p_bits in (16, 8, 4):
        attn = sptrans.q_bcsr_softmax(ri, ro, logits, 0.125, 7.0, V, batch, p_bits).cpu().numpy().view(np.uint8)
        for i in range(batch):
            assert not oatt.unpack_p_reference(attn[i], cols.size, V, p_bits)[~real].any()


@pytest.mark.parametrize("alignment", [8, 16])
@pytest.mark.parametrize("layout", [sddmm.OUT_REFERENCE, sddmm.OUT_VECTOR])
@pytest.mark.parametrize("k", [64, 576])
def test_masked_product_overwrites_its_output(alignment, layout, k, poisoned):
    rng = np.random.default_rng(alignment)
    V = 8
    ro = np.concatenate([[0], np.cumsum(COUNTS)]).astype(np.int32)
    cols = np.concatenate([np.sort(rng.permutation(KEYS)[:c]) for c in COUNTS]).astype(np.int32)
    mask = sddmm.DeviceMask.upload(formats.VectorCSR(len(COUNTS), KEYS, V, ro, cols), alignment)
    assert mask.covered == (alignment == 8)
    lhs = rng.integers(-128, 128, size=(len(COUNTS) * V, k))
    rhs = rng.integers(-128, 128, size=(KEYS, k))
    a, b = packed(lhs, 8), packed(rhs, 8)
    poisoned()
    out = mask.sddmm(8, a, b, k, layout=layout).cpu().numpy()
    slots = out.reshape(-1, V, 8).transpose(0, 2, 1).reshape(-1, V) if layout == sddmm.OUT_REFERENCE \
        else out.reshape(-1, V)
    exp = np.zeros_like(slots)
    for i in range(len(COUNTS)):
        s, e = int(mask.pairs[2 * i]), int(mask.pairs[2 * i + 1])
        exp[s:e] = rhs[mask.cols[s:e]] @ lhs[i * V:(i + 1) * V].T
    assert np.array_equal(slots, exp)


@pytest.mark.parametrize("bits", [16, 8, 4])
@pytest.mark.parametrize("V", [8, 4, 2])
def test_softmax_of_infinities_and_nan(bits, V):
    """A row whose sum is no number (a NaN or +inf logit, every logit -inf) has
    every P at the lower clamp, as fminf(fmaxf(NaN, lo), hi) gives; a -inf beside
    finite logits has P = 0 and changes nothing else.  Rows short and longer
    than the registers hold; the maxima ignore NaN."""
    scale = {16: 32767.0, 8: 127.0, 4: 7.0}[bits]
    low = -(1 << (bits - 1))
    order, pairs, cols = ragged_mask(32, seed=V)
    rng = np.random.default_rng(bits + V)
    logits = (rng.standard_normal((1, cols.size, V)) * 16).astype(np.float16)
    clean = logits.copy()
    rows = [i for i in range(len(COUNTS)) if COUNTS[i] > 0]
    kind = {}                                  # (row, v) -> how its P ends
    for n, i in enumerate(rows):
        s, e = int(pairs[2 * i]), int(pairs[2 * i + 1])
        v, at = n % V, s + (7 * n) % (e - s)
        k = ("nan", "inf", "all -inf", "-inf", "signalling nan")[n % 5]
        if k == "-inf" and e - s == 1:
            k = "nan"
        if k == "all -inf":
            logits[0, s:e, v] = -np.inf
        elif k == "signalling nan":
            logits.view(np.uint16)[0, at, v] = 0x7C01
        else:
            logits[0, at, v] = {"nan": np.nan, "inf": np.inf, "-inf": -np.inf}[k]
        if k == "-inf":
            clean[0, at, v] = np.float16(-60000)         # an exponential of 0 as well
        kind[i, v] = k
    print(f"softmax of non-finite logits bits={bits} V={V}", flush=True)
    attn = sptrans.q_bcsr_softmax(dev(order), dev(pairs), dev(logits.reshape(1, -1)), 0.125, scale, V, 1, bits)
    got = oatt.unpack_p_reference(attn.cpu().numpy().view(np.uint8)[0], cols.size, V, bits)
    exp = oatt.ref_softmax_f16(clean.reshape(1, -1), pairs, order, V, 0.125, scale, bits)[0]
    for (i, v), k in kind.items():
        s, e = int(pairs[2 * i]), int(pairs[2 * i + 1])
        if k != "-inf":
            exp[s:e, v] = low
        else:
            hit = np.isneginf(logits[0, s:e, v].astype(np.float32))
            assert (got[s:e, v][hit] == 0).all()
    # one step from rounding at a step's edge, as for finite logits
    assert np.abs(got - exp).max() <= 1
    assert (got != exp).sum() <= max(4, got.size // 100)
    for (i, v), k in kind.items():
        if k != "-inf":
            assert (got[pairs[2 * i]:pairs[2 * i + 1], v] == low).all()


@pytest.mark.parametrize("heads,samples,L", [(2, 3, 131), (10, 1, 129), (20, 2, 40)])
@pytest.mark.parametrize("qk_bits,range4", [(8, 0), (8, 1), (4, 0), (4, 1)])
@pytest.mark.parametrize("bias", [True, False])
def test_in_projection_entry(heads, samples, L, qk_bits, range4, bias):
    """Every E the entry takes (2 to 20 heads), ragged rows, without a bias: Q
    within an fp16 step of the 64-bit product, K and V within one quantization
    step, and the K and V columns of qkv and what follows each buffer as they were."""
    E = heads * 64
    gen = torch.Generator(device="cuda").manual_seed(E + L)
    rows = L * samples
    x = (torch.randn((rows, E), generator=gen, device="cuda") * 0.7).half()
    w = (torch.randn((3 * E, E), generator=gen, device="cuda") / E ** 0.5).half()
    b = (torch.randn(3 * E, generator=gen, device="cuda") * 0.2).half() if bias else None
    n = samples * heads
    qkv = Owned(rows * 3 * E * 2)
    kb = L * 64 * qk_bits // 8
    ks, vs = [Owned(kb) for _ in range(n)], [Owned(L * 64) for _ in range(n)]
    descs = []
    for i in range(n):
        d = attention._AttnMatrixC()
        d.L, d.m_vec, d.k, d.v = L, 0, ks[i].ptr, vs[i].ptr
        descs.append(bytes(d))
    mats = torch.frombuffer(bytearray(b"".join(descs)), dtype=torch.uint8).cuda()
    print(f"in-projection entry heads={heads} samples={samples} L={L} qk={qk_bits} bias={bias}", flush=True)
    _lib.check(_lib.lib().mc_attn_in_projection_f16(L, samples, heads, x.data_ptr(), w.data_ptr(),
                                                    b.data_ptr() if bias else None, 36.0, qk_bits, range4,
                                                    mats.data_ptr(), qkv.ptr, stream()), "in_projection")
    y = x.double() @ w.double().T
    y = (y + b.double() if bias else y).cpu().numpy()
    raw = qkv.bytes().view(np.uint16).reshape(rows, 3 * E)
    assert (raw[:, E:] == 0xFFFF).all()
    q = raw[:, :E].copy().view(np.float16).astype(np.float64)
    # half an fp16 step for the store, and the fp32 sum of at most 1280 products (sums below 8 here)
    assert (np.abs(q - y[:, :E]) <= np.maximum(np.abs(y[:, :E]), 2.0 ** -14) * 2.0 ** -11 + 1280 * 2.0 ** -24 * 8).all()
    wrong = total = 0
    for i in range(n):
        s, h = divmod(i, heads)
        for part, buf, bits, four in ((1, ks[i], qk_bits, qk_bits == 4), (2, vs[i], 8, range4)):
            lo, hi = (-8, 7) if four else (-128, 127)
            c = part * E + h * 64
            exp = np.trunc(np.clip(y[s::samples, c:c + 64].astype(np.float16).astype(np.float64) * 36.0, lo, hi))
            got = formats.unpack_lanes(buf.bytes(), bits, L * 64, signed=True).reshape(L, 64)
            d = np.abs(got - exp)
            assert d.max() <= 1
            wrong, total = wrong + int((d != 0).sum()), total + d.size
    # an fp16 y differs from the exact one's rounding at about 1 in 500 for the
    # longest sums, a truncation then at less than 1 in 10
    assert wrong <= total // 1000


@pytest.fixture
def guarded(monkeypatch):
    """Every tensor that torch.empty and torch.zeros allocate is followed by a guard."""
    made = []

    def guarded_fill(fill):
        def make(shape, dtype, device):
            n = int(np.prod(shape))
            size = n * dtype.itemsize
            buf = torch.full((size + 8 * GUARD,), FILL, dtype=torch.uint8, device=device)
            buf[:size] = fill
            made.append((buf, size))
            return buf[:size].view(dtype).view(shape)
        return make

    def check():
        torch.cuda.synchronize()
        assert made and all((buf[size:] == FILL).all() for buf, size in made), "written past the end"

    monkeypatch.setattr(torch, "empty", guarded_fill(FILL))
    monkeypatch.setattr(torch, "zeros", guarded_fill(0))
    yield check
    monkeypatch.undo()


@pytest.mark.parametrize("V", [8, 4, 2])
@pytest.mark.parametrize("last", [1, 9, 20, 36, 41])
def test_masks_that_end_inside_a_group(V, last, guarded):
    """The last row's slots are the mask's last (no padding up to a multiple of
    8, 16 or 32): the ops answer for these slots what they answer for the same
    mask with its padding, and store nothing past their outputs."""
    counts = COUNTS + (last,)
    order, pairs, cols = ragged_mask(32, seed=V + last, counts=counts)
    cut = int(pairs[-1])
    assert cut % 8 and cut + 31 >= cols.size
    short = cols[:cut]
    rng = np.random.default_rng(V)
    for k in (64, 576):                        # fp16 stored by the kernel; int32 and a second pass
        lhs = rng.integers(-8, 8, size=(2, len(counts) * V, k))
        rhs = rng.integers(-8, 8, size=(2, KEYS, k))
        ri, ro, a, b = dev(order), dev(pairs), packed(lhs, 8), packed(rhs, 8)
        whole = sptrans.bsddmm_8b(ri, ro, dev(cols), a, b, V, 8, 324.0)
        got = sptrans.bsddmm_8b(ri, ro, dev(short), a, b, V, 8, 324.0)
        one = sptrans.sddmm_8b(ri, ro, dev(short), a[0], b[0], V, 8, 324.0)
        assert got.is_contiguous() and torch.equal(got, whole[:, :cut * V]) and torch.equal(one, got[0])
    logits = whole
    for bits in (16, 8, 4):
        if cut * V * bits % 32:
            continue                           # refused: no whole number of words
        exp = sptrans.q_bcsr_softmax(ri, ro, logits, 0.125, 7.0, V, 2, bits)
        got = sptrans.q_bcsr_softmax(ri, ro, logits[:, :cut * V], 0.125, 7.0, V, 2, bits)
        assert got.is_contiguous() and torch.equal(got, exp[:, :cut * V * bits // 32])
    guarded()
