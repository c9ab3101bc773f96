"""The default SpMM tile for wide products (four dwords of B per lane): every
pair and signedness with one and two MFMA row tiles, widths around the lane,
tile and workgroup edges (a row's last lane then repeats its neighbour's
columns), rows empty, short and longer than one staged chunk.  Exact against a
dense product in float64."""
import numpy as np
import pytest
import torch

from magicube_amd import formats, spmm, synthetic

pytestmark = pytest.mark.gpu

PAIRS = [(8, 8), (16, 8), (12, 8), (16, 16), (8, 4)]


@pytest.mark.parametrize("pair", PAIRS)
@pytest.mark.parametrize("V", [8, 4, 2])
@pytest.mark.parametrize("signed", [True, False])
def test_widths(pair, V, signed):
    lhs, rhs = pair
    m_vec, K = 1024, 72
    rng = np.random.default_rng(V + lhs + rhs)
    counts = rng.integers(0, 24, size=m_vec)
    counts[:4] = (0, K, 65, 1)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    cols = np.concatenate([np.sort(rng.permutation(K)[:c]) for c in counts]).astype(np.int32)
    csr = formats.VectorCSR(m_vec, K, V, offsets, cols)
    a = synthetic.random_lanes(csr.nnz_vec * V, lhs, signed, 1)
    dev = spmm.DeviceSpmm.upload(formats.prepare_spmm(csr, formats.pack_lanes(a, lhs), lhs, rhs))
    dense = np.zeros((m_vec, V, K))
    rows = np.repeat(np.arange(m_vec), counts)
    for v in range(V):
        dense[rows, v, cols] = a.reshape(-1, V)[:, v]
    dense = torch.from_numpy(dense.reshape(-1, K)).cuda()
    for n in (136, 256, 260, 264, 508, 512, 516, 776, 1028):
        if n % (32 // rhs):
            continue
        b = synthetic.random_lanes(K * n, rhs, signed, n)
        rhs_t = torch.from_numpy(formats.pack_lanes(b, rhs).view(np.int32)).cuda()
        # a canary after the output's last row: nothing is stored past a row's end
        buf = torch.full((m_vec * V * n + 64,), 7, dtype=torch.int32, device="cuda")
        out = buf[:m_vec * V * n].view(-1, n)
        print(f"spmm {pair} V={V} signed={signed} n={n}", flush=True)
        dev.matmul(rhs_t, n, out=out, sign=spmm.SIGNED if signed else spmm.UNSIGNED)
        torch.cuda.synchronize()
        exact = dense @ torch.from_numpy(b.reshape(K, n).astype(np.float64)).cuda()
        assert torch.equal(out, exact.to(torch.int64).to(torch.int32))
        assert (buf[m_vec * V * n:] == 7).all()


def test_long_rows():
    """Rows of several staged chunks (1024 slots) at a ragged width."""
    m_vec, K, V, n = 1024, 3000, 2, 1028
    csr = synthetic.poisson_block_mask(m_vec * V, K, V, 0.3, 5)
    a = synthetic.random_lanes(csr.nnz_vec * V, 8, True, 1)
    b = synthetic.random_lanes(K * n, 8, True, 2)
    dev = spmm.DeviceSpmm.upload(formats.prepare_spmm(csr, formats.pack_lanes(a, 8), 8, 8))
    out = dev.matmul(torch.from_numpy(formats.pack_lanes(b, 8).view(np.int32)).cuda(), n)
    dense = np.zeros((m_vec, V, K))
    rows = np.repeat(np.arange(m_vec), np.diff(csr.row_offsets))
    for v in range(V):
        dense[rows, v, csr.col_indices] = a.reshape(-1, V)[:, v]
    exact = torch.from_numpy(dense.reshape(-1, K)).cuda() @ torch.from_numpy(b.reshape(K, n).astype(np.float64)).cuda()
    assert torch.equal(out, exact.to(torch.int64).to(torch.int32))
