"""The SpMM tiles with four dwords of B per lane, exact against a dense product
in float64: the default of wide products with long rows (short ones take a
narrower tile), and both such tiles by their number, for two MFMA row tiles too."""
import numpy as np
import pytest
import torch

from magicube_amd import formats, spmm, synthetic

pytestmark = pytest.mark.gpu

K = 400


def product(pair, V, signed, m_vec, counts, widths, config, seed):
    lhs, rhs = pair
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    rng = np.random.default_rng(seed)
    cols = np.concatenate([np.sort(rng.permutation(K)[:c]) for c in counts]).astype(np.int32)
    csr = formats.VectorCSR(m_vec, K, V, offsets, cols)
    a = synthetic.random_lanes(csr.nnz_vec * V, lhs, signed, 1)
    dev = spmm.DeviceSpmm.upload(formats.prepare_spmm(csr, formats.pack_lanes(a, lhs), lhs, rhs))
    dense = np.zeros((m_vec, V, K))
    rows = np.repeat(np.arange(m_vec), counts)
    for v in range(V):
        dense[rows, v, cols] = a.reshape(-1, V)[:, v]
    dense = torch.from_numpy(dense.reshape(-1, K)).cuda()
    for n in widths:
        if n % (32 // rhs):
            continue
        b = synthetic.random_lanes(K * n, rhs, signed, n)
        rhs_t = torch.from_numpy(formats.pack_lanes(b, rhs).view(np.int32)).cuda()
        # a canary after the output's last row
        buf = torch.full((m_vec * V * n + 64,), 7, dtype=torch.int32, device="cuda")
        out = buf[:m_vec * V * n].view(-1, n)
        print(f"spmm {pair} V={V} signed={signed} n={n} config={config}", flush=True)
        dev.matmul(rhs_t, n, out=out, sign=spmm.SIGNED if signed else spmm.UNSIGNED, config=config)
        torch.cuda.synchronize()
        exact = dense @ torch.from_numpy(b.reshape(K, n).astype(np.float64)).cuda()
        assert torch.equal(out, exact.to(torch.int64).to(torch.int32))
        assert (buf[m_vec * V * n:] == 7).all()
    return csr


@pytest.mark.parametrize("pair,V", [((8, 8), 8), ((8, 8), 2), ((16, 8), 4), ((12, 8), 4), ((16, 16), 4)])
@pytest.mark.parametrize("signed", [True, False])
def test_default_tile_of_long_rows(pair, V, signed, mclib):
    """Rows of 330 slots on average, some empty or full, at widths beside the
    lane, tile and workgroup edges."""
    m_vec = 1024
    counts = np.random.default_rng(V).integers(290, 380, size=m_vec)
    counts[:5] = (0, K, 65, 1, 0)
    widths = (132, 136, 256, 260, 264, 508, 512, 772, 776, 1028)
    product(pair, V, signed, m_vec, counts, widths, None, V)
    tiles = {n: mclib.mc_spmm_default_config(*pair, 0 if signed else 1, m_vec, V, n, K, int(counts.mean())) for n in widths}
    assert tiles[772] == tiles[1028] == 24


@pytest.mark.parametrize("config", [24, 25])
@pytest.mark.parametrize("pair,V", [((8, 8), 8), ((16, 8), 8), ((16, 8), 2), ((12, 8), 8), ((16, 16), 8), ((16, 16), 2)])
@pytest.mark.parametrize("signed", [True, False])
def test_four_dword_tiles(config, pair, V, signed):
    """V = 8 with several digit planes is two MFMA row tiles: the columns of two
    rows at a time are recombined and pass through LDS."""
    counts = np.array([0, K, 65, 1, 64, 63, 130, 0, 399, 17] * 3)
    product(pair, V, signed, len(counts), counts, (272, 512, 528, 1040), config, config + V)
