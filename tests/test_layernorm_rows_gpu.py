"""mc_layernorm_f16 at the edges of its rows per wave (two of 1024 and 512
columns, four of 256) and with a weight and bias that start on any half:
within the bound of test_layernorm_gpu.py, nothing stored past the last row."""
import pytest
import torch

from tests.test_layernorm_gpu import _reference, _run, _within_one_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols", [256, 512, 1024])
@pytest.mark.parametrize("rows", [1, 2, 3, 4, 5, 15, 16, 17, 33])
def test_layernorm_row_edges(cols, rows):
    g = torch.Generator(device="cuda").manual_seed(cols + rows)
    # activations 8 bytes into their buffers, weight and bias one half into theirs
    x = (torch.randn(rows * cols + 4, device="cuda", generator=g) * 3 + 1).half()[4:].view(rows, cols)
    res = (torch.randn(rows * cols + 4, device="cuda", generator=g) * 2).half()[4:].view(rows, cols)
    w = (torch.rand(cols + 1, device="cuda", generator=g) + 0.5).half()[1:]
    b = torch.randn(cols + 1, device="cuda", generator=g).half()[1:]
    buf = torch.full((rows * cols + 68,), 7.0, dtype=torch.float16, device="cuda")
    out = buf[4:4 + rows * cols].view(rows, cols)
    for r in (None, res):
        print(f"layernorm cols={cols} rows={rows} residual={r is not None}", flush=True)
        _within_one_step(_run(x, r, w, b, 1e-5, out=out), _reference(x, r, w, b, 1e-5))
        assert (buf[:4] == 7).all() and (buf[4 + rows * cols:] == 7).all()
