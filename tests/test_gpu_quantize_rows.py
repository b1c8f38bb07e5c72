"""The row quantizer and the tile packer at the edges of their register-held
rows, against the oracle bit for bit."""
import numpy as np
import pytest

from test_gpu_parity import say

pytestmark = pytest.mark.gpu


# cols: below / at / past each register-held width, K % 16 tails of float4s, widths
# that stay on the general kernel (not a multiple of 4, above 8192)
@pytest.mark.parametrize("cols", [4, 20, 1028, 2044, 2048, 2052, 4096, 4108, 6144, 6156, 8192, 8196, 2046])
def test_quantize_rows_widths(lin, orc, dev, cols):
    import torch
    say(f"quantize rows cols={cols}")
    rng = np.random.default_rng(cols)
    x = rng.standard_normal((5, cols)).astype(np.float32)
    x[1] = 0.0
    x[2, cols - 1] = np.nan            # in the K % 16 tail where cols has one
    x[3, cols // 2] = np.inf
    x[4, :] = np.float32(1e-39) * rng.integers(-9, 10, cols)
    want_q, want_s = orc.quantize_rows(x)
    q = torch.empty((5, cols), dtype=torch.int8, device=dev)
    s = torch.empty(5, device=dev)
    lin.quantize_rows_dev(torch.from_numpy(x).to(dev), q, s)
    np.testing.assert_array_equal(q.cpu().numpy(), want_q)
    np.testing.assert_array_equal(s.cpu().numpy(), want_s)


# row groups of 16 rows, four to a work-group; a ragged last k-block
@pytest.mark.parametrize("rows,cols", [(1, 64), (17, 100), (64, 128), (65, 1000), (130, 6144)])
def test_pack_tiles_round_trip(lin, dev, rows, cols):
    import torch
    say(f"pack tiles {rows} x {cols}")
    rng = np.random.default_rng(rows + cols)
    w = rng.integers(-127, 128, (rows, cols), dtype=np.int8)
    W = lin.DeviceWeights.from_codes(torch.from_numpy(w).to(dev), torch.ones(rows, device=dev))
    x = torch.eye(cols, device=dev)[:min(cols, 200)].contiguous()
    y = torch.empty((x.shape[0], rows), device=dev)
    lin.w8a8_linear_f32_dev(x, W, y)   # unit rows: codes 127, scale 1 / 127
    W.close()
    np.testing.assert_allclose(y.cpu().numpy(), w[:, :x.shape[0]].T.astype(np.float32), rtol=2.0 ** -22)
