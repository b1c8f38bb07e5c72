"""GPU parity of the int8 quadrant GEMM on grouped planes (w8a32_linear past
the small batches): every tile configuration and K slice count, at the edges
of tiles, token groups, k-blocks and the stage ring."""
import numpy as np
import pytest

from test_gpu_parity import assert_nonfinite_row, make, plant_inf, rel_l2, say

pytestmark = pytest.mark.gpu
F = np.float32


# tokens: one past a group of 16, below / at / past a 64-token tile column;
# K: shorter than the stage ring, a partial last k-block, an odd block count
@pytest.mark.parametrize("T,N,K", [(17, 200, 64), (33, 6300, 300), (63, 12288, 192), (64, 260, 6144), (65, 130, 4160),
                                   (145, 1000, 2048)])
def test_w8a32_planes_configs(lin, orc, T, N, K):
    """The four int8 planes of a token hold it to 2^-32 of its absmax and their
    products sum exactly, so an output carries the roundings of the fold and
    the scales alone: at most 8 x 2^-24 of the largest plane sum, well inside a
    relative L2 of 5e-7 of the float64 product (random signs: the sums are
    within a factor of ten of their terms' norm).  Integer sums make every
    configuration and slice count give the same bits.  A NaN row gives NaN, a
    row with infinities the oracle's NaN / +Inf / -Inf."""
    import torch
    say(f"w8a32 planes T={T} N={N} K={K}")
    rng = np.random.default_rng(T + N + K)
    x, w, s = make(rng, T, N, K)
    b = rng.standard_normal(N).astype(F)
    nan_row, inf_row = T - 1, T - 2
    x[nan_row, 5] = np.nan
    plant_inf(x, w, inf_row)
    fine = [r for r in range(T) if r not in (nan_row, inf_row)]
    want = (x[fine].astype(np.float64) @ w.astype(np.float64).T) * s + b
    want_inf = orc.w8a32_linear(x[[inf_row, inf_row]], w, s, bias=b)[0]
    lib = lin.load_library()
    W = lin.DeviceWeights.from_codes(w, s)
    xd, bd = torch.from_numpy(x).cuda(), torch.from_numpy(b).cuda()
    first = None
    try:
        for cfg, split in [(-1, 0), (3, 0), (4, 0), (6, 0), (6, 2), (6, 3), (6, 4), (7, 0), (7, 3), (-1, 8)]:
            say(f"  cfg={cfg} split={split}")
            assert lib.tl_gemm_i8_set_cfg(cfg) == 0 and lib.tl_gemm_i8_set_split(split) == 0
            y = torch.full((T, N), 7.0, device="cuda")
            for _ in range(2):                   # twice: the arrival counters are back at zero
                lin.w8a32_linear_dev(xd, W, y, bias=bd)
            got = y.cpu().numpy()
            if first is None:
                first = got
                assert rel_l2(got[fine], want) <= 5e-7
                assert np.isnan(got[nan_row]).all()
                assert_nonfinite_row(got[inf_row], want_inf)
            np.testing.assert_array_equal(got, first)
    finally:
        lib.tl_gemm_i8_set_cfg(-1)
        lib.tl_gemm_i8_set_split(0)
        W.close()
