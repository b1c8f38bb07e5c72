"""GPU parity of the 16-bit wave-grid GEMM (w8a16_linear past the small batches):
every tile configuration and K slice count, at the edges of tiles, row groups,
k-blocks and the stage ring, for both activation and all output types."""
import numpy as np
import pytest

from test_gpu_parity import make, row_rel_l2, say

pytestmark = pytest.mark.gpu

CONFIGS = [(-1, 0), (4, 0), (5, 0), (6, 0), (7, 0), (8, 0), (6, 3), (7, 4), (8, 2)]


# rows: one past a row group, below / at / past a tile; N: a partial row group, not a
# multiple of the store width; K: shorter than the ring, a ragged last k-block
# (multiples of 8: other K take the generic kernel), an odd block count
@pytest.mark.parametrize("M,N,K,xt,yt", [(33, 200, 64, "f16", "f32"), (129, 1030, 72, "bf16", "bf16"),
                                         (255, 129, 200, "bf16", "f16"), (256, 12288, 192, "f16", "f16"),
                                         (257, 388, 1096, "bf16", "f32"), (321, 513, 4160, "f16", "bf16")])
def test_w8a16_configs(lin, dev, M, N, K, xt, yt):
    """Products of 16-bit x and int8 w are exact in fp32, so an output carries the
    fp32 roundings of its K-term sum, the scale and the bias: with random signs
    about sqrt(K) 2^-24 of the terms' norm, well inside a row-relative L2 of 1e-5;
    16-bit outputs add one rounding to nearest, at most half a unit of the last
    place of each value: 2^-8 of it for bf16, 2^-11 for fp16.  The rows of NaN and Inf stay in their own rows: every other
    row is as close, and columns of x past K (the next row in memory) add
    nothing."""
    import torch
    types = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
    rng = np.random.default_rng(M + N + K)
    x, w, s = make(rng, M, N, K)
    b = rng.standard_normal(N).astype(np.float32)
    xd = torch.from_numpy(x).to(dev).to(types[xt])
    xd[M - 2, :] = float("nan")
    xd[5, :] = float("inf")
    fine = [r for r in range(M) if r not in (5, M - 2)]
    want = (xd[fine].double().cpu().numpy() @ w.astype(np.float64).T) * s + b
    lib = lin.load_library()
    W = lin.DeviceWeights.from_codes(w, s)
    bd = torch.from_numpy(b).to(dev)
    bar = 1e-5 + {"f32": 0.0, "bf16": 2.0 ** -8, "f16": 2.0 ** -11}[yt]
    try:
        for cfg, split in CONFIGS:
            say(f"w8a16 wave grid M={M} N={N} K={K} {xt}->{yt} cfg={cfg} split={split}")
            assert lib.tl_gemm_b16_set_plan(cfg, split) == 0
            y = torch.full((M + 1, N), 7.0, device=dev, dtype=types[yt])
            for _ in range(2):                   # twice: the arrival counters are back at zero
                lin.w8a16_linear_dev(xd, W, y[:M], bias=bd)
            got = y.float().cpu().numpy()
            assert (got[M] == 7.0).all()
            e = row_rel_l2(got[fine], want)
            assert e.max() <= bar, (cfg, split, int(e.argmax()), float(e.max()))
            assert not np.isfinite(got[[5, M - 2]]).any()
    finally:
        lib.tl_gemm_b16_set_plan(-1, 0)
        W.close()
