"""A GEMM's kernel, configuration and K slices are chosen once a call: work-space
is sized for the choice that the launch runs, also when another thread changes a
tuning override between the two."""
import ctypes

import pytest

from test_gpu_parity import say

A_I8, A_BF16 = 0, 1
OUT_F32, OUT_I32 = 0, 3
vp, i32 = ctypes.c_void_p, ctypes.c_int


class GemmLaunch(ctypes.Structure):          # csrc/tl_kernels.h
    _fields_ = [("amode", i32), ("A", vp), ("lda", i32), ("Bt", vp), ("ws", vp), ("xs", vp), ("bias", vp), ("Y", vp),
                ("ldy", i32), ("M", i32), ("N", i32), ("K", i32), ("ep", i32), ("out", i32), ("part", vp), ("cnt", vp),
                ("zero_tile", vp), ("xe", vp), ("xraw", vp), ("ldxr", i32), ("planes_grouped", ctypes.c_bool), ("whole", ctypes.c_bool),
                ("kernel", i32), ("cfg", i32), ("split", i32)]


def resolve(lib, L):
    part, counters = ctypes.c_size_t(), ctypes.c_size_t()
    lib.tlk_gemm_resolve(ctypes.byref(L), ctypes.byref(part), ctypes.byref(counters))
    return part.value, counters.value


def override(lib, amode, split):
    if amode == A_I8:
        assert lib.tl_gemm_i8_set_split(split) == 0
    else:
        assert lib.tl_gemm_b16_set_plan(7 if split else -1, split) == 0


# both on 64 x 128 tiles: int8 configuration 1, 16-bit configuration 7
@pytest.mark.parametrize("amode,kernel,cfg", [(A_I8, 1, 1), (A_BF16, 2, 7)])
def test_unresolved_is_refused_and_sizes_fit_the_choice(lin, amode, kernel, cfg):
    lib = lin.load_library()
    zeros = (ctypes.c_uint8 * 1024)()
    L = GemmLaunch(amode=amode, A=ctypes.addressof(zeros) & ~15, lda=4096, M=100, N=256, K=4096, kernel=-1, split=1,
                   zero_tile=ctypes.addressof(zeros), xs=ctypes.addressof(zeros))
    assert lib.tlk_launch_gemm(ctypes.byref(L), None) == 1          # hipErrorInvalidValue, nothing is launched
    try:
        override(lib, amode, 2)
        part, counters = resolve(lib, L)
    finally:
        override(lib, amode, 0)
    assert (L.kernel, L.cfg, L.split) == (kernel, cfg, 2)
    tiles = 2 * 2                                                   # 100 x 256 over 64 x 128
    assert (part, counters) == (tiles * 2 * 64 * 128 * 4, tiles)


@pytest.mark.gpu
@pytest.mark.parametrize("amode", [A_I8, A_BF16])
@pytest.mark.parametrize("M,N,K", [(200, 2048, 6144), (65, 272, 4096)])
def test_override_between_sizing_and_launch(lin, dev, amode, M, N, K):
    """Sized for 2 slices, launched after the override went to 16: the launch runs
    2, nothing past its partial sums is written, the sums are exact (small whole
    numbers) and the counters are back at zero."""
    import torch
    say(f"resolved plan amode={amode} M={M} N={N} K={K}")
    lib = lin.load_library()
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randint(-3, 4, (M, K), generator=g).float()
    w = torch.randint(-3, 4, (N, K), generator=g).float()
    x[:, 0] = w[:, 0] = 127.0                                       # absmax 127: codes are the values, scales 1
    want = (x.double() @ w.double().T).float()

    def tiles(a):
        t = torch.empty((a.shape[0] + 15) // 16 * 16 * a.shape[1], dtype=torch.uint8, device=dev)
        s = torch.empty((a.shape[0] + 15) // 16 * 16, device=dev)
        lin.w8a8_quantize_tiles_dev(a.to(dev), t, s)
        return t, s

    wt, ws = tiles(w)
    A, xs = tiles(x) if amode == A_I8 else (x.to(dev, torch.bfloat16), ws)
    y = torch.full((M, N), -1.0, device=dev)
    zero = torch.zeros(1024, dtype=torch.uint8, device=dev)
    L = GemmLaunch(amode=amode, A=A.data_ptr(), lda=K, Bt=wt.data_ptr(), ws=ws.data_ptr(), xs=xs.data_ptr(),
                   Y=y.data_ptr(), ldy=N, M=M, N=N, K=K, ep=0, out=OUT_F32, zero_tile=zero.data_ptr(), kernel=-1, split=1)
    try:
        override(lib, amode, 2)
        part, counters = resolve(lib, L)
        assert L.split == 2 and part > 0
        override(lib, amode, 16)
        pbuf = torch.full((part // 4 + 4096,), 123, dtype=torch.int32, device=dev)
        cbuf = torch.zeros(counters + 64, dtype=torch.int32, device=dev)
        L.part, L.cnt = pbuf.data_ptr(), cbuf.data_ptr()
        for _ in range(2):
            assert lib.tlk_launch_gemm(ctypes.byref(L), vp(torch.cuda.current_stream().cuda_stream)) == 0
        torch.cuda.synchronize()
    finally:
        override(lib, amode, 0)
    assert (pbuf[part // 4:] == 123).all() and (cbuf == 0).all()
    assert torch.equal(y.cpu(), want)


class RowsPlan(ctypes.Structure):            # csrc/tl_kernels.h
    _fields_ = [(n, i32) for n in ("tg", "nkb", "cpt", "kbs", "split", "r", "blocks")]


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(2, 2048, 6144), (7, 270, 4096)])
def test_rows_override_between_sizing_and_launch(lin, dev, M, N, K):
    """The same for the digit rows of up to 8 fp32 tokens: planned in 2 slices (or
    the fewest that fit), launched after the override went to 16."""
    import torch
    say(f"rows plan M={M} N={N} K={K}")
    lib = lin.load_library()
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randint(-3, 4, (M, K), generator=g).float()
    w = torch.randint(-3, 4, (N, K), generator=g).float()
    w[:, 0] = 127.0
    want = (x.double() @ w.double().T).float()
    wt = torch.zeros((N + 15) // 16 * 16 * K, dtype=torch.uint8, device=dev)
    ws = torch.zeros((N + 15) // 16 * 16, device=dev)
    lin.w8a8_quantize_tiles_dev(w.to(dev), wt, ws)
    xd = x.to(dev)
    y = torch.full((M, N), -1.0, device=dev)
    L = GemmLaunch(amode=3, A=xd.data_ptr(), lda=K, Bt=wt.data_ptr(), ws=ws.data_ptr(), Y=y.data_ptr(), ldy=N, M=M, N=N,
                   K=K, ep=0, out=OUT_F32, kernel=-1, split=1)
    plan = RowsPlan()
    lib.tlk_rows_workspace_bytes.restype = lib.tlk_rows_counter_count.restype = ctypes.c_size_t
    try:
        assert lib.tl_rows_set_split(2) == 0
        lib.tlk_rows_plan(M, N, K, ctypes.byref(plan))
        part = lib.tlk_rows_workspace_bytes(ctypes.byref(plan), M, N)
        assert 2 <= plan.split <= 4 and part == plan.split * M * N * 4
        assert lib.tl_rows_set_split(16) == 0
        pbuf = torch.full((part // 4 + 4096,), 123, dtype=torch.int32, device=dev)
        cbuf = torch.zeros(lib.tlk_rows_counter_count(N) + 64, dtype=torch.int32, device=dev)
        L.part, L.cnt = pbuf.data_ptr(), cbuf.data_ptr()
        for _ in range(2):
            assert lib.tlk_launch_rows(ctypes.byref(L), ctypes.byref(plan),
                                       vp(torch.cuda.current_stream().cuda_stream)) == 0
        torch.cuda.synchronize()
    finally:
        assert lib.tl_rows_set_split(0) == 0
    assert (pbuf[part // 4:] == 123).all() and (cbuf == 0).all()
    # the planes hold a value to 2^-32 of its row's absmax; the fold, the scale and
    # the slices' sum round at most 16 times, each within 2^-24 of the sum of terms
    assert ((y.cpu() - want).abs() <= 16 * 2.0 ** -24 * (x.abs() @ w.abs().T)).all()


@pytest.mark.gpu
def test_capture_without_split_workspace(lin, dev):
    """A shape that the planner gives K slices, captured on a stream that has no
    work-space for them (it cannot be allocated under capture): whole tiles, the same
    bits as the eager call, in every replay."""
    import torch
    M, N, K = 64, 6144, 6144
    say(f"int8 GEMM captured without a work-space M={M} N={N} K={K}")
    g = torch.Generator().manual_seed(7)
    W = lin.DeviceWeights.quantize(torch.randn(N, K, generator=g).to(dev))
    t = torch.empty(M * K, dtype=torch.uint8, device=dev)
    s = torch.empty(M, device=dev)
    y, captured = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev)
    x = torch.randn(M, K, generator=g)
    lin.w8a8_quantize_tiles_dev(x.to(dev), t, s)
    lin.w8a8_linear_tiles_dev(t, s, W, y)
    torch.cuda.synchronize()
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        lin.w8a8_linear_tiles_dev(t, s, W, captured)
    for i in range(3):
        lin.w8a8_quantize_tiles_dev((x * (i + 1)).to(dev).roll(i, 0), t, s)
        lin.w8a8_linear_tiles_dev(t, s, W, y)
        captured.fill_(-1.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, y)
    del graph
    W.close()


@pytest.mark.gpu
def test_16bit_capture_without_split_workspace(lin, dev):
    """The same for 16-bit rows, whose sums are taken in another order then: each
    output within K 2^-24 of the sum of its terms' magnitudes, twice (the bound of
    fp32 summation in any order, on both sides)."""
    import torch
    M, N, K = 333, 2048, 6144
    say(f"16-bit GEMM captured without a work-space M={M} N={N} K={K}")
    g = torch.Generator().manual_seed(8)
    w = torch.randn(N, K, generator=g)
    W = lin.DeviceWeights.quantize(w.to(dev))
    x = torch.randn(M, K, generator=g).bfloat16()
    xd = x.to(dev)
    y, captured = torch.empty(M, N, device=dev), torch.empty(M, N, device=dev)
    lin.w8a16_linear_dev(xd, W, y)
    torch.cuda.synchronize()
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph, stream=stream):
        lin.w8a16_linear_dev(xd, W, captured)
    bar = 2 * K * 2.0 ** -24 * (x.float().abs().to(dev) @ (w.abs().to(dev) * 1.01).t().contiguous())
    for _ in range(3):
        captured.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert ((captured - y).abs() <= bar).all()
    del graph
    W.close()
