"""GPU attention alone against the oracle's attention, on the same inputs.

The decoder-level tests hold hidden rows to relative L2 1e-3, a bar set by
the reference's fast-exp SiLU (a last-bit difference can double one mlp
element).  Attention has no such amplifier, so here the GPU kernels get the
oracle's exact inputs through test hooks and are held to tight bars:

  * decode (tl_attn_decode_dev: q/k head RMSNorm, M-RoPE at the rotary
    position, K/V append at the cache position, GQA attention over the
    cache; reference kernel/decoder.c:72-118, kernel/ops.c:22-56 and
    :233-289, kernel/kv_cache.c:53-64, kernel/attention.c:172-224):
    the appended V row bit-exact, the appended K row and the attention
    output within relative L2 1e-6 and 1e-5 (only summation orders differ:
    tree sums here, sequential chains in the reference), earlier cache rows
    untouched;
  * prefill (tl_attn_prefill_dev: causal flash attention over the cache,
    kernel/attention.c:252-381): relative L2 1e-5 against the oracle's
    attention_prefill, also with the longest query tiles split in two halves
    and for a chunk attending to cached rows before it (CHUNKED_PREFILL_MODE,
    compared with the matching rows of one causal pass over all tokens).

A wrong rotation sign, a dropped norm weight, an off-by-one mask or a
misplaced softmax rescale moves these outputs by O(1), far above the bars.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32
NQ, NKV, HD = 16, 8, 128


def say(msg):
    print(f"[case] {msg}", flush=True)


def rel_l2(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


def _decode_reference(orc, qkv, qn, kn, cos, sin, kc, vc, pos, rope_pos):
    q = orc.rmsnorm(qkv[:NQ * HD].reshape(NQ, HD), qn).reshape(-1)
    k = orc.rmsnorm(qkv[NQ * HD:(NQ + NKV) * HD].reshape(NKV, HD), kn).reshape(-1)
    v = qkv[(NQ + NKV) * HD:]
    q, k = orc.mrope_apply(q, k, cos, sin, rope_pos)
    kc = kc.copy()
    vc = vc.copy()
    kc[:, pos] = k.reshape(NKV, HD)
    vc[:, pos] = v.reshape(NKV, HD)
    return orc.attention_decode(q, kc, vc, pos + 1), kc, vc


@pytest.mark.parametrize("pos,rope_pos", [(0, 0), (63, 63), (64, 64), (130, 500), (1199, 1199), (1455, 1455),
                                          (1711, 1711), (2047, 2047)])
def test_attn_decode_matches_oracle(lin, orc, dev, pos, rope_pos):
    import torch
    say(f"attention decode pos={pos} rope_pos={rope_pos}")
    lib = lin.load_library()
    max_seq = 2048
    rng = np.random.default_rng(pos * 7 + rope_pos)
    qkv = (rng.standard_normal((NQ + 2 * NKV) * HD) * 1.5).astype(F)
    qn = (1 + 0.1 * rng.standard_normal(HD)).astype(F)
    kn = (1 + 0.1 * rng.standard_normal(HD)).astype(F)
    cos, sin = orc.rope_tables(max_seq)
    kc = np.zeros((NKV, max_seq, HD), F)
    vc = np.zeros((NKV, max_seq, HD), F)
    # earlier rows: normalised-size keys (as the norm leaves them), values O(1)
    kc[:, :pos] = rng.standard_normal((NKV, pos, HD)).astype(F)
    vc[:, :pos] = rng.standard_normal((NKV, pos, HD)).astype(F)
    want, kw, vw = _decode_reference(orc, qkv, qn, kn, cos, sin, kc, vc, pos, rope_pos)

    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    args = [t(qkv), t(qn), t(kn), t(cos), t(sin)]
    for chunk in (32, 64, 128):              # positions per work-group, every kernel variant
        assert lib.tl_attn_set_chunk(chunk) == 0
        try:
            kd, vd = t(kc), t(vc)
            out = torch.full((NQ * HD,), np.nan, dtype=torch.float32, device=dev)
            rc = lib.tl_attn_decode_dev(*[a.data_ptr() for a in args], kd.data_ptr(), vd.data_ptr(), max_seq,
                                        pos, rope_pos, out.data_ptr(), None)
            assert rc == 0, lin.check(lib, "tl_attn_decode_dev")
        finally:
            lib.tl_attn_set_chunk(0)
        _check_decode(kd.cpu().numpy(), vd.cpu().numpy(), out.cpu().numpy(), kc, vc, kw, vw, want, pos)


def _check_decode(kg, vg, og, kc, vc, kw, vw, want, pos):
    np.testing.assert_array_equal(vg[:, pos], vw[:, pos])              # V appended as is
    assert rel_l2(kg[:, pos], kw[:, pos]) <= 1e-6, rel_l2(kg[:, pos], kw[:, pos])
    np.testing.assert_array_equal(kg[:, :pos], kc[:, :pos])            # earlier rows untouched
    np.testing.assert_array_equal(vg[:, :pos], vc[:, :pos])
    assert np.all(kg[:, pos + 1:] == 0) and np.all(vg[:, pos + 1:] == 0)
    assert np.all(np.isfinite(og))
    assert rel_l2(og, want) <= 1e-5, rel_l2(og, want)
    # per head too: a head-local mistake must not hide in the global norm
    for h in range(NQ):
        assert rel_l2(og[h * HD:(h + 1) * HD], want[h * HD:(h + 1) * HD]) <= 1e-5, h


def _prefill_inputs(rng, T):
    q = (rng.standard_normal((T, NQ * HD)) * 1.2).astype(F)
    k = (rng.standard_normal((T, NKV * HD)) * 1.2).astype(F)
    v = rng.standard_normal((T, NKV * HD)).astype(F)
    return q, k, v


def _run_prefill(lin, dev, q_rows, k, v, max_seq, key0, qoff, split):
    """q_rows: the S queries; k/v: token-major rows stored at cache rows 0..T-1."""
    import torch
    lib = lin.load_library()
    S, T = q_rows.shape[0], k.shape[0]
    qkv = np.zeros((S, (NQ + 2 * NKV) * HD), F)
    qkv[:, :NQ * HD] = q_rows
    kc = np.zeros((NKV, max_seq, HD), F)
    vc = np.zeros((NKV, max_seq, HD), F)
    kc[:, :T] = k.reshape(T, NKV, HD).transpose(1, 0, 2)
    vc[:, :T] = v.reshape(T, NKV, HD).transpose(1, 0, 2)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)
    qd, kd, vd = t(qkv), t(kc), t(vc)
    out = torch.full((S, NQ * HD), np.nan, dtype=torch.float32, device=dev)
    rc = lib.tl_attn_prefill_dev(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), S, max_seq, key0,
                                 qoff, 1 if split else 0, None)
    assert rc == 0, lin.check(lib, "tl_attn_prefill_dev")
    return out.cpu().numpy()


@pytest.mark.parametrize("S", [1, 64, 65, 130, 330, 1200])
@pytest.mark.parametrize("split", [False, True])
def test_attn_prefill_matches_oracle(lin, orc, dev, S, split):
    say(f"attention prefill S={S} split={split}")
    rng = np.random.default_rng(S * 3 + split)
    q, k, v = _prefill_inputs(rng, S)
    want = orc.attention_prefill(q, k, v)
    got = _run_prefill(lin, dev, q, k, v, 2048, 0, 0, split)
    assert np.all(np.isfinite(got))
    assert rel_l2(got, want) <= 1e-5, rel_l2(got, want)
    for t0 in sorted({0, S // 2, S - 1}):      # single rows: early, middle, last (longest key range)
        assert rel_l2(got[t0], want[t0]) <= 1e-5, t0


@pytest.mark.parametrize("base,S", [(64, 64), (100, 36), (1000, 200), (1136, 64)])
def test_attn_chunked_prefill_matches_oracle(lin, orc, dev, base, S):
    """A chunk of S queries at rows base.. attending to every cached row
    before it: the rows base..base+S-1 of one causal pass over base + S
    tokens."""
    say(f"attention chunked prefill base={base} S={S}")
    rng = np.random.default_rng(base + S)
    T = base + S
    q, k, v = _prefill_inputs(rng, T)
    want = orc.attention_prefill(q, k, v)[base:]
    for split in (False, True):
        got = _run_prefill(lin, dev, q[base:], k, v, 2048, 0, base, split)
        assert rel_l2(got, want) <= 1e-5, (split, rel_l2(got, want))


def _growing_inputs(rng, T, kind):
    """q, k, v whose scores make a query's running maximum move in later key
    tiles: "creep" raises every score a little from tile to tile (under a
    factor e^5 a tile), "climb" by more than that, "planted" raises single late
    keys for single queries (one lane of a wave grows, its neighbours do not),
    "jump" lifts every key past the middle at once (the two halves of a split
    key range have far apart maxima)."""
    q, k, v = _prefill_inputs(rng, T)
    u = rng.standard_normal(HD).astype(F)
    u *= F(np.sqrt(HD) / np.linalg.norm(u))             # |u|^2 = HD, so (x u).(y u) / sqrt(HD) = x y sqrt(HD)
    q, k = q.reshape(T, NQ, HD), k.reshape(T, NKV, HD)
    if kind == "planted":
        for j in range(40, T, 97):                      # key j towards the queries 3 and 20 rows further on
            for i, gain in ((j + 3, 0.6), (j + 20, 1.8)):
                if i < T:
                    k[j] += F(gain) * q[i, ::2]
    else:
        tile = (np.arange(T) // 64).astype(F)
        lift = {"creep": 3.0 * tile, "climb": 12.0 * tile, "jump": 40.0 * (np.arange(T) >= T // 2)}[kind]
        lift = np.minimum(lift, 60.0).astype(F)
        q += F(0.5) * u
        k += (lift / F(0.5 * np.sqrt(HD)))[:, None, None] * u
    return q.reshape(T, -1).astype(F), k.reshape(T, -1).astype(F), v


@pytest.mark.parametrize("kind", ["creep", "climb", "planted", "jump"])
@pytest.mark.parametrize("S,base", [(130, 0), (333, 0), (259, 77), (2048, 0)])
def test_attn_prefill_growing_maxima(lin, dev, S, base, kind):
    """Rows whose maximum grows in later key tiles, by little and by much, for
    some queries of a wave and not for others, and across the middle of a
    split key range, against float64, split and unsplit (2048 rows: the launch
    order's full 32 tiles).

    A score of q.k / sqrt(HD) in fp32 is off by at most e = (HD + 2) 2^-24
    |q| |k| / sqrt(HD); the largest of a query bounds the relative error of its
    weights by 2 e + 2^-22 (maximum and own score, the difference, the
    exponential).  An output is a weighted mean of values, so it moves by at
    most twice that times the largest |v|, plus the two sums' roundings."""
    import torch
    say(f"attention prefill S={S} base={base} {kind}")
    T = base + S
    q, k, v = _growing_inputs(np.random.default_rng(S + base), T, kind)
    q64 = torch.from_numpy(q[base:]).to(dev).double().reshape(S, NQ, HD).transpose(0, 1)
    k64 = torch.from_numpy(k).to(dev).double().reshape(T, NKV, HD).transpose(0, 1)
    v64 = torch.from_numpy(v).to(dev).double().reshape(T, NKV, HD).transpose(0, 1)
    mask = torch.ones((S, T), dtype=torch.bool, device=dev).tril(base)
    want = torch.empty((S, NQ, HD), dtype=torch.float64, device=dev)
    bar = torch.empty((S, NQ), dtype=torch.float64, device=dev)
    grew = False
    for h in range(NQ):
        s = q64[h] @ k64[h // 2].t().contiguous() / HD ** 0.5
        s.masked_fill_(~mask, float("-inf"))
        want[:, h] = torch.softmax(s, 1) @ v64[h // 2]
        e = (HD + 2) * 2.0 ** -24 * q64[h].norm(dim=1) * k64[h // 2].norm(dim=1).max() / HD ** 0.5
        bar[:, h] = (2 * (2 * e + 2.0 ** -22) + 2 * T * 2.0 ** -24) * v64[h // 2].abs().max()
        tile_max = torch.stack([t.amax(1) for t in s.split(64, 1)], 1)
        before = torch.cummax(tile_max, 1).values[:, :-1]
        grew |= bool(((tile_max[:, 1:] > before) & before.isfinite()).any())
    assert grew
    for split in (False, True):
        got = _run_prefill(lin, dev, q[base:], k, v, 2048, 0, base, split)
        err = (torch.from_numpy(got).to(dev).double().reshape(S, NQ, HD) - want).abs().amax(2)
        assert bool((err <= bar).all()), (split, float((err / bar).max()))


def _fma32(a, b, c):
    return (a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)).astype(F)


def _softmax_steps(scores, split):
    """The online softmax over 64-key tiles in fp32, one rounding per step, of
    scores [S, T] (float32, masked ones -3e38): the weights before
    normalisation [S, T], and the sum.  With two halves, the state of each and
    their combination in order."""
    import torch
    exp = lambda a: torch.exp(torch.from_numpy(np.ascontiguousarray(a, F)).cuda()).cpu().numpy()
    S, T = scores.shape
    parts = []
    for lo, hi in split:
        m, l = np.full(S, -3.0e38, F), np.zeros(S, F)
        o = np.zeros((S, T), F)
        for t0 in range(64 * lo, 64 * hi, 64):
            s = np.full((S, 64), -3.0e38, F)
            s[:, :min(64, T - t0)] = scores[:, t0:t0 + 64]
            m_new = np.maximum(m, s.max(1))
            resc = exp(m - m_new)
            p = np.where(s > F(-1.0e38), exp(s - m_new[:, None]), F(0))
            lanes = np.zeros((S, 4), F)                 # lane group g sums keys 16b + 4r + g
            for j in range(0, 64, 4):
                lanes = lanes + p[:, j:j + 4]
            ps = (lanes[:, 0] + lanes[:, 1]) + (lanes[:, 2] + lanes[:, 3])
            l = _fma32(l, resc, ps)
            o *= resc[:, None]
            o[:, t0:t0 + 64] = p[:, :min(64, T - t0)]
            m = m_new
        parts.append((m, l, o))
    if len(parts) == 1:
        return parts[0][2], parts[0][1]
    (m0, l0, o0), (m1, l1, o1) = parts
    M = np.maximum(m0, m1)
    a0, a1 = exp(m0 - M), exp(m1 - M)
    return o0 * a0[:, None] + o1 * a1[:, None], l0 * a0 + l1 * a1


@pytest.mark.parametrize("S", [17, 64, 100, 128])
@pytest.mark.parametrize("split", [False, True])
def test_attn_prefill_softmax_steps_bit_exact(lin, dev, S, split):
    """The softmax's own arithmetic, bit for bit: scale, subtract the running
    maximum, exp, rescale, each rounded to fp32 once.  Small integers in q and
    k make every score exact, and value row j is the unit vector of dimension
    j, so that an output is one key's weight over the sum and no order of
    summation inside an MFMA shows.  With `split` two key tiles may be taken in
    halves, which rounds in another place; an output has to equal one of the
    two forms."""
    say(f"attention prefill softmax steps S={S} split={split}")
    rng = np.random.default_rng(S)
    q = np.zeros((S, NQ, HD), F)
    k = np.zeros((S, NKV, HD), F)
    q[:, :, :24] = rng.integers(-4, 5, (S, NQ, 24))
    k[:, :, :24] = rng.integers(-4, 5, (S, NKV, 24))
    q[:, :, 30] = 1.0
    k[:, :, 30] = (np.arange(S) // 8 * 7)[:, None]      # maxima that move from tile to tile
    v = np.zeros((S, NKV, HD), F)
    v[np.arange(S), :, np.arange(S)] = 1.0
    got = _run_prefill(lin, dev, q.reshape(S, -1), k.reshape(S, -1), v.reshape(S, -1), 2048, 0, 0, split)
    got = got.reshape(S, NQ, HD)
    scale = F(0.08838834764831843)                      # 1 / sqrt(HD), as the kernel gets it
    causal = np.tril(np.ones((S, S), bool))
    for h in range(NQ):
        s = np.where(causal, (q[:, h] @ k[:, h // 2].T) * scale, F(-3.0e38)).astype(F)
        ntiles = -(-S // 64)
        forms = [[(0, ntiles)]] + ([[(0, 1), (1, 2)]] if split and ntiles == 2 else [])
        want = []
        for f in forms:
            w, l = _softmax_steps(s, f)
            want.append(w * (F(1) / l)[:, None])
        rows = [np.array([np.array_equal(got[i, h, :S], w[i]) for i in range(S)]) for w in want]
        bad = np.flatnonzero(~np.logical_or.reduce(rows))
        assert bad.size == 0, (h, bad[:5], got[bad[0], h, :S], want[0][bad[0]])
