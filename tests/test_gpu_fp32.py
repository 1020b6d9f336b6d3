"""The fp32 matrix-core kernels (csrc/attn_f32.hip, the fp32 tiles of
csrc/gemm_ring.h) at the edges of their tiles, against float64.

Bounds: fp32 sums of n products are off by at most n 2^-24 times the sum of
the absolute products; attention results by assert_close's 1e-4 of the
largest value."""
import pytest
import torch

from oracle import decoder as O
from tests._tol import assert_close

pytestmark = pytest.mark.gpu


def _randn(shape, seed, dev):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dev)


# 64 x 64 tiles (fewer 128 x 128 tiles than CUs) and 128 x 128 tiles; K a few
# elements into a step, one row, weight gradients over odd token counts
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (65, 72, 40), (256, 688, 256), (2056, 2200, 40)])
@pytest.mark.parametrize("layout", [(False, False), (False, True), (True, True), (True, False)],
                         ids=["X_Wt", "dY_W", "dYt_X", "At_B"])
def test_gemm_fp32_tiles(dev, M, N, K, layout):
    from zorse_amd import kernels as K_
    a_km, b_km = layout
    if a_km:
        M, K = -(-M // 8) * 8, K if not b_km else K + 3
    print(f"gemm fp32 {M}x{N}x{K} {layout}", flush=True)
    pad = torch.full(((K if a_km else M) + 1, (M if a_km else K) + 8), float("nan"), device=dev)
    a = pad[:-1, :-8]
    a.copy_(_randn(a.shape, 1, dev))
    bpad = torch.full(((K if b_km else N) + 1, (N if b_km else K) + 8), float("nan"), device=dev)
    b = bpad[:-1, :-8]
    b.copy_(_randn(b.shape, 2, dev))
    r = _randn((M, N), 3, dev)
    out = torch.full((M + 1, N + 8), 7.0, device=dev)
    K_.gemm(a, b, a_kmajor=a_km, b_kmajor=b_km, residual=r, out=out[:M, :N])
    am = (a.t() if a_km else a).double().contiguous()
    bm = (b if b_km else b.t()).double().contiguous()
    ref = torch.mm(am, bm) + r.double()
    bound = (K + 2) * 2.0 ** -24 * (torch.mm(am.abs(), bm.abs()) + r.double().abs())
    assert bool(((out[:M, :N].double() - ref).abs() <= bound).all())
    assert bool((out[M:] == 7).all()) and bool((out[:, N:] == 7).all())


# B, Sq, Skv, Hq, Hkv, d, causal, window: one row, tile edges at 32 and 64,
# head dims off 4, GQA, cross lengths, windows
CASES = [(1, 1, 1, 1, 1, 16, True, 0), (2, 31, 31, 2, 1, 64, True, 0),
         (1, 65, 65, 4, 2, 50, True, 33), (1, 130, 130, 2, 2, 128, True, 0),
         (1, 33, 97, 4, 4, 100, False, 0), (1, 97, 32, 2, 1, 66, False, 0),
         (2, 128, 128, 4, 4, 64, True, 0), (1, 64, 64, 3, 1, 110, True, 1)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c))
def test_attention_fp32(dev, case):
    from zorse_amd import kernels as K
    B, Sq, Skv, Hq, Hkv, d, causal, window = case
    print(f"attention fp32 {case}", flush=True)
    q, do = _randn((B, Sq, Hq, d), 10, "cpu"), _randn((B, Sq, Hq, d), 11, "cpu")
    k, v = _randn((B, Skv, Hkv, d), 12, "cpu"), _randn((B, Skv, Hkv, d), 13, "cpu")
    dq_, dk_, dv_ = (t.to(dev) for t in (q, k, v))
    o, lse = K.attn_fwd(dq_, dk_, dv_, causal=causal, window=window)
    ro, rlse = O.attention(q.double(), k.double(), v.double(), causal, window)
    assert_close(o, ro, torch.float32, "o")
    assert_close(lse, rlse, torch.float32, "lse")
    got = K.attn_bwd(dq_, dk_, dv_, o, do.to(dev), lse, causal=causal, window=window)
    ref = O.attention_bwd(q.double(), k.double(), v.double(), do.double(), causal, window)
    # dS = P (dP - delta) cancels (wholly for a query with one visible key):
    # dP and delta are sums of d products, each off by up to (d + 2) 2^-24 of
    # their absolute products, carried into dq / dk by k / q and the scale
    big = [t.abs().max().item() for t in (do, v, q, k)]
    floor = (d + 2) * 2.0 ** -24 * d * big[0] * big[1] * max(big[2:]) / d ** 0.5
    for name, g, r in zip(("dq", "dk", "dv"), got, ref):
        diff = (g.double().cpu() - r).abs().max().item()
        assert diff <= 1e-4 * r.abs().max().item() + (floor if name != "dv" else 0), (name, diff)


def test_attention_fp32_masked_values_do_not_leak(dev):
    """An infinity or NaN in a position a row does not see leaves the row's
    result as it was, bit for bit within the sums' rounding: the last 9 tokens
    hold infinities, the other rows match a run on the shorter sequence."""
    from zorse_amd import kernels as K
    S, keep, H, d = 70, 61, 2, 48
    q, k, v, do = (_randn((2, S, H, d), 20 + i, dev) for i in range(4))
    for t in (q, k, v, do):
        t[:, keep:] = float("inf")
        t[:, keep + 3] = float("nan")
    o, lse = K.attn_fwd(q, k, v, causal=True)
    short = [t[:, :keep].contiguous() for t in (q, k, v, do)]
    so, slse = K.attn_fwd(*short[:3], causal=True)
    assert_close(o[:, :keep], so.double(), torch.float32, "o")
    assert_close(lse[..., :keep], slse.double(), torch.float32, "lse")
    dq, _, _ = K.attn_bwd(q, k, v, o, do, lse, causal=True)
    sdq, _, _ = K.attn_bwd(*short[:3], so, short[3], slse, causal=True)
    assert_close(dq[:, :keep], sdq.double(), torch.float32, "dq")


def _rows_reference(q, k, v, do, window):
    """Causal attention and its gradients in float64 over the keys each query
    sees, a row at a time, so that a hidden infinity or NaN never meets a zero
    weight.  [S, d] each."""
    S, scale = q.shape[0], q.shape[1] ** -0.5
    o, (dq, dk, dv) = torch.zeros_like(q), (torch.zeros_like(t) for t in (q, k, v))
    for i in range(S):
        js = slice(max(0, i - window + 1) if window else 0, i + 1)
        p = torch.softmax((k[js] @ q[i]) * scale, 0)
        o[i] = p @ v[js]
        ds = p * (v[js] @ do[i] - o[i] @ do[i]) * scale
        dq[i] = ds @ k[js]
        dk[js] += torch.outer(ds, q[i])
        dv[js] += torch.outer(p, do[i])
    return o, dq, dk, dv


@pytest.mark.parametrize("window", [0, 9])
@pytest.mark.parametrize("d", [64, 18])
@pytest.mark.parametrize("kind", ["minus_inf_scores", "nan_key", "nan_query"])
def test_attention_fp32_nonfinite_rows_stay_nonfinite(dev, kind, d, window):
    """A query whose visible scores are all -inf, or one of them NaN, has no
    softmax: its output is NaN, and so are the gradients that its weights reach
    -- not zeros, which would hide it from the loss.  The NaNs are where the
    float64 rows have them and the finite values are theirs."""
    from zorse_amd import kernels as K
    S = 40
    q, k, v, do = (_randn((S, d), 30 + i, "cpu") for i in range(4))
    if kind == "minus_inf_scores":
        q, k[:6] = q.abs(), float("-inf")
    elif kind == "nan_key":
        k[7, 3] = float("nan")
    else:
        q[5, 2] = float("nan")
    dev4 = [t.to(dev)[None, :, None] for t in (q, k, v, do)]
    o, lse = K.attn_fwd(*dev4[:3], causal=True, window=window)
    got = (o, *K.attn_bwd(*dev4[:3], o, dev4[3], lse, causal=True, window=window))
    ref = _rows_reference(*(t.double() for t in (q, k, v, do)), window)
    for name, g, r in zip(("o", "dq", "dk", "dv"), got, ref):
        g = g[0, :, 0].double().cpu()
        # an infinite weight times a gradient may be infinite or NaN
        assert torch.equal(g.isfinite(), r.isfinite()), name
        ok = r.isfinite()
        assert_close(torch.where(ok, g, 0), torch.where(ok, r, 0), torch.float32, name)


# S, d, aligned: one token, both sides of the row kernels' limits (S d of 128 at
# 1024 heads, 512 at 4096 up to four tokens, two thirds of that unaligned), and
# the padded element counts of each instance
@pytest.mark.parametrize("S,d,heads,causal,window,rope", [
    (1, 64, 1024, True, 0, False), (4, 32, 1024, True, 0, True), (5, 32, 1024, True, 0, False),
    (8, 16, 1024, False, 0, False), (4, 128, 4096, True, 2, True), (3, 6, 1026, True, 0, True),
    (2, 70, 4098, True, 0, True), (1, 126, 1024, True, 0, False), (7, 13, 1026, False, 0, False)])
def test_attention_fp32_short_sequences(dev, S, d, heads, causal, window, rope):
    """Many sequences of a few tokens: the row kernels, GQA of two heads each,
    in the dimensions where a pass of one kind meets one of the other (the keys'
    heads are half the queries')."""
    from zorse_amd import kernels as K
    from zorse_amd.functional import rope_tables
    B, Hq, Hkv = heads // 2, 4, 2  # the keys' heads: `heads`; the queries': twice as many
    print(f"short sequences S={S} d={d} heads={heads}", flush=True)
    q, do = _randn((B, S, Hq, d), 40, "cpu"), _randn((B, S, Hq, d), 41, "cpu")
    k, v = _randn((B, S, Hkv, d), 42, "cpu"), _randn((B, S, Hkv, d), 43, "cpu")
    g = [t.to(dev) for t in (q, k, v)]
    o, lse = K.attn_fwd(*g, causal=causal, window=window)
    ro, rlse = O.attention(q.double(), k.double(), v.double(), causal, window)
    assert_close(o, ro, torch.float32, "o")
    assert_close(lse, rlse, torch.float32, "lse")
    got = K.attn_bwd(*g, o, do.to(dev), lse, causal=causal, window=window)
    ref = O.attention_bwd(q.double(), k.double(), v.double(), do.double(), causal, window)
    big = [t.abs().max().item() for t in (do, v, q, k)]
    floor = (d + 2) * 2.0 ** -24 * d * big[0] * big[1] * max(big[2:]) / d ** 0.5
    for name, x, r in zip(("dq", "dk", "dv"), got, ref):
        diff = (x.double().cpu() - r).abs().max().item()
        assert diff <= 1e-4 * r.abs().max().item() + (floor if name != "dv" else 0), (name, diff)
    if rope:  # the fused rotation is the rotation pass over the plain gradients
        for inter in (False, True):
            cos, sin = rope_tables(S, d, 1e4, torch.float32, dev, inter)
            rot = K.attn_bwd(*g, o, do.to(dev), lse, causal=causal, window=window,
                             rope=(cos, sin, None, inter))
            want = [t.clone() for t in got]
            K.rope_(want[0], want[1], cos, sin, interleaved=inter, inverse=True)
            for x, r in zip(rot, want):
                assert_close(x, r.double(), torch.float32, "rope")


def test_attention_fp32_short_sequences_cost_their_rows(dev):
    """Attention over 65536 sequences of one token takes less than 8 times as
    long as over 4096 (12 us, the floor of a launch; 0.5 ms when every sequence
    takes a workgroup of 64 rows)."""
    from zorse_amd import kernels as K

    def best(B):
        x = _randn((B, 1, 1, 16), 50, dev)
        K.attn_fwd(x, x, x)
        times = []
        for _ in range(5):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            for _ in range(10):
                K.attn_fwd(x, x, x)
            t1.record()
            t1.synchronize()
            times.append(t0.elapsed_time(t1))
        return min(times)
    assert best(65536) < 8 * best(4096)


@pytest.mark.parametrize("S,d", [(1, 4), (5, 35)])
def test_attention_fp32_more_workgroups_than_one_grid_dimension(dev, S, d):
    """2^24 + 64 heads: 2^32 threads and more, past what one grid dimension of a
    launch holds, for the row kernels and for the tiles.  Every head holds the
    same values (expanded views) and gives the same bits."""
    from zorse_amd import kernels as K
    B, H = (1 << 18) + 1, 64
    print(f"{B * H} heads of {S} x {d}", flush=True)
    one = [_randn((1, S, 1, d), 60 + i, dev) for i in range(4)]
    q, k, v, do = (t.expand(B, S, H, d) for t in one)
    want, wlse = K.attn_fwd(*one[:3])
    o, lse = K.attn_fwd(q, k, v)
    assert torch.equal(o[:1, :, :1], o[-1:, :, -1:])
    assert_close(o[:1, :, :1], want.double(), torch.float32, "o")
    for t in o.split(1 << 14):
        assert bool((t == o[:1, :, :1]).all())
    del o
    assert_close(lse[:1, :1], wlse.double(), torch.float32, "lse")
    assert bool((lse == lse[:1, :1]).all())
    grads = K.attn_bwd(q, k, v, want.expand(B, S, H, d), do, lse)
    ref = K.attn_bwd(*one[:3], want, one[3], wlse)
    for g, r in zip(grads, ref):
        assert_close(g[:1, :, :1], r.double(), torch.float32, "gradient")
        for t in g.split(1 << 14):
            assert bool((t == g[:1, :, :1]).all())
