"""The attention kernels for head dims between 34 and 126 other than 64
(zk_attn_*_ragged) at the edges of their tiles: next to the same problem
zero-padded to 64 / 128 through the kernels for those, whose sums run over the
same products in the same order."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

# B, Sq, Skv, Hq, Hkv, d, causal, window, dtype: one row, tile edges, every
# number of 16-element steps, dims off 4, GQA, cross lengths, windows
CASES = [(1, 1, 1, 1, 1, 34, True, 0, torch.bfloat16),
         (2, 33, 33, 2, 1, 48, True, 0, torch.float16),
         (1, 130, 130, 2, 2, 62, True, 17, torch.bfloat16),
         (1, 257, 257, 4, 2, 68, True, 0, torch.bfloat16),
         (1, 64, 129, 2, 2, 84, False, 0, torch.float16),
         (2, 96, 31, 2, 1, 96, False, 0, torch.bfloat16),
         (1, 128, 128, 3, 3, 100, True, 0, torch.bfloat16),
         (1, 95, 95, 4, 4, 110, True, 40, torch.float16),
         (1, 65, 65, 1, 1, 126, True, 0, torch.bfloat16)]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c[:8]))
def test_ragged_head_dims_match_padded(dev, case):
    from zorse_amd import kernels as K
    B, Sq, Skv, Hq, Hkv, d, causal, window, dtype = case
    print(f"ragged attention {case}", flush=True)
    dp = 64 if d < 64 else 128
    gen = torch.Generator().manual_seed(d)

    def rand(S, H):
        return torch.randn(B, S, H, d, generator=gen).to(dtype).to(dev)

    # q, k, v as the heads of one row when their lengths agree, with infinities
    # before and after every tensor's own elements: neighbours must not leak in
    def embed(t):
        buf = torch.full((B, t.shape[1], t.shape[2] + 2, d), float("inf"), dtype=dtype, device=dev)
        buf[:, :, 1:-1] = t
        return buf[:, :, 1:-1]

    q, k, v, do = rand(Sq, Hq), rand(Skv, Hkv), rand(Skv, Hkv), rand(Sq, Hq)
    pad = [torch.nn.functional.pad(t, (0, dp - d)).contiguous() for t in (q, k, v, do)]
    kw = dict(causal=causal, window=window, scale=1.0 / math.sqrt(d))
    o_ref, lse_ref = K.attn_fwd(*pad[:3], **kw)
    g_ref = K.attn_bwd(*pad[:3], o_ref, pad[3], lse_ref, **kw)
    out = embed(torch.full_like(q, 7.0))
    qe, ke, ve, de = (embed(t) for t in (q, k, v, do))
    assert K.attn_ragged_takes(qe, ke, ve, de, out)
    o, lse = K.attn_fwd(qe, ke, ve, out=out, ragged=True, **kw)
    outs = [embed(torch.full_like(t, 7.0)) for t in (q, k, v)]
    g = K.attn_bwd(qe, ke, ve, o, de, lse, dq=outs[0], dk=outs[1], dv=outs[2], ragged=True, **kw)
    assert torch.equal(lse, lse_ref)
    assert torch.equal(o, o_ref[..., :d])
    for t in (out, *outs):  # the neighbouring heads are untouched
        whole = t._base
        assert bool(torch.isinf(whole[:, :, 0]).all()) and bool(torch.isinf(whole[:, :, -1]).all())
    # the backward's delta adds the same squares in the same order, so the
    # gradients differ at most where fp32 contraction of the epilogue does
    for a, b in zip(g, g_ref):
        b = b[..., :d]
        scale = float(b.float().abs().max())
        assert float((a.float() - b.float()).abs().max()) <= 2.0 ** -8 * scale


@pytest.mark.parametrize("d,pairing", [(36, False), (68, True), (100, False), (84, True)])
@pytest.mark.parametrize("heads", [(1, 1), (5, 2), (32, 8)])
def test_rope_other_head_dims(dev, d, pairing, heads):
    """rope_ on head dims that are multiples of 4 (4-byte accesses) gives the
    bytes of the general pass, which odd row offsets still take."""
    from zorse_amd import kernels as K
    Hq, Hkv = heads
    B, S = 2, 37
    gen = torch.Generator().manual_seed(d)
    x = torch.randn(B, S, (Hq + Hkv) * d, generator=gen).bfloat16().to(dev)
    ang = torch.rand(S, d // 2, generator=gen).to(dev) * 6.28
    cos, sin = ang.cos(), ang.sin()
    odd = torch.empty(B, S, (Hq + Hkv) * d + 1, dtype=x.dtype, device=dev)
    odd[..., 1:] = x
    for inverse in (False, True):
        got = x.clone()
        for buf, off in ((got, 0), (odd, 1)):
            view = buf[..., off:].unflatten(-1, (Hq + Hkv, d))
            K.rope_(view[:, :, :Hq], view[:, :, Hq:], cos, sin, interleaved=pairing,
                    inverse=inverse)
        assert torch.equal(got, odd[..., 1:])
        odd[..., 1:] = x
