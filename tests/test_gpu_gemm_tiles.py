"""The masked MFMA GEMM tiles (csrc/gemm_ring.h and the ragged form of the
256 x 256 pipeline) at the sizes where each can go wrong: one row, one K step,
edges one element past a tile, K a few elements into a step, token counts off
every grid.  Operands are views into NaN-filled buffers, so that a value read
past an edge shows up in the result, and outputs views into buffers whose
margin must stay untouched.  The shapes reach every tile on a 256-CU device
(named beside them).

Against the float64 product of the same rounded inputs every element is
within one storage ulp: one rounding of an fp32 sum whose error (at most
688 products of O(1) values) is far below half an ulp of bf16 / fp16."""
import pytest
import torch

from tests.test_gpu_kernels import _assert_within_ulp

pytestmark = pytest.mark.gpu

# M, N, K along / K-major B
ALONG_K = [(1, 360, 8), (33, 72, 40), (130, 200, 264),       # 64 x 64
           (74, 8416, 688),                                   # 64 x 128, split over K
           (197, 8240, 232),                                  # 128 x 128, split over K
           (1857, 8304, 8),                                   # 128 x 128
           (2184, 3656, 456)]                                 # 256 x 256, masked
WEIGHT_GRADIENT = [(16, 40, 13), (264, 136, 1),               # 64 x 64
                   (600, 232, 5),                             # 128 x 128
                   (1144, 2056, 33), (1424, 8216, 661)]       # 256 x 256, masked


def _view(rows, cols, dtype, g, dev, scale=1.0):
    """A [rows, cols] view inside a NaN-filled buffer."""
    buf = torch.full((rows + 3, cols + 24), float("nan"), device=dev, dtype=dtype)
    v = buf[1:rows + 1, 8:cols + 8]
    v.copy_(scale * torch.randn(rows, cols, generator=g, device=dev))
    return v


def _run(M, N, K, a_km, b_km, dtype, dev, res):
    from zorse_amd import kernels as K_
    print(f"gemm tile {M}x{N}x{K} a_kmajor={a_km} b_kmajor={b_km} {dtype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a = _view(K if a_km else M, M if a_km else K, dtype, g, dev)
    b = _view(K if b_km else N, N if b_km else K, dtype, g, dev, 0.05)
    r = _view(M, N, dtype, g, dev) if res else None
    buf = torch.full((M + 2, N + 16), 7.0, device=dev, dtype=dtype)
    out = buf[1:M + 1, 8:N + 8]
    K_.gemm(a, b, a_kmajor=a_km, b_kmajor=b_km, residual=r, out=out)
    am, bm = (a.t() if a_km else a).double(), (b if b_km else b.t()).double()
    ref = torch.mm(am.contiguous(), bm.contiguous())
    if res:
        ref += r.double()
    _assert_within_ulp(out, ref, dtype, f"{M}x{N}x{K}")
    out.fill_(7.0)
    assert bool((buf == 7.0).all()), "wrote outside the output view"


@pytest.mark.parametrize("b_km", [False, True], ids=["X_Wt", "dY_W"])
@pytest.mark.parametrize("M,N,K", ALONG_K)
def test_gemm_tiles_along_k(dev, M, N, K, b_km):
    _run(M, N, K, False, b_km, torch.bfloat16, dev, res=not b_km)
    if M < 200:
        _run(M, N, K, False, b_km, torch.float16, dev, res=b_km)


@pytest.mark.parametrize("M,N,K", WEIGHT_GRADIENT)
def test_gemm_tiles_weight_gradient(dev, M, N, K):
    _run(M, N, K, True, True, torch.bfloat16, dev, res=False)
    if M < 300:
        _run(M, N, K, True, True, torch.float16, dev, res=True)


def test_gemm_misaligned_equals_aligned(dev):
    """Operands whose rows are not 16-byte aligned take the general kernel,
    which sums K in the same order as the 64 x 64 tile: the same bits."""
    from zorse_amd import kernels as K_
    g = torch.Generator(device=dev).manual_seed(5)
    a = torch.randn(100, 264, generator=g, device=dev).to(torch.bfloat16)
    b = torch.randn(72, 264, generator=g, device=dev).to(torch.bfloat16)
    odd = torch.zeros(100, 271, device=dev, dtype=torch.bfloat16)[:, 3:267]
    odd.copy_(a)
    assert torch.equal(K_.gemm(odd, b), K_.gemm(a, b))


# B, S, K, Hq, Hkv, d: tiles 64 (heads of 64 in the epilogue, of 128 by the
# pass), 64 x 128, 128 split, 128, masked 256, 128 x 256
@pytest.mark.parametrize("B,S,K,Hq,Hkv,d,inter", [
    (3, 11, 72, 4, 2, 64, False), (3, 11, 72, 2, 1, 128, True), (2, 37, 688, 64, 1, 128, False),
    (1, 197, 232, 62, 1, 128, True), (3, 619, 8, 63, 1, 128, False),
    (1, 2184, 456, 27, 1, 128, False), (4, 512, 512, 22, 1, 128, False),
    (4, 512, 256, 40, 4, 64, True)])
def test_gemm_rope_tiles(dev, B, S, K, Hq, Hkv, d, inter):
    """The RoPE epilogue of each tile writes what the product and the RoPE
    pass write, with positions that wrap inside a tile."""
    from zorse_amd import kernels as K_
    from zorse_amd.functional import rope_tables
    print(f"gemm_rope tile B={B} S={S} K={K} {Hq}:{Hkv}x{d}", flush=True)
    g = torch.Generator(device=dev).manual_seed(7)
    x = _view(B * S, K, torch.bfloat16, g, dev)
    w = _view((Hq + 2 * Hkv) * d, K, torch.bfloat16, g, dev, 0.05)
    cos, sin = rope_tables(S, d, 1e4, torch.bfloat16, dev, inter)
    got = K_.gemm_rope(x, w, seq_len=S, rot_cols=(Hq + Hkv) * d, head_dim=d, cos=cos, sin=sin,
                       interleaved=inter)
    ref = K_.gemm(x, w)
    K_.rope_(ref[:, :Hq * d].view(B, S, Hq, d),
             ref[:, Hq * d:(Hq + Hkv) * d].view(B, S, Hkv, d), cos, sin, interleaved=inter)
    assert torch.equal(got, ref)


@pytest.mark.parametrize("M,F,K", [(8, 24, 64), (72, 4216, 704), (200, 4120, 256), (1864, 4152, 64),
                                   (2184, 1832, 448)])
def test_gemm_swiglu_tiles(dev, M, F, K):
    """The SwiGLU epilogue of each masked tile: g and u within an ulp, z the
    SwiGLU kernel's bits, z^T its transpose."""
    from zorse_amd import kernels as K_
    print(f"gemm_swiglu tile {M}x{F}x{K}", flush=True)
    g = torch.Generator(device=dev).manual_seed(9)
    x = _view(M, K, torch.bfloat16, g, dev)
    wg = _view(F, K, torch.bfloat16, g, dev, 0.05)
    wu = _view(F, K, torch.bfloat16, g, dev, 0.05)
    gu, z, zt = K_.gemm_swiglu(x, wg, wu, transposed=True)
    xm = x.double()
    _assert_within_ulp(gu[:, :F], torch.mm(xm, wg.double().t().contiguous()), torch.bfloat16, "g")
    _assert_within_ulp(gu[:, F:], torch.mm(xm, wu.double().t().contiguous()), torch.bfloat16, "u")
    assert torch.equal(z, K_.swiglu_fwd(gu[:, :F], gu[:, F:]))
    assert torch.equal(zt, z.t())
