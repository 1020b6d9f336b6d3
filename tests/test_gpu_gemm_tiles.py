"""The MFMA GEMM tiles (csrc/gemm_ring.h, the 256 x 256 pipeline on its grid and
masked) at the sizes where each can go wrong: one row, one K step,
edges one element past a tile, K a few elements into a step, token counts off
every grid.  Operands are views into NaN-filled buffers, so that a value read
past an edge shows up in the result, and outputs views into buffers whose
margin must stay untouched.  Each case names its tile on a 256-CU device and
asserts it (the tile rule's constants may move the shapes: choose others then).

Against the float64 product of the same rounded inputs every element is
within one storage ulp: one rounding of an fp32 sum whose error (at most
1031 products of O(1) values) is far below half an ulp of bf16 / fp16."""
import pytest
import torch

from tests.test_gpu_kernels import _assert_within_ulp

pytestmark = pytest.mark.gpu

# M, N, K along / K-major B, tile
ALONG_K = [(1, 360, 8, "64"), (33, 72, 40, "64"), (130, 200, 264, "64"),
           (74, 8416, 688, "64x128 k2"), (197, 8240, 232, "128 k2"), (1857, 8304, 8, "128"),
           (2184, 3656, 456, "256 masked"), (768, 2816, 256, "128x256"), (1280, 6656, 512, "256")]
WEIGHT_GRADIENT = [(16, 40, 13, "64"), (264, 136, 1, "64"), (600, 232, 5, "64"),
                   (200, 8296, 5, "128"), (1144, 2056, 33, "128"), (1424, 8216, 661, "256 masked"),
                   (136, 6888, 1031, "256 masked"), (256, 6912, 1024, "256")]


def _view(rows, cols, dtype, g, dev, scale=1.0):
    """A [rows, cols] view inside a NaN-filled buffer."""
    buf = torch.full((rows + 3, cols + 24), float("nan"), device=dev, dtype=dtype)
    v = buf[1:rows + 1, 8:cols + 8]
    v.copy_(scale * torch.randn(rows, cols, generator=g, device=dev))
    return v


def _run(M, N, K, a_km, b_km, dtype, dev, res, tile=None):
    from zorse_amd import kernels as K_
    print(f"gemm tile {M}x{N}x{K} a_kmajor={a_km} b_kmajor={b_km} {dtype}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    a = _view(K if a_km else M, M if a_km else K, dtype, g, dev)
    b = _view(K if b_km else N, N if b_km else K, dtype, g, dev, 0.05)
    r = _view(M, N, dtype, g, dev) if res else None
    buf = torch.full((M + 2, N + 16), 7.0, device=dev, dtype=dtype)
    out = buf[1:M + 1, 8:N + 8]
    assert tile in (None, K_.gemm_tile(M, N, K, a.stride(0), b.stride(0), out.stride(0), dtype,
                                       a_km, b_km, r.stride(0) if res else -1))
    K_.gemm(a, b, a_kmajor=a_km, b_kmajor=b_km, residual=r, out=out)
    am, bm = (a.t() if a_km else a).double(), (b if b_km else b.t()).double()
    ref = torch.mm(am.contiguous(), bm.contiguous())
    if res:
        ref += r.double()
    _assert_within_ulp(out, ref, dtype, f"{M}x{N}x{K}")
    out.fill_(7.0)
    assert bool((buf == 7.0).all()), "wrote outside the output view"


@pytest.mark.parametrize("b_km", [False, True], ids=["X_Wt", "dY_W"])
@pytest.mark.parametrize("M,N,K,tile", ALONG_K)
def test_gemm_tiles_along_k(dev, M, N, K, tile, b_km):
    _run(M, N, K, False, b_km, torch.bfloat16, dev, not b_km, tile)
    if M < 200:
        _run(M, N, K, False, b_km, torch.float16, dev, b_km, tile)


@pytest.mark.parametrize("M,N,K,tile", WEIGHT_GRADIENT)
def test_gemm_tiles_weight_gradient(dev, M, N, K, tile):
    _run(M, N, K, True, True, torch.bfloat16, dev, False, tile)
    if M < 300:
        _run(M, N, K, True, True, torch.float16, dev, True, tile)


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


# B, S, K, Hq, Hkv, d, tile ("general": the product and the pass, where a 64 x 64
# tile cannot hold a head of 128)
ROPE = [(3, 11, 72, 4, 2, 64, "64"), (3, 11, 72, 2, 1, 128, "general"),
        (2, 37, 688, 64, 1, 128, "64x128 k2"), (2, 37, 688, 128, 2, 64, "64x128 k2"),
        (1, 197, 232, 63, 1, 128, "128 k2"), (1, 197, 232, 127, 1, 64, "128 k2"),
        (3, 619, 8, 63, 1, 128, "128"), (3, 619, 8, 126, 2, 64, "128"),
        (1, 2184, 456, 27, 1, 128, "256 masked"), (1, 2184, 456, 54, 2, 64, "256 masked"),
        (4, 512, 512, 22, 1, 128, "128x256"), (4, 512, 256, 40, 4, 64, "128x256"),
        (5, 256, 512, 50, 1, 128, "256"), (5, 256, 512, 100, 2, 64, "256")]


@pytest.mark.parametrize("inter,explicit", [(False, False), (True, False), (False, True),
                                            (True, True)])
@pytest.mark.parametrize("B,S,K,Hq,Hkv,d,tile", ROPE)
def test_gemm_rope_tiles(dev, B, S, K, Hq, Hkv, d, tile, inter, explicit):
    """The RoPE epilogue of each tile writes what the product and the RoPE
    pass write, with positions that wrap inside a tile."""
    from zorse_amd import kernels as K_
    from zorse_amd.functional import rope_tables
    from zorse_amd._abi import dtype_code, lib
    print(f"gemm_rope tile B={B} S={S} K={K} {Hq}:{Hkv}x{d}", flush=True)
    g = torch.Generator(device=dev).manual_seed(7)
    x = _view(B * S, K, torch.bfloat16, g, dev)
    w = _view((Hq + 2 * Hkv) * d, K, torch.bfloat16, g, dev, 0.05)
    n_pos = S + 13 if explicit else S
    pos = torch.randperm(n_pos, generator=g, device=dev)[:S] if explicit else None
    cos, sin = rope_tables(n_pos, d, 1e4, torch.bfloat16, dev, inter)
    N, rot = (Hq + 2 * Hkv) * d, (Hq + Hkv) * d
    assert tile == K_.GEMM_TILES[lib().zk_gemm_rope_tile(
        B * S, N, K, x.stride(0), w.stride(0), N, S, rot, d, n_pos, dtype_code(x.dtype))]
    got = K_.gemm_rope(x, w, seq_len=S, rot_cols=rot, head_dim=d, cos=cos, sin=sin, positions=pos,
                       interleaved=inter)
    ref = K_.gemm(x, w)
    K_.rope_(ref[:, :Hq * d].view(B, S, Hq, d), ref[:, Hq * d:rot].view(B, S, Hkv, d), cos, sin,
             positions=pos, interleaved=inter)
    assert torch.equal(got, ref)


@pytest.mark.parametrize("M,F,K,tile", [
    (8, 24, 64, "64"), (72, 4216, 704, "64x128 k2"), (200, 4120, 256, "128 k2"),
    (1864, 4152, 64, "128"), (2184, 1832, 448, "128"), (2184, 1832, 512, "256 masked")])
def test_gemm_swiglu_tiles(dev, M, F, K, tile):
    """The SwiGLU epilogue of each masked tile: g and u within an ulp, z the
    SwiGLU kernel's bits, z^T its transpose."""
    from zorse_amd import kernels as K_
    from zorse_amd._abi import dtype_code, lib
    print(f"gemm_swiglu tile {M}x{F}x{K}", flush=True)
    g = torch.Generator(device=dev).manual_seed(9)
    x = _view(M, K, torch.bfloat16, g, dev)
    wg = _view(F, K, torch.bfloat16, g, dev, 0.05)
    wu = _view(F, K, torch.bfloat16, g, dev, 0.05)
    assert tile == K_.GEMM_TILES[lib().zk_gemm_swiglu_tile(M, F, K, x.stride(0), wg.stride(0), 2 * F,
                                                           dtype_code(x.dtype))]
    gu, z, zt = K_.gemm_swiglu(x, wg, wu, transposed=True)
    xm = x.double()
    _assert_within_ulp(gu[:, :F], torch.mm(xm, wg.double().t().contiguous()), torch.bfloat16, "g")
    _assert_within_ulp(gu[:, F:], torch.mm(xm, wu.double().t().contiguous()), torch.bfloat16, "u")
    assert torch.equal(z, K_.swiglu_fwd(gu[:, :F], gu[:, F:]))
    assert torch.equal(zt, z.t())
