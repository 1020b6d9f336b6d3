"""rope_copy gives the bytes of a copy rotated in place, from contiguous and
strided sources (which it leaves alone), for one position, few and many heads,
and for the sources its kernel does not take."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,S,Hq,Hkv,d,dtype,inter,off", [
    (1, 1, 1, 1, 64, torch.bfloat16, False, 0), (2, 33, 3, 1, 128, torch.float16, True, 0),
    (2, 37, 32, 8, 128, torch.bfloat16, False, 8), (3, 65, 40, 40, 64, torch.float16, False, 8),
    (1, 9, 4, 2, 128, torch.bfloat16, True, 2), (1, 9, 4, 2, 96, torch.bfloat16, False, 0),
    (1, 9, 4, 2, 64, torch.float32, False, 0)])
def test_rope_copy(dev, B, S, Hq, Hkv, d, dtype, inter, off):
    from zorse_amd import kernels as K
    g = torch.Generator().manual_seed(S)
    buf = torch.randn(B, S, (Hq + Hkv) * d + off, generator=g).to(dtype).to(dev)
    heads = buf[..., off:].unflatten(-1, (Hq + Hkv, d))
    q, k, before = heads[:, :, :Hq], heads[:, :, Hq:], buf.clone()
    ang = torch.rand(S + 3, d // 2, generator=g).to(dev) * 6.28
    cos, sin = ang.cos(), ang.sin()
    qo, ko = K.rope_copy(q, k, cos, sin, interleaved=inter)
    qr, kr = q.contiguous().clone(), k.contiguous().clone()
    K.rope_(qr, kr, cos, sin, interleaved=inter)
    assert torch.equal(qo, qr) and torch.equal(ko, kr) and torch.equal(buf, before)
    assert qo.is_contiguous() and ko.is_contiguous()


@pytest.mark.parametrize("shape", [(0, 4, 2, 64), (2, 0, 2, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rope_copy_refuses_empty_tensors(dev, shape, dtype):
    """As rope_ does, whatever the kernel: no position to rotate is an error."""
    from zorse_amd import kernels as K
    q = torch.zeros(shape, device=dev, dtype=dtype)
    cos = torch.ones(4, shape[3] // 2, device=dev)
    with pytest.raises(RuntimeError, match="zk_rope"):
        K.rope_copy(q, q, cos, cos)
