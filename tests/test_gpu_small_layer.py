"""Small layers order their weight-gradient products behind the compute stream's
work instead of on the side stream: same kernels, same bytes -- also for a flat
buffer that is a view further on in its storage."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,strided", [(48, False), (48, True), (640, False)])
def test_in_order_and_side_stream_agree(monkeypatch, tokens, strided):
    import zorse_amd.layer as L
    spec = L.LayerSpec(hidden=256, heads=4, kv_heads=2, head_dim=64, ffn=512)
    gen = torch.Generator().manual_seed(tokens)
    flat = (torch.randn(spec.numel, generator=gen) * 0.05).bfloat16().cuda()
    if strided:  # a view further on in its buffer
        flat = torch.cat([flat.new_zeros(24), flat])[24:]
    x = torch.randn(1, tokens, spec.hidden, generator=gen).bfloat16().cuda()
    dout = torch.randn(1, tokens, spec.hidden, generator=gen).bfloat16().cuda()
    got = []
    for limit in (0.0, float("inf")):
        monkeypatch.setattr(L, "SIDE_STREAM_FLOPS", limit)
        xr, fr = x.clone().requires_grad_(), flat.detach().requires_grad_()
        out = L.DecoderLayerFunction.apply(xr, fr, spec, None)
        out.backward(dout)
        got.append((out.detach(), xr.grad, fr.grad))
    for a, b in zip(*got):
        assert torch.equal(a, b)


@pytest.mark.parametrize("missing", [8, 128 + 8])
def test_flat_parameter_too_short(missing):
    """A flat parameter that ends inside the norm weights is the kernels'
    ValueError about the weight's shape."""
    import zorse_amd.layer as L
    spec = L.LayerSpec(hidden=128, heads=2, kv_heads=1, head_dim=64, ffn=256)
    flat = torch.zeros(spec.numel - missing, device="cuda", dtype=torch.bfloat16)
    x = torch.zeros(1, 16, 128, device="cuda", dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="weight shape"):
        L.DecoderLayerFunction.apply(x, flat, spec, None)
