"""The output layer's loss at the edges of its passes: column counts around one
sweep of the forward kernel (8192 columns), more rows than the one-workgroup
passes have threads, an ignore_index inside the vocabulary, nothing but ignored
rows, and logits of -inf."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,V,chunk,ignore", [(1, 8, 8, -100), (3, 8192, 8192, 5),
                                              (1030, 8200, 4096, -100), (17, 16392, 16392, 0)])
def test_mean_loss_edges(dev, T, V, chunk, ignore):
    from zorse_amd.lm_head import lm_head_cross_entropy
    g = torch.Generator().manual_seed(V)
    x = torch.randn(T, 16, generator=g)
    w = torch.randn(V, 16, generator=g)
    labels = torch.randint(0, V, (T,), generator=g)
    labels[::4] = ignore
    if T == 1:
        labels[0] = 3
    xd, wd = x.to(dev).requires_grad_(), w.to(dev).requires_grad_()
    loss = lm_head_cross_entropy(xd, wd, labels.to(dev), chunk=chunk, ignore_index=ignore)
    (3.0 * loss).backward()
    xr, wr = x.double().requires_grad_(), w.double().requires_grad_()
    ref = torch.nn.functional.cross_entropy(xr @ wr.t(), labels, ignore_index=ignore)
    (3.0 * ref).backward()
    # fp32 logits of 16 products (2^-24 of their sum each way) and sums of V terms
    assert abs(loss.item() - ref.item()) <= 1e-5 * (1 + abs(ref.item()))
    for a, b in ((xd.grad, xr.grad), (wd.grad, wr.grad)):
        assert float((a.double().cpu() - b).norm()) <= 2e-5 * float(b.norm())


def test_all_rows_ignored(dev):
    from zorse_amd.lm_head import lm_head_cross_entropy
    x = torch.randn(5, 16, device=dev, requires_grad=True)
    w = torch.randn(64, 16, device=dev, requires_grad=True)
    loss = lm_head_cross_entropy(x, w, torch.full((5,), -100, device=dev))
    loss.backward()
    assert loss.item() == 0 and not bool(x.grad.any()) and not bool(w.grad.any())


def test_minus_infinity_logits(dev):
    """Columns of -inf (a masked vocabulary), also as a thread's whole sweep,
    weigh nothing."""
    from zorse_amd import lm_head as LH
    rows, cols = 2, 8192 + 64
    logits = torch.full((rows, cols), float("-inf"), device=dev)
    logits[:, 8200:8208] = 1.0
    m = torch.full((rows,), float("-inf"), device=dev)
    s, t = torch.zeros(rows, device=dev), torch.zeros(rows, device=dev)
    LH._fwd_chunk(logits, torch.tensor([8201, -1], device=dev), 0, m, s, t)
    assert torch.equal(m, torch.ones_like(m)) and torch.allclose(s, torch.full_like(s, 8.0))
    assert t.tolist() == [1.0, 0.0]


@pytest.mark.parametrize("bad", [4096, -1])
def test_bad_labels_are_refused_before_any_product(dev, bad):
    """A label out of range raises with no logits (67 MB here) allocated."""
    from zorse_amd.lm_head import lm_head_cross_entropy
    T, V = 4096, 4096
    x, w = torch.randn(T, 64, device=dev), torch.randn(V, 64, device=dev)
    labels = torch.zeros(T, dtype=torch.int64, device=dev)
    labels[T - 1] = bad
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    with pytest.raises(ValueError, match="labels must lie in"):
        lm_head_cross_entropy(x, w, labels)
    assert torch.cuda.max_memory_allocated() - before < 1 << 20
