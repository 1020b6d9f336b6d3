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


@pytest.mark.parametrize("T", [16384, 16385, 20480, 40001])
def test_labels_and_mean_over_many_rows(dev, T):
    """Both sides of the row count from which the labels and the mean take more
    than one workgroup: row labels, counts, log-sum-exp and loss."""
    from zorse_amd._abi import check, lib, ptr, stream_handle
    from zorse_amd.lm_head import lm_head_cross_entropy
    g = torch.Generator().manual_seed(T)
    given = torch.randint(0, 50, (T,), generator=g)
    given[::5], given[T - 1], given[7] = -100, 50, -3
    out = torch.empty(T, dtype=torch.int64, device=dev)
    acc = torch.empty(4, T, device=dev)
    stats, host = torch.full((2,), 9, device=dev), torch.full((2,), 9).pin_memory()
    lab = given.to(dev)
    check(lib().zk_ce_labels(ptr(lab), T, 50, -100, ptr(out), ptr(acc[0]), ptr(acc[1]), ptr(acc[2]),
                             ptr(stats), ptr(host), stream_handle(dev)), "zk_ce_labels")
    torch.cuda.synchronize()
    keep = given != -100
    want = [int(keep.sum()), int((keep & ((given < 0) | (given >= 50))).sum())]
    assert host.tolist() == want and stats.tolist() == want
    assert torch.equal(out.cpu(), torch.where(keep, given, -1))
    assert bool((acc[0] == float("-inf")).all()) and not bool(acc[1:3].any())
    run_max, run_sum, target = torch.randn(3, T, generator=g).abs().add(0.5).to(dev)
    m, lse, loss = run_max.clone(), torch.empty(T, device=dev), torch.empty((), device=dev)
    check(lib().zk_ce_finish(ptr(out), T, ptr(m), ptr(run_sum), ptr(target), ptr(stats), ptr(lse),
                             ptr(loss), stream_handle(dev)), "zk_ce_finish")
    ref = run_max.double() + run_sum.double().log()
    assert ((lse.double() - ref).abs() <= 1e-6 * (1 + ref.abs())).all()
    mean = (ref - target.double())[out >= 0].sum().item() / want[0]
    # T terms of O(1), summed in fp32 over 1024 lanes and the groups
    assert abs(loss.item() - mean) <= 2.0 ** -18
    with pytest.raises(ValueError, match="labels must lie in"):
        lm_head_cross_entropy(torch.randn(T, 8, device=dev), torch.randn(50, 8, device=dev), lab)


def test_many_rows_cost_their_bandwidth(dev):
    """The labels of 262144 rows take less than 5 times as long as 8192 (11 us
    against 7; 94 when one workgroup walks them all)."""
    from zorse_amd._abi import check, lib, ptr, stream_handle

    def best(T):
        lab, out = torch.zeros(2, T, dtype=torch.int64, device=dev)
        acc, stats = torch.empty(3, T, device=dev), torch.empty(2, dtype=torch.int64, device=dev)
        host, times = torch.empty(2, dtype=torch.int64, pin_memory=True), []
        for _ in range(6):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            for _ in range(10):
                check(lib().zk_ce_labels(ptr(lab), T, 8, -100, ptr(out), ptr(acc[0]), ptr(acc[1]),
                                         ptr(acc[2]), ptr(stats), ptr(host), stream_handle(dev)),
                      "zk_ce_labels")
            t1.record()
            t1.synchronize()
            times.append(t0.elapsed_time(t1) / 10)
        print(f"labels of {T} rows {min(times) * 1e3:.1f} us", flush=True)
        return min(times)
    assert best(262144) < 5 * best(8192)
