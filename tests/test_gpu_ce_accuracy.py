"""The forward cross-entropy chunk's exponentials: as accurate as the library's
expf, and right at the ends of the range."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _chunk(x):
    from zorse_amd._abi import check, dtype_code, lib, ptr, stream_handle
    rows, cols = x.shape
    labels = torch.zeros(rows, dtype=torch.int64, device=x.device)
    run_max = torch.full((rows,), float("-inf"), device=x.device)
    run_sum, target = torch.zeros(2, rows, device=x.device)
    check(lib().zk_ce_fwd_chunk(ptr(x), rows, cols, cols, ptr(labels), 0, ptr(run_max),
                                ptr(run_sum), ptr(target), dtype_code(x.dtype),
                                stream_handle(x.device)), "zk_ce_fwd_chunk")
    return run_max.double().cpu(), run_sum.double().cpu()


def test_exponentials_are_within_an_ulp(dev):
    """640 e^-t + 1 per thread, t from 5.6 to 8, with nothing else rounded: each
    thread counts 640 logits of -t exactly and rescales the count when it meets
    its 0 (the rest of that sweep is -inf); the 256 threads' equal sums double
    exactly.  Bound: e^-t within an ulp and a half (3 2^-24) of it, at most 0.7 of
    the sum, and one rounding of the sum.  2^(t log2 e) of the rounded product is
    off by 3.1e-7 here."""
    rows, sweeps = 512, 20
    t = torch.linspace(5.6, 8.0, rows, dtype=torch.float64).float()
    x = torch.full((rows, (sweeps + 1) * 8192), float("-inf"), device=dev)
    x[:, :sweeps * 8192] = -t.to(dev)[:, None]
    x[:, sweeps * 8192:].view(rows, 4, 256, 8)[:, 3, :, 7] = 0
    run_max, run_sum = _chunk(x)
    assert bool((run_max == 0).all())
    ref = 256 * (1 + 32 * sweeps * torch.exp(-t.double()))
    assert ((run_sum - ref) / ref).abs().max().item() <= (0.7 * 3 + 1) * 2.0 ** -24


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("cols", [2048, 9000])
def test_range_ends(dev, cols, dtype):
    """-inf logits add nothing, wherever they are; an infinity or NaN makes the
    sum NaN; logits at the ends of the type's range stay in it."""
    big = torch.finfo(dtype).max
    x = torch.randn(6, cols, generator=torch.Generator().manual_seed(cols)).to(dtype)
    x[0, ::2] = float("-inf")
    x[1, :cols - 1] = float("-inf")
    x[2, 7], x[2, 8:] = big, -big
    x[3, 1:] = -big
    x[4, 100] = float("nan")
    x[5, cols - 1] = float("inf")
    run_max, run_sum = _chunk(x.to(dev))
    got, ref = run_max + run_sum.log(), torch.logsumexp(x.double(), 1)
    ok = [0, 1, 2, 3]
    assert torch.equal(run_max[ok], x[ok].double().max(1).values)
    assert ((got - ref)[ok].abs() <= 1e-6 * ref[ok].abs()).all()
    assert bool(run_sum[[4, 5]].isnan().all())
