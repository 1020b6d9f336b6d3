"""The two passes that rotate head dims other than 64 and 128 (position-major, and
the general one for few heads at many positions) write the same bytes, and few
heads do not cost what many do."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _tables(n, half, dev):
    ang = torch.rand(n, half, generator=torch.Generator().manual_seed(1)).to(dev) * 6.28
    return ang.cos(), ang.sin()


@pytest.mark.parametrize("inter", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,H", [(16, 16), (100, 3), (252, 2)])
def test_few_heads_are_rotated_as_many(dev, d, H, dtype, inter):
    """All heads at once (a wavefront's work or more a position) and each by
    itself."""
    from zorse_amd import kernels as K
    S = 331
    q = torch.randn(1, S, H, d, generator=torch.Generator().manual_seed(d)).to(dtype).to(dev)
    cos, sin = _tables(S, d // 2, dev)
    many, one = q.clone(), q.clone()
    K.rope_(many, None, cos, sin, interleaved=inter)
    for h in range(H):
        K.rope_(one[:, :, h:h + 1], None, cos, sin, interleaved=inter)
    assert torch.equal(many, one)


def test_one_head_costs_less_than_sixteen(dev):
    """At 65536 positions of 16: 7 us against 35 (35 when a position costs a
    workgroup whatever it holds)."""
    from zorse_amd import kernels as K
    cos, sin = _tables(65536, 8, dev)

    def best(H):
        q = torch.randn(1, 65536, H, 16, device=dev).bfloat16()
        K.rope_(q, None, cos, sin)
        times = []
        for _ in range(5):
            t0, t1 = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            t0.record()
            for _ in range(10):
                K.rope_(q, None, cos, sin)
            t1.record()
            t1.synchronize()
            times.append(t0.elapsed_time(t1))
        return min(times)
    assert best(1) < 0.7 * best(16)


def test_more_positions_than_one_grid_dimension(dev):
    """2^24 positions (2^32 threads of the position-major pass, past what a launch
    holds) of 64 heads of 4: the general pass, every position's rotation."""
    from zorse_amd import kernels as K
    S, H, d = 1 << 24, 64, 4
    print(f"rope {S} positions of {H} x {d}", flush=True)
    base = torch.randn(1, 8, H, d, generator=torch.Generator().manual_seed(2)).bfloat16().to(dev)
    cos, sin = _tables(8, d // 2, dev)
    want = base.clone()
    K.rope_(want, None, cos, sin)
    q = base.expand(S // 8, 8, H, d).reshape(1, S, H, d)
    K.rope_(q, None, cos, sin, positions=torch.arange(S, device=dev) % 8)
    for part in q.view(S // 8, 8, H, d).split(1 << 17):
        assert bool((part == want).all())
