"""Products whose reduction is split over workgroups (zk_gemm_ws): at the
edges of the three tiles it uses, with the last range shorter than the others,
against the float64 product -- within one storage ulp, as a single pass is (at
most 512 fp32 additions of 32-product sums an output, rounding errors far below
the ulp and the floor of 2^-20 of the largest output) --
and with operands inside NaN-filled buffers."""
import pytest
import torch

from tests.test_gpu_gemm_tiles import _run, _view

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b_km", [False, True], ids=["X_Wt", "dY_W"])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8192), (33, 200, 8200), (100, 520, 8192),
                                   (130, 1544, 8200), (257, 1288, 12296), (2046, 1536, 16392)])
def test_split_products(dev, M, N, K, b_km):
    from zorse_amd._abi import dtype_code, lib
    dt = dtype_code(torch.bfloat16)
    assert lib().zk_gemm_workspace(M, N, K, K + 24, 0, N + 24 if b_km else K + 24, int(b_km),
                                   N + 16, -1, dt) > 0
    for dtype in (torch.bfloat16, torch.float16) if M < 2000 else (torch.bfloat16,):
        _run(M, N, K, False, b_km, dtype, dev, res=dtype == torch.float16)


def test_short_workspace_runs_in_one_pass(dev):
    """Too small or misaligned a workspace, or none: the single pass's bits."""
    from zorse_amd._abi import check, dtype_code, lib, ptr, stream_handle
    g = torch.Generator(device=dev).manual_seed(3)
    a = _view(33, 8200, torch.bfloat16, g, dev)
    b = _view(200, 8200, torch.bfloat16, g, dev)
    dt, outs = dtype_code(torch.bfloat16), []
    need = lib().zk_gemm_workspace(33, 200, 8200, a.stride(0), 0, b.stride(0), 0, 200, -1, dt)
    ws = torch.empty(need + 16, dtype=torch.uint8, device=dev)
    for w, n in ((None, 0), (ws, need - 1), (ws[8:], need)):
        out = torch.empty(33, 200, dtype=torch.bfloat16, device=dev)
        check(lib().zk_gemm_ws(ptr(a), a.stride(0), 0, ptr(b), b.stride(0), 0, ptr(out), 200, None,
                               0, 33, 200, 8200, dt, ptr(w) if w is not None else None, n,
                               stream_handle(dev)), "zk_gemm_ws")
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
