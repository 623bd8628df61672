"""Combine and gather backward around the token counts where a row's pieces go
to waves of their own (1024, 8192) and for rows of 1, 2, 3 and more pieces of
1 KB: a token's result is, bit for bit, that of a call on the first 64 tokens."""
import pytest
import torch

from moe_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("K", [3, 8, 20])  # 20: the kernel for any K
@pytest.mark.parametrize("H,dtype", [(512, torch.bfloat16), (512, torch.float32),
                                     (1344, torch.bfloat16), (1344, torch.float32)])
def test_rows_in_pieces(K, H, dtype):
    print(f"row pieces K={K} H={H} {dtype}", flush=True)
    E, most, few = 32, 8193, 64
    g = torch.Generator(device=DEV).manual_seed(H + K)
    idx = torch.rand(most, E, generator=g, device=DEV).topk(K, dim=-1).indices
    rows = torch.randn(most * K, H, generator=g, device=DEV).to(dtype)  # of (token, k)
    w = torch.rand(most, K, generator=g, device=DEV)
    add = torch.randn(most, H, generator=g, device=DEV).to(dtype)

    def run(T):
        plan = ops.permute(idx[:T].contiguous(), E)
        y = rows[plan.row_src.long()]
        return (ops.combine(y, plan, w[:T]), ops.gather_backward(y, plan),
                ops.gather_backward(y, plan, addend=add[:T]))

    want = run(few)
    ref = (rows[:few * K].double().view(few, K, H) * w[:few, :, None].double()).sum(1)
    lim = 2.0 ** -7 if dtype == torch.bfloat16 else (K + 2) * 2.0 ** -24
    mags = (rows[:few * K].double().abs().view(few, K, H) * w[:few, :, None].double()).sum(1)
    assert bool(((want[0].double() - ref).abs() <= lim * mags).all())
    for T in (1024, 1025, 8192, most):
        for a, b in zip(run(T), want):
            assert torch.equal(a[:few], b)
