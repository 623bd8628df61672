"""The token-grouped GEMMs on tiles that hold 1, 2, 3 or 4 of their 64-row
units: experts with row counts at every edge of a unit and of a tile, where
the host picks 256-row tiles (512 rows per expert and more) and where the
plan picks the height.

Bounds: gate_up, y and d_xs are fp32 sums of K exact products rounded once to
bf16: |error| <= 2^-8 |value| + K 2^-23 sum |a||b|.  The fused backward rounds
three times in a row (silu, products, result): rows within 3 * 2^-8 of the
fp64 ones in 2-norm."""
import pytest
import torch

from moe_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
EDGES = [1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 319, 320, 321, 0, 384, 385,
         449, 511, 512, 513, 577]


def _close(got, want, mags, K):
    err = (got.double() - want).abs()
    assert bool((err <= want.abs() * 2.0 ** -8 + K * 2.0 ** -23 * mags + 1e-30).all())


@pytest.mark.parametrize("more", [0, 512])
def test_partial_tiles(more):
    H, I = 192, 320
    counts = [c + (more if c else 0) for c in EDGES]
    E, T = len(counts), sum(counts)
    print(f"row units: {E} experts, {T} rows", flush=True)
    g = torch.Generator(device=DEV).manual_seed(3)
    ids = torch.repeat_interleave(torch.arange(E, device=DEV),
                                  torch.tensor(counts, device=DEV))
    ids = ids[torch.randperm(T, generator=g, device=DEV)].reshape(T, 1)
    plan = ops.permute(ids, E)

    def rnd(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g, device=DEV) * scale).bfloat16()

    x, dout, act, dgu = rnd(T, H), rnd(T, H), rnd(T, I), rnd(T, 2 * I)
    w1, w2 = rnd(E, 2 * I, H, scale=0.1), rnd(E, H, I, scale=0.1)
    w = torch.rand(T, 1, generator=g, device=DEV) + 0.5
    gu, a = ops.gemm_gate_up_swiglu(x, plan, w1)
    y = ops.gemm_down(act, plan, w2)
    dxs = ops.gemm_gate_up_backward_dx(dgu, plan, w1)
    d_gu, act_w, dw = ops.gemm_down_backward_fused(dout, plan, w2, gu, w)
    torch.cuda.synchronize()
    src, off = plan.row_src.long(), plan.offsets.tolist()
    for e in range(E):
        r = slice(off[e], off[e + 1])
        if off[e] == off[e + 1]:
            continue
        t = src[r]
        xe, a1, a2 = x[t].double(), w1[e].double(), w2[e].double()
        _close(gu[r], xe @ a1.T, xe.abs() @ a1.abs().T, H)
        _close(y[r], act[r].double() @ a2.T, act[r].double().abs() @ a2.abs().T, I)
        _close(dxs[r], dgu[r].double() @ a1, dgu[r].double().abs() @ a1.abs(), 2 * I)
        gate, up = gu[r].double().split(I, dim=1)
        sg = torch.sigmoid(gate)
        ar = gate * sg * up
        da = dout[t].double() @ a2
        want = {"act": (a[r], ar), "act_w": (act_w[r], w[t] * ar),
                "d_gate_up": (d_gu[r], w[t] * torch.cat(
                    [da * up * sg * (1 + gate * (1 - sg)), da * gate * sg], dim=1))}
        for name, (got, ref) in want.items():
            rel = (got.double() - ref).norm(dim=1) / ref.norm(dim=1)
            assert float(rel.max()) <= 3 * 2.0 ** -8, (name, e)
        # <d_out, y> per row: bf16 act and g, fp32 sums
        dot, mag = (da * ar).sum(1), (da.abs() * ar.abs()).sum(1)
        assert bool(((dw[t, 0].double() - dot).abs() <= 4 * 2.0 ** -9 * mag).all())
