"""The fp32 grouped GEMMs (bf16 matrix cores, three-term split) against fp64.

Bound per element: with K the contracted length and u = 2^-24, the kernel adds
ceil(K/16) MFMA results of at most 16 exact products hi*hi into one fp32
accumulator and five times as many small ones, worth at most 2^-7 of |a||b|,
into another, every MFMA with at most 17 roundings; it leaves out products of
at most 2^-24 of |a||b| and adds the two accumulators.  To first order |error|
<= (18 * ceil(K/16) + 3) * u * sum |a||b|.

That bound grows with K and does not see a lost third term, so the 2-norm
errors are also held against a chain of fp32 fused multiply-adds over the same
terms (test_f32_gemms_no_further_than_fp32_chain)."""
import pytest
import torch

from moe_amd import experts_forward, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bound(K):
    return (18 * ((K + 15) // 16) + 3) * 2.0 ** -24


def _plan(T, E, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    idx = torch.rand(T, E, generator=g, device=DEV).topk(K, dim=-1).indices
    return ops.permute(idx, E), g


def _wide(g, *shape):
    """N(0,1) values over 2^-12 .. 2^12, so that all three terms matter."""
    x = torch.randn(*shape, generator=g, device=DEV)
    return x * torch.exp2(torch.randint(-12, 13, shape, generator=g, device=DEV).float())


def _check(got, want, mags, K):
    assert torch.isfinite(got).all()
    err = (got.double() - want).abs()
    assert bool((err <= _bound(K) * mags + 1e-300).all()), float((err / mags.clamp_min(1e-300)).max())


CASES = [
    (1, 64, 1, 1, 64),         # one row, smallest H and I
    (128, 64, 1, 1, 128),      # one full tile
    (129, 320, 3, 2, 64),      # tile remainders in rows and columns
    (777, 256, 16, 4, 192),    # ragged experts
    (2048, 1024, 16, 4, 768),  # the XS layer
    (40, 128, 64, 6, 320),     # tiny groups, empty experts
]


@pytest.mark.parametrize("T,H,E,K,I", CASES)
def test_f32_gemms_against_fp64(T, H, E, K, I):
    print(f"f32 split T={T} H={H} E={E} K={K} I={I}", flush=True)
    plan, g = _plan(T, E, K, T + E)
    S = T * K
    tok = plan.row_src.long() // K
    off = plan.offsets.tolist()
    x, w1, w2 = _wide(g, T, H), _wide(g, E, 2 * I, H), _wide(g, E, H, I)
    act, dgu, dy = _wide(g, S, I), _wide(g, S, 2 * I), _wide(g, S, H)
    gu, _ = ops.gemm_gate_up_swiglu(x, plan, w1)
    y = ops.gemm_down(act, plan, w2)
    dxs = ops.gemm_gate_up_backward_dx(dgu, plan, w1)
    dw2 = ops.gemm_down_backward_dw(dy, act, plan, w2.shape)
    dw1 = ops.gemm_gate_up_backward_dw(dgu, x, plan, w1.shape)
    torch.cuda.synchronize()
    for e in range(E):
        r = slice(off[e], off[e + 1])
        n = off[e + 1] - off[e]
        if n == 0:
            assert not dw1[e].any() and not dw2[e].any()
            continue
        xe = x[tok[r]].double()
        a1, a2, ac, dg, d = (t.double() for t in (w1[e], w2[e], act[r], dgu[r], dy[r]))
        _check(gu[r], xe @ a1.T, xe.abs() @ a1.abs().T, H)
        _check(y[r], ac @ a2.T, ac.abs() @ a2.abs().T, I)
        _check(dxs[r], dg @ a1, dg.abs() @ a1.abs(), 2 * I)
        _check(dw2[e], d.T @ ac, d.abs().T @ ac.abs(), n)
        _check(dw1[e], dg.T @ xe, dg.abs().T @ xe.abs(), n)


MODES = ["gate_up", "down", "down_dx", "gate_up_dx", "down_dw", "gate_up_dw"]


def _operands(mode, K, seed, nonzero=0):
    """Operands a [M,K], b [N,K] of one expert, N(0,1); with `nonzero`, a keeps
    that many terms per row.  M, N have tile remainders."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    M, N = {"down_dw": (192, 64), "gate_up_dw": (384, 64), "gate_up": (130, 384)}.get(mode, (130, 192))
    a, b = torch.randn(M, K, generator=g, device=DEV), torch.randn(N, K, generator=g, device=DEV)
    if nonzero and nonzero < K:
        at = torch.rand(M, K, generator=g, device=DEV).topk(nonzero, dim=-1).indices
        a = torch.zeros_like(a).scatter_(1, at, a.gather(1, at))
    return a, b


def _product(mode, a, b):
    """a b^T by one of the six GEMMs, for one expert."""
    rows = a.shape[1] if mode.endswith("_dw") else a.shape[0]
    plan = ops.permute(torch.zeros(rows, 1, dtype=torch.int64, device=DEV), 1)
    if mode == "gate_up":
        return ops.gemm_gate_up_swiglu(a, plan, b[None].contiguous())[0]
    if mode == "down":
        return ops.gemm_down(a, plan, b[None].contiguous())
    if mode == "gate_up_dx":
        return ops.gemm_gate_up_backward_dx(a, plan, b.T[None].contiguous())
    if mode == "down_dx":  # at gate = 64 and up = 1 the tail gives d_gate = d_act, d_up = 64 d_act
        gu = torch.ones(rows, 2 * b.shape[0], device=DEV)
        gu[:, :b.shape[0]] = 64.0
        d = ops.gemm_down_backward_dx_dswiglu(a, plan, b.T[None].contiguous(), gu)
        assert torch.equal((d[:, :b.shape[0]] * 64).nan_to_num(), d[:, b.shape[0]:].nan_to_num())
        return d[:, :b.shape[0]]
    at, bt = a.T.contiguous(), b.T.contiguous()
    if mode == "down_dw":
        return ops.gemm_down_backward_dw(at, bt, plan, (1, a.shape[0], b.shape[0]))[0]
    return ops.gemm_gate_up_backward_dw(at, bt, plan, (1, a.shape[0], b.shape[0]))[0]


def _chain32(a, b):
    """a b^T as a chain of fp32 fused multiply-adds in k order."""
    acc = torch.zeros(a.shape[0], b.shape[0], device=DEV)
    for k in range(a.shape[1]):
        acc = (acc.double() + a[:, k, None].double() * b[None, :, k].double()).float()
    return acc


def _terms(x):
    hi = x.bfloat16().float()
    mid = (x - hi).bfloat16().float()
    return mid.double(), (x - hi - mid).double()


def _left_out(a, b, eight):
    """The part of a b^T that the kernel leaves out (eight of nine products, or six)."""
    (am, al), (bm, bl) = _terms(a), _terms(b)
    d = al @ bl.T
    return d if eight else d + am @ bl.T + al @ bm.T


CHAIN = ([(m, K, nz) for m in MODES[:4] for K, nz in [(128, 1), (128, 2), (128, 4), (256, 16),
                                                      (768, 64), (128, 128), (768, 768)]]
         + [(m, K, nz) for m in MODES[4:] for K, nz in [(1, 1), (2, 2), (3, 3), (32, 32), (33, 33),
                                                        (200, 4), (200, 200)]])


@pytest.mark.parametrize("mode,K,nonzero", CHAIN)
def test_f32_gemms_no_further_than_fp32_chain(mode, K, nonzero):
    """2-norm distance from 64 bits: that of a chain of fp32 fused multiply-adds
    over the same terms, with what the kernel leaves out added in quadrature
    (and 1% for what rounds below that)."""
    print(f"f32 split {mode} K={K} nonzero={nonzero}", flush=True)
    a, b = _operands(mode, K, 7 * K + nonzero, nonzero)
    want = a.double() @ b.double().T
    err = (_product(mode, a, b).double() - want).norm()
    chain = (_chain32(a, b).double() - want).norm()
    left = _left_out(a, b, mode.endswith("_dw") and K <= 32).norm()
    assert float(err) <= 1.01 * float((chain ** 2 + left ** 2).sqrt()), float(err / want.norm())


def test_f32_down_dx_dswiglu_tail():
    """dX + dSwiGLU on ordinary gates, no further from 64 bits than the same
    formulas in fp32 on the fp32 chain's d_act."""
    T, H, I = 200, 192, 128
    g = torch.Generator(device=DEV).manual_seed(4)
    dy, w2 = torch.randn(T, H, generator=g, device=DEV), torch.randn(H, I, generator=g, device=DEV)
    gu = torch.randn(T, 2 * I, generator=g, device=DEV) * 3
    plan = ops.permute(torch.zeros(T, 1, dtype=torch.int64, device=DEV), 1)

    def tail(da, gu):
        gate, up = gu.split(I, dim=1)
        s = torch.sigmoid(gate)
        return torch.cat([da * up * s * (1 + gate * (1 - s)), da * gate * s], dim=1)

    want = tail(dy.double() @ w2.double(), gu.double())
    err = (ops.gemm_down_backward_dx_dswiglu(dy, plan, w2[None], gu).double() - want).norm()
    assert float(err) <= float((tail(_chain32(dy, w2.T), gu).double() - want).norm())


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("ea,eb", [(-112, 0), (-120, 0), (-128, 20), (-140, 40), (50, -140),
                                   (-62, -62), (100, -100), (110, -90), (60, 60)])
def test_f32_gemms_magnitudes(mode, ea, eb):
    """Operands near 2^ea and 2^eb, subnormal ones among them: as far from 64
    bits as at 1."""
    print(f"f32 split {mode} 2^{ea} x 2^{eb}", flush=True)
    a, b = _operands(mode, 256, 3)
    a = torch.ldexp(a.double(), torch.tensor(ea, device=DEV)).float()
    b = torch.ldexp(b.double(), torch.tensor(eb, device=DEV)).float()
    want = a.double() @ b.double().T
    err = (_product(mode, a, b).double() - want).norm()
    assert float(err / want.norm()) <= float((_chain32(a, b).double() - want).norm() / want.norm())


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan"), 3.4e38])
def test_f32_gemms_nonfinite(bad):
    """A value that is not finite (or overflows as bf16) reaches exactly the
    elements that the plain fp32 product gives it, with their infinities and
    NaNs, and the rest of its tile keeps the fp32 accuracy."""
    print(f"f32 split non-finite {bad}", flush=True)
    T, H, I = 200, 128, 192
    plan = ops.permute(torch.zeros(T, 1, dtype=torch.int64, device=DEV), 1)
    g = torch.Generator(device=DEV).manual_seed(5)
    act = torch.randn(T, I, generator=g, device=DEV)
    w2 = torch.randn(1, H, I, generator=g, device=DEV) * 0.25
    act[3, 17], act[150, 0] = bad, bad
    w2[0, 70, 5] = bad
    w2[0, 10, 17] = 0.0  # inf * 0 = NaN at (3, 10)
    y = ops.gemm_down(act, plan, w2)
    torch.cuda.synchronize()
    want = act.double() @ w2[0].double().T
    big = want.abs() > 3.4028235677973366e38  # beyond fp32
    fin = torch.isfinite(want) & ~big
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    assert torch.equal(torch.isinf(y), torch.isinf(want) | big)
    assert torch.equal(y[torch.isinf(y)] > 0, want[torch.isinf(y)] > 0)
    mags = act.double().abs() @ w2[0].double().abs().T
    err = (y.double() - want).abs()[fin]
    # elements taken from the fp32 MFMA: one rounding per two products
    assert bool((err <= max(_bound(I), I * 2.0 ** -24) * mags[fin]).all())


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("bad", [float("inf"), float("nan"), -3.4e38])
def test_f32_gemms_nonfinite_stays_in_its_rows(mode, bad):
    """In every GEMM: the elements of a non-finite (or bf16-overflowing) value's
    row and column are the fp32 product's, all others of the tile keep the bits
    that they have without it."""
    print(f"f32 split {mode} non-finite {bad}", flush=True)
    a, b = _operands(mode, 256, 17)
    clean = _product(mode, a, b)
    a[3, 17], a[125, 255] = bad, bad
    b[40, 5] = bad
    b[10, 17] = 0.0  # inf * 0 = NaN at (3, 10)
    got = _product(mode, a, b)
    want = a.double() @ b.double().T
    big = want.abs() > 3.4028235677973366e38  # beyond fp32
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want) | big)
    assert torch.equal(got[torch.isinf(got)] > 0, want[torch.isinf(got)] > 0)
    fin = torch.isfinite(got)
    mags = a.double().abs() @ b.double().abs().T
    assert bool(((got.double() - want).abs()[fin] <= 256 * 2.0 ** -24 * mags[fin]).all())
    rows = [i for i in range(a.shape[0]) if i not in (3, 125)]
    cols = [i for i in range(b.shape[0]) if i not in (10, 40)]
    assert torch.equal(got[rows][:, cols], clean[rows][:, cols])


def test_f32_layer_gradients_against_fp64():
    T, H, E, K, I = 513, 192, 8, 2, 128
    g = torch.Generator(device=DEV).manual_seed(9)
    x = torch.randn(T, H, generator=g, device=DEV)
    w1 = torch.randn(E, 2 * I, H, generator=g, device=DEV) * 0.1
    w2 = torch.randn(E, H, I, generator=g, device=DEV) * 0.1
    p, idx = torch.softmax(torch.randn(T, E, generator=g, device=DEV), -1).topk(K, dim=-1)
    dout = torch.randn(T, H, generator=g, device=DEV)
    leaves = [t.clone().requires_grad_(True) for t in (x, p, w1, w2)]
    out = experts_forward(leaves[0], idx, *leaves[1:])
    out.backward(dout)
    l64 = [t.double().requires_grad_(True) for t in (x, p, w1, w2)]
    ref = torch.zeros(T, H, dtype=torch.float64, device=DEV)
    for e in range(E):
        t, k = (idx == e).nonzero(as_tuple=True)
        gate, up = (l64[0][t] @ l64[2][e].T).split(I, dim=1)
        y = (torch.nn.functional.silu(gate) * up) @ l64[3][e].T
        ref = ref.index_add(0, t, y * l64[1][t, k][:, None])
    ref.backward(dout.double())
    for got, want in [(out, ref)] + [(a.grad, b.grad) for a, b in zip(leaves, l64)]:
        # three contractions of at most 256 terms, each no further than a chain of fp32
        # multiply-adds (2.9e-7 at 256 terms), in quadrature, and the fp32 tail's roundings
        assert float((got.detach().double() - want.detach()).norm() / want.detach().norm()) < 6e-7
