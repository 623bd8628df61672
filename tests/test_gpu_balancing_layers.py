"""The load-balancing losses over a model's layers at once: layer counts past
one launch's 32, layers of two shapes, every gradient kernel (lanes filled or
not), chunks of 64 and of 256 tokens, ragged sequences, misaligned inputs.
fp32 data with fp64 sums: loss within 1e-6 of the fp64 oracle, gradients
within 1e-5 of the largest (the fp32 arithmetic of a token's 16 to 256
terms); bf16 gradients within their rounding, 2^-8."""
import pytest
import torch

from moe_amd import _lib, ops
from moe_amd import balancing as Bal
from oracle import balancing_oracle as B

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _layers(shapes, E, dtype, seed, softmax=False):
    g = torch.Generator().manual_seed(seed)
    out = []
    for T in shapes:
        z = torch.randn(T, E, generator=g)
        out.append((torch.softmax(z, -1) if softmax else torch.sigmoid(z)).to(dtype))
    return out, g


def _compare(loss, ref, gin, ref_in, dtype):
    loss.backward()
    ref_g = torch.autograd.grad(ref, ref_in)
    torch.cuda.synchronize()
    assert abs(loss.item() - ref.item()) <= (1e-6 if dtype == torch.float32 else 1e-2) * ref.item()
    for x, rg in zip(gin, ref_g):
        lim = (2.0 ** -8 if dtype == torch.bfloat16 else 1e-5) * rg.abs().max()
        assert (x.grad.double().cpu() - rg).abs().max() <= lim


SEQ = [
    # layers' tokens, sequences, E, K, selected given, dtype
    ((96,) * 33, 2, 64, 6, True, torch.float32),          # two launches
    ((520, 520, 260), 2, 128, 8, True, torch.float32),    # layers of two shapes
    ((2060,) * 3, 4, 128, 4, False, torch.float32),       # 64-token chunks, a ragged last one
    ((16384,) * 16, 1, 128, 4, True, torch.float32),      # 256-token chunks
    ((65,) * 2, 1, 32, 2, False, torch.float32),
    ((300,) * 2, 1, 256, 8, True, torch.bfloat16),
    ((130,) * 2, 2, 100, 4, False, torch.float32),        # lanes partly empty
    ((50,) * 2, 1, 1792, 8, False, torch.float32),
]


@pytest.mark.parametrize("shapes,bsz,E,K,given,dtype", SEQ)
def test_seq_loss_layers(shapes, bsz, E, K, given, dtype):
    print(f"seq loss {len(shapes)} x {shapes[0]} B={bsz} E={E} {dtype}", flush=True)
    layers, g = _layers(shapes, E, dtype, sum(shapes) + E)
    sel = tuple(torch.rand(T, E, generator=g).topk(K, dim=-1).indices for T in shapes)
    ref_in = [x.double().requires_grad_(True) for x in layers]
    ref = B.seq_aux_loss(tuple(ref_in), E, K, bsz, sel if given else None)
    gin = [x.to(DEV).requires_grad_(True) for x in layers]
    loss = Bal.seq_load_balancing_loss_func(
        tuple(gin), E, K, batch_size=bsz,
        selected_experts=tuple(s.to(DEV) for s in sel) if given else None)
    _compare(loss, ref, gin, ref_in, dtype)


SWITCH = [
    ((96,) * 33, 64, 6, torch.float32, False),
    ((520, 260), 128, 8, torch.float32, False),
    ((4096,) * 4, 128, 8, torch.float32, True),
    ((777,) * 2, 100, 3, torch.float32, True),
    ((130,) * 2, 63, 4, torch.float32, False),   # E not a multiple of 4
    ((300,) * 3, 256, 8, torch.bfloat16, False),
    ((40,) * 2, 1792, 8, torch.float32, False),
]


@pytest.mark.parametrize("shapes,E,K,dtype,masked", SWITCH)
def test_switch_loss_layers(shapes, E, K, dtype, masked):
    print(f"switch loss {len(shapes)} x {shapes[0]} E={E} {dtype} masked={masked}", flush=True)
    layers, g = _layers(shapes, E, dtype, sum(shapes) + E, softmax=True)
    mask = (torch.rand(1, shapes[0], generator=g) > 0.3).float() if masked else None
    ref_in = [x.double().requires_grad_(True) for x in layers]
    ref = B.switch_aux_loss(tuple(ref_in), E, K, attention_mask=mask)
    gin = [x.to(DEV).requires_grad_(True) for x in layers]
    loss = Bal.load_balancing_loss_func(tuple(gin), E, K,
                                        attention_mask=mask.to(DEV) if masked else None)
    _compare(loss, ref, gin, ref_in, dtype)


def test_layers_of_odd_alignment():
    """Contiguous [T,E] views that start 4 bytes into their storage."""
    T, E, K = 200, 64, 4
    layers, _ = _layers((T, T), E, torch.float32, 7)
    ref_in = [x.double().requires_grad_(True) for x in layers]
    ref = B.seq_aux_loss(tuple(ref_in), E, K, 1)
    gin = []
    for x in layers:
        v = torch.empty(T * E + 1, device=DEV)[1:].view(T, E)
        v.copy_(x)
        gin.append(v.requires_grad_(True))
    loss = Bal.seq_load_balancing_loss_func(tuple(gin), E, K)
    _compare(loss, ref, gin, ref_in, torch.float32)


def _seq_loss64(p, sel, L, E, K, B):
    """The fp64 loss of moe_amd_seq_aux_loss on L layers that are all p, without
    its scale factors: sum over layers, sequences and experts of counts * mean."""
    T = p.shape[0]
    n = int(_lib.load().moe_amd_seq_aux_loss_workspace_size(L, T, E, B))
    ws = torch.empty(n, device=DEV, dtype=torch.uint8)
    out = torch.empty(L * B * E + 1, device=DEV, dtype=torch.float64)
    loss = torch.empty((), device=DEV)
    ops._call("moe_amd_seq_aux_loss", Bal._ptr_array([p] * L), Bal._ptr_array([sel] * L), L, 0, T, E,
              K, B, 1.0, 1.0, 1.0, ws.data_ptr(), n, out.data_ptr(), out[-1:].data_ptr(),
              loss.data_ptr(), ops._stream(p))
    return out[-1].item()


@pytest.mark.parametrize("E", [64, 256, 320])  # 8 and 16 lanes per token, a wave per token
@pytest.mark.parametrize("L", [1, 16, 128])
def test_sums_are_fp64_beyond_16_tokens(E, L):
    """Expert 0 gets 1 from every 256th token and 2^-29 from the others, which
    an fp32 sum that holds a 1 loses.  At most the 15 other tokens of such a
    token's lane group may be added to it in fp32."""
    print(f"sums E={E} L={L}", flush=True)
    T, tiny = 16384, 2.0 ** -29
    p = torch.zeros(T, E, device=DEV)
    p[:, 0] = tiny
    p[::256, 0] = 1.0
    ones = T // 256
    want, limit = ones + (T - ones) * tiny, 15 * ones * tiny
    _, loss = Bal._switch_loss(E, 1, None, None, *[p] * L)  # = E * sums[0] / (L T)
    assert abs(loss.item() * T / E - want) <= limit
    assert abs(Bal.topk_stats(p, 1)[1][0].item() - want) <= limit
    p[:, 1] = 1.0  # row sums of 1 (in fp32)
    p[::256, 1] = 0.0
    sel = torch.zeros(T, 1, device=DEV, dtype=torch.int64)
    assert abs(_seq_loss64(p, sel, L, E, 1, 1) / L - want) <= limit  # counts T times mean


@pytest.mark.parametrize("E,K", [(32, 2), (64, 6), (128, 4), (256, 8)])
def test_seq_gradient_inner_product_in_fp64(E, K):
    """2-norm distance of the gradient from 64 bits: that of the formula with
    fp32 row sums (as a tree) and quotients but an fp64 inner product, within
    5% for another order of the row sums.  An fp32 inner product is 40% off."""
    print(f"seq gradient E={E}", flush=True)
    B_, S, L = 8, 1024, 2
    g = torch.Generator(device=DEV).manual_seed(E)
    layers = [torch.sigmoid(torch.randn(B_ * S, E, generator=g, device=DEV)).requires_grad_(True)
              for _ in range(L)]
    sel = [p.detach().topk(K, dim=-1).indices for p in layers]
    Bal.seq_load_balancing_loss_func(tuple(layers), E, K, B_, tuple(sel)).backward()
    got = emulated = 0.0
    for p, s in zip(layers, sel):
        p32, p64 = p.detach(), p.detach().double()
        f = torch.zeros_like(p64).scatter_(1, s, 1.0).reshape(B_, S, E).sum(1) * (E / (K * S))
        c = (f / (L * B_ * S)).repeat_interleave(S, dim=0)
        n64 = p64.sum(-1, keepdim=True) + 1e-20
        want = (c - (c * p64 / n64).sum(-1, keepdim=True)) / n64
        n32 = p32
        while n32.shape[1] > 1:
            n32 = n32[:, 0::2] + n32[:, 1::2]
        em = (c - (c * (p32 / n32).double()).sum(-1, keepdim=True)).float() / n32
        got += float((p.grad.double() - want).square().sum())
        emulated += float((em.double() - want).square().sum())
    assert got <= 1.05 ** 2 * emulated


def test_switch_gradient_of_fp64_layers_keeps_fp64_upstream():
    """An upstream gradient past fp32's range, on layers whose loss is fp64."""
    layers, _ = _layers((64, 64), 32, torch.float32, 3, softmax=True)
    grads = []
    for up in (1.0, 2.0 ** 130):
        gin = [x.to(DEV, torch.float64).requires_grad_(True) for x in layers]
        loss = Bal.load_balancing_loss_func(tuple(gin), 32, 4)
        assert loss.dtype == torch.float64
        loss.backward(torch.tensor(up, dtype=torch.float64, device=DEV))
        grads.append([x.grad for x in gin])
    for a, b in zip(*grads):
        assert a.abs().max() > 0 and torch.equal(a * 2.0 ** 130, b)


@pytest.mark.parametrize("T,Bz,E,K,given,dtype", [
    (520, 2, 128, 8, True, torch.float32), (300, 1, 64, 6, False, torch.float32),
    (260, 4, 256, 8, True, torch.bfloat16), (130, 2, 100, 4, False, torch.float32),
    (96, 2, 1792, 8, True, torch.float32),
])
def test_one_layer_entry_points_match_whole_model_ones(T, Bz, E, K, given, dtype):
    """moe_amd_seq_stats, moe_amd_seq_aux_backward and moe_amd_switch_aux_backward
    against the whole-model entry points with one layer: the coefficients (sums
    of whole numbers) and the gradients bit for bit, the loss to fp64 rounding."""
    print(f"one layer T={T} B={Bz} E={E} {dtype}", flush=True)
    (p,), g = _layers((T,), E, dtype, T + E)
    p, code, lib = p.to(DEV), ops._dtype_code(dtype), _lib.load()
    sel = torch.rand(T, E, generator=g).topk(K, dim=-1).indices.to(DEV) if given else None
    st, f64 = ops._stream(p), dict(device=DEV, dtype=torch.float64)
    sel_ptr = sel.data_ptr() if given else None
    n = int(lib.moe_amd_seq_stats_workspace_size(T, E, Bz))
    ws, counts, mean = torch.empty(n, device=DEV, dtype=torch.uint8), torch.empty(Bz, E, **f64), \
        torch.empty(Bz, E, **f64)
    ops._call("moe_amd_seq_stats", p.data_ptr(), code, sel_ptr, T, E, K, Bz, ws.data_ptr(), n,
              counts.data_ptr(), mean.data_ptr(), st)
    n = int(lib.moe_amd_seq_aux_loss_workspace_size(1, T, E, Bz))
    ws = torch.empty(n, device=DEV, dtype=torch.uint8)
    coef, loss64 = torch.empty(Bz, E, **f64), torch.empty((), **f64)
    loss, up = torch.empty((), device=DEV), torch.ones((), device=DEV)
    ops._call("moe_amd_seq_aux_loss", Bal._ptr_array([p]), Bal._ptr_array([sel]), 1, code, T, E, K, Bz,
              0.5, 0.25, 2.0, ws.data_ptr(), n, coef.data_ptr(), loss64.data_ptr(), loss.data_ptr(), st)
    assert torch.equal(coef, counts * 0.5 * 0.25)
    want = float((counts * 0.5 * mean).sum() * 2.0)
    assert abs(loss64.item() - want) <= 1e-13 * want
    one, all_ = torch.empty_like(p), torch.empty_like(p)
    ops._call("moe_amd_seq_aux_backward", p.data_ptr(), code, coef.data_ptr(), T, E, Bz, one.data_ptr(),
              st)
    ops._call("moe_amd_seq_aux_loss_backward", Bal._ptr_array([p]), 1, code, coef.data_ptr(),
              up.data_ptr(), T, E, Bz, Bal._ptr_array([all_]), st)
    assert torch.equal(one, all_) and bool(one.any())
    w = torch.rand(T, generator=g).to(DEV)
    for tok_w in (None, w):
        ptr = tok_w.data_ptr() if tok_w is not None else None
        ops._call("moe_amd_switch_aux_backward", coef.data_ptr(), ptr, T, E, code, one.data_ptr(), st)
        ops._call("moe_amd_switch_aux_loss_backward", coef.data_ptr(), up.data_ptr(), ptr, 1, T, E, code,
                  Bal._ptr_array([all_]), st)
        assert torch.equal(one, all_)
        want = coef[0].float()[None] * (tok_w[:, None] if tok_w is not None else 1.0)
        assert torch.equal(one, want.expand(T, E).to(dtype))
