"""Backward kernels at the edges of their work splits, against autograd of the
CPU oracle."""

import pytest
import torch

from oracle import mrsa_oracle as O

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import mrsa
    from mrsa.route_weights import route_weights_backward

DEV = "cuda:0"


@pytest.mark.parametrize("B,L,C,Hkv,G,K", [
    (1, 1, 3, 1, 1, 1),
    (2, 17, 40, 3, 7, 32),       # workgroups of 16 tokens, the second one partial
    (1, 1200, 960, 4, 8, 24),    # the largest bias held in LDS; lanes past the last slot
    (1, 300, 961, 2, 8, 20),     # beyond it: atomics per slot; slots not in whole groups
    (1, 700, 64, 4, 7, 40),
])
def test_route_weights_backward_splits_vs_oracle(B, L, C, Hkv, G, K):
    print(f"[gpu-case] route weights backward B={B} L={L} C={C} G={G} K={K}", flush=True)
    g = torch.Generator().manual_seed(70 + C)
    Hq = Hkv * G
    scores = torch.randn(B, L, Hq, K, generator=g).bfloat16()
    idx = torch.randint(-1, C, (B, L, Hkv, K), generator=g).int()
    idx[..., 0].clamp_(min=0)  # (autograd of the oracle is NaN at rows with no routed chunk)
    bias = torch.randn(B, C, Hkv, G, generator=g)
    lse = torch.randn(B, L, Hq, generator=g) + 2.0
    g_rw = torch.randn(B, L, Hq, K, generator=g).bfloat16()
    g_lw = torch.randn(B, L, Hq, generator=g).bfloat16()
    off, scl = torch.full((1,), 0.3), torch.full((1,), 1.2)
    ins = [t.double().requires_grad_() for t in (scores, bias, lse)]
    gates = [t.clone().requires_grad_() for t in (off, scl)]
    rw, lw = O.route_weights(ins[0], idx, ins[1], ins[2], gate_offset=gates[0],
                             gate_scale=gates[1])
    want = torch.autograd.grad([rw, lw], ins + gates, [g_rw.to(rw.dtype), g_lw.to(lw.dtype)])
    got = route_weights_backward(
        scores.to(DEV), idx.to(DEV), bias.to(DEV), lse.to(DEV), g_rw.to(DEV), g_lw.to(DEV),
        gate_offset=off.to(DEV), gate_scale=scl.to(DEV))
    # fp32 recomputation of the probabilities: 1e-5 of each gradient's largest
    # term; the sums over rows (bias, gates) also reorder up to B L G K terms
    for name, a, b, rel in (("scores", got[0], want[0], 1e-5), ("bias", got[1], want[1], 1e-4),
                            ("lse", got[2], want[2], 1e-5)):
        a, b = a.double().cpu(), b.double()
        assert (a - b).abs().max() <= rel * max(1.0, float(b.abs().max())), name
    terms = B * L * Hq
    for a, b in ((got[3][1], want[3]), (got[3][0], want[4])):
        assert abs(float(a) - float(b)) <= 1e-5 * terms


@pytest.mark.parametrize("Lq,C,Hkv,G,K,keep,alibi,scale", [
    (1, 1, 1, 1, 1, False, False, 1.0),      # one pair
    (17, 1, 2, 8, 1, False, True, 1.0),      # 17 pairs of one chunk: one past a round of 16
    (257, 1, 1, 4, 1, False, False, 1.0),    # one pair past a work unit: two units are added
    (513, 3, 2, 7, 2, True, False, 1.0),     # keep rows that drop whole chunks
    (130, 5, 1, 5, 3, False, False, 30.0),   # logits past 2^64: the stabilised second pass
    (130, 5, 1, 3, 4, True, True, 30.0),
])
def test_routed_backward_splits_vs_oracle(Lq, C, Hkv, G, K, keep, alibi, scale):
    print(f"[gpu-case] routed backward Lq={Lq} C={C} Hkv={Hkv} G={G} K={K} {keep} {alibi}",
          flush=True)
    g = torch.Generator().manual_seed(90 + Lq + G)
    r = lambda *s: torch.randn(*s, generator=g)
    Hq = Hkv * G
    q, do = (r(1, Lq, Hq, 128) * scale).bfloat16(), r(1, Lq, Hq, 128).bfloat16()
    k, v = r(1, C * 64, Hkv, 128).bfloat16(), r(1, C * 64, Hkv, 128).bfloat16()
    w = torch.rand(1, Lq, Hq, K, generator=g).bfloat16()
    idx = torch.rand(1, Lq, Hkv, max(C, K), generator=g).topk(K, -1).indices.int()
    idx[idx >= C] = -1               # (K > C: lists that end early)
    if C > 1:
        idx[0, 1, 0, :] = 1          # one chunk in every slot
    valid = torch.rand(1, C * 64, generator=g) > 0.1
    if C > 2:
        valid[0, 64:128] = False     # a chunk with no visible key
    tk = None
    if keep:
        tk = torch.rand(1, Lq, Hkv, K, 64, generator=g) > 0.4
        tk[0, ::3, :, 0] = False
        tk = tk.to(torch.int8)
    slope = torch.rand(Hq, generator=g) if alibi else None

    def grads(fn, dev, dtype, **kw):
        ins = [t.to(dev, dtype).requires_grad_() for t in (q, k, v, w)]
        dv = lambda t: None if t is None else t.to(dev)
        out = fn(*ins, idx.to(dev), dv(valid), token_keep=dv(tk), slope=dv(slope), **kw)
        out.backward(do.to(dev, dtype))
        return [t.grad.double().cpu() for t in ins]

    got = grads(lambda *a, **kw: mrsa.HiLS_block_M_head(*a[:5], key_valid=a[5], **kw), DEV,
                torch.bfloat16)
    want = grads(O.selected_attention, "cpu", torch.float32)
    # dS and w P are rounded to bf16 once before the products and the gradients
    # once after (2^-9 each, independent roundings): 2^-8 of a gradient's norm
    # each way bounds both
    for name, a, b in zip(("dq", "dk", "dv", "dw"), got, want):
        assert torch.isfinite(a).all(), name
        assert (a - b).norm() <= 2.0 ** -7 * b.norm() + 1e-6, name


@pytest.mark.parametrize("B,L,Hkv,G,W,inert,odd_rows", [
    (1, 1, 1, 1, 0, 0, False),           # one row: every streamed row past it repeats it
    (1, 10, 2, 7, 4, 0, False),          # 70 rows: a second tile of 6
    (2, 130, 1, 3, 17, 64, False),       # a second key block of 2 keys
    (1, 257, 3, 2, 300, 64, True),       # every row seen; dK / dV in parts
    (1, 333, 2, 5, 40, 0, True),         # waves that skip tiles at both window ends
    (1, 200, 1, 96, 33, 0, False),       # one position spans two tiles
    (1, 1100, 1, 8, 500, 64, True),      # 8 parts
    (1, 33000, 1, 1, 33000, 64, False),  # more key tiles than the inert-key table holds
])
def test_window_backward_streams_and_parts_vs_float64(B, L, Hkv, G, W, inert, odd_rows):
    print(f"[gpu-case] window backward B={B} L={L} Hkv={Hkv} G={G} W={W}", flush=True)
    from mrsa.local_attention import local_attention_autograd, local_attention_backward

    g = torch.Generator().manual_seed(40 + L + G)
    q, do = (torch.randn(B, L, Hkv * G, 128, generator=g).bfloat16() for _ in range(2))
    k, v = (torch.randn(B, L, Hkv, 128, generator=g).bfloat16() for _ in range(2))
    valid = torch.ones(B, L, dtype=torch.bool)
    if odd_rows:
        valid = torch.rand(B, L, generator=g) > 0.1
    if L > 4096:  # (the dense form is too large: one row block's dQ, which reads every key)
        rows = slice(L - 64, L)
    else:
        rows = slice(0, L)
    ref = [t.to(DEV).double().requires_grad_() for t in (q[:, rows], k, v)]
    dead = ~valid.to(DEV)
    i = torch.arange(L, device=DEV)
    if inert:
        dead = dead | ((i + 1) % inert == 0)[None]
    far = (i[rows, None] - i[None]).abs() > W
    parts, lse = [], []
    for h in range(Hkv * G):
        live = (~dead).double()[..., None]
        s = ref[0][:, :, h] @ (ref[1][:, :, h // G] * live).transpose(1, 2) / 128 ** 0.5
        s = s.masked_fill(far, float("-inf"))
        p = torch.softmax(s, -1)
        lse.append(torch.logsumexp(s.detach(), -1))
        parts.append(p @ (ref[2][:, :, h // G] * live))
    out = torch.stack(parts, 2)
    want = torch.autograd.grad(out, ref, do[:, rows].to(DEV).double())
    ins = [t.to(DEV).requires_grad_() for t in (q, k, v)]
    if G <= 8:
        got, _ = local_attention_autograd(*ins, valid.to(DEV), W, inert)
        got = torch.autograd.grad(got, ins, do.to(DEV))
    else:  # (past the forward kernel's heads)
        got = local_attention_backward(*[t.detach() for t in ins], valid.to(DEV),
                                       out.detach().bfloat16(), torch.stack(lse, 2).float(),
                                       do.to(DEV), W, inert)
    # P and dS are rounded to bf16 before their products and the gradients after
    # (2^-9 each, independent); D comes from the bf16 output (2^-9 of |dO| |O|)
    for name, a, b in zip(("dq", "dk", "dv"), got, want):
        a = a[:, rows].double() if name == "dq" else a.double()
        assert torch.isfinite(a).all(), name
        if name == "dq" or L <= 4096:
            assert (a - b).norm() <= 2.0 ** -7 * b.norm() + 2.0 ** -8 * L ** 0.5, name


@pytest.mark.parametrize("C,alibi", [(257, False), (300, True)])
def test_routed_backward_walks_that_join_vs_oracle(C, alibi):
    """Past 256 chunks the dQ walk (and the ALiBi forward) start where other
    walks are."""

    print(f"[gpu-case] routed backward, joined walks C={C} alibi={alibi}", flush=True)
    g = torch.Generator().manual_seed(C)
    Lq, Hkv, G, K = 300, 2, 3, 6
    r = lambda *s: torch.randn(*s, generator=g).bfloat16()
    q, do = r(1, Lq, Hkv * G, 128), r(1, Lq, Hkv * G, 128)
    k, v = r(1, C * 64, Hkv, 128), r(1, C * 64, Hkv, 128)
    w = torch.rand(1, Lq, Hkv * G, K, generator=g).bfloat16()
    idx = torch.rand(1, Lq, Hkv, C, generator=g).topk(K, -1).indices.int()  # any order
    idx[0, 3] = -1
    idx[0, 5, :, 2:] = -1
    idx[0, 10:40, :, 4] = idx[0, 10:40, :, 1]   # a chunk twice
    valid = torch.rand(1, C * 64, generator=g) > 0.1
    slope = torch.rand(Hkv * G, generator=g) if alibi else None

    ref = [t.float().requires_grad_() for t in (q, k, v, w)]
    out = O.selected_attention(*ref, idx, valid, slope=slope)
    want = [out.detach()] + list(torch.autograd.grad(out, ref, do.float()))
    for _ in range(3):           # each launch joins where the one before it ended
        ins = [t.to(DEV).requires_grad_() for t in (q, k, v, w)]
        out = mrsa.HiLS_block_M_head(*ins, idx.to(DEV), key_valid=valid.to(DEV),
                                     slope=None if slope is None else slope.to(DEV))
        got = [out.detach()] + list(torch.autograd.grad(out, ins, do.to(DEV)))
        # the bounds of test_routed_backward_splits_vs_oracle; a repeated chunk's
        # weights are added in bf16 first (2^-9 more)
        for name, a, b in zip(("out", "dq", "dk", "dv", "dw"), got, want):
            a, b = a.double().cpu(), b.double()
            assert torch.isfinite(a).all(), name
            assert (a - b).norm() <= 2.0 ** -7 * b.norm(), name


@pytest.mark.parametrize("keep,alibi", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_routed_backward_ignores_what_excluded_keys_hold(keep, alibi, value):
    """NaN or infinite K rows of invalid keys reach no gradient but dQ (whose
    product dS . K meets them with dS = 0)."""

    print(f"[gpu-case] routed backward, {value} in invalid keys keep={keep} alibi={alibi}",
          flush=True)
    g = torch.Generator().manual_seed(31)
    Lq, C, Hkv, G, K = 70, 4, 2, 3, 3
    r = lambda *s: torch.randn(*s, generator=g).bfloat16()
    q, do = r(1, Lq, Hkv * G, 128), r(1, Lq, Hkv * G, 128)
    k, v = r(1, C * 64, Hkv, 128), r(1, C * 64, Hkv, 128)
    w = torch.rand(1, Lq, Hkv * G, K, generator=g).bfloat16()
    idx = torch.rand(1, Lq, Hkv, C, generator=g).topk(K, -1).indices.int()
    valid = torch.rand(1, C * 64, generator=g) > 0.2
    tk = (torch.rand(1, Lq, Hkv, K, 64, generator=g) > 0.2).to(torch.int8) if keep else None
    slope = torch.rand(Hkv * G, generator=g) if alibi else None

    def grads(kk):
        ins = [t.to(DEV).requires_grad_() for t in (q, kk, v, w)]
        mrsa.HiLS_block_M_head(*ins, idx.to(DEV), key_valid=valid.to(DEV),
                               token_keep=None if tk is None else tk.to(DEV),
                               slope=None if slope is None else slope.to(DEV)
                               ).backward(do.to(DEV))
        return [t.grad.double().cpu() for t in ins]

    want = grads(k)
    bad = k.clone()
    bad[~valid] = value
    got = grads(bad)
    # the same terms in another order, each gradient rounded to bf16 once
    for name, a, b in list(zip(("dq", "dk", "dv", "dw"), got, want))[1:]:
        assert torch.isfinite(a).all(), name
        assert (a - b).norm() <= 2.0 ** -8 * b.norm(), name
