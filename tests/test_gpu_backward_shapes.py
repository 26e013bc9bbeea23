"""Backward kernels at the edges of their work splits, against autograd of the
CPU oracle."""

import pytest
import torch

from oracle import mrsa_oracle as O

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
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
