"""Route scoring and top-k at the edges of its kernels' ranges (16-chunk tiles,
64 / 128 / 256-chunk instances, 16 or 32 queries per workgroup, the scan path's
16- and 64-chunk stages) against the CPU oracle."""

import pytest
import torch

from oracle import mrsa_oracle as O

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import mrsa
    from mrsa.sparse_attention import kv_fragments, selected_attention_launch
    from mrsa.topk import route_topk_launch

DEV = "cuda:0"
NEAR_TIE = 1e-5


@pytest.mark.parametrize("B,L,C,Hkv,G,topk", [
    (1, 1, 1, 1, 7, 8),            # one row, one chunk: slots past the picks are -1
    (1, 17, 16, 2, 8, 16),
    (2, 33, 64, 4, 7, 32),
    (1, 4100, 64, 4, 4, 32),       # 32 queries per workgroup, last one partial
    (1, 4097, 65, 4, 7, 32),
    (1, 31, 128, 1, 1, 64),
    (1, 130, 129, 3, 7, 20),       # a topk with no 16-byte output rows
    (1, 50, 255, 2, 5, 32),
    (1, 1025, 257, 4, 7, 32),      # scan path: C = 1 mod 16 and 64
    (2, 683, 304, 3, 3, 24),
    (1, 4099, 320, 1, 8, 64),
    (1, 4097, 2049, 1, 2, 24),     # one chunk past the pick's 32-per-lane instance
    (2, 2050, 4096, 1, 1, 64),     # the most chunks
])
def test_route_topk_tile_edges_vs_oracle(B, L, C, Hkv, G, topk):
    print(f"[gpu-case] route tile edges B={B} L={L} C={C} Hkv={Hkv} G={G} K={topk}", flush=True)
    g = torch.Generator().manual_seed(1000 + L + C)
    q5 = torch.randn(B, L, Hkv, G, 128, generator=g).bfloat16()
    lmk = (0.5 * torch.randn(B, C, Hkv * G, 128, generator=g)).bfloat16()
    lse4 = torch.randn(B, L, Hkv, G, generator=g) + 3.0
    bias4 = torch.randn(B, C, Hkv, G, generator=g)
    drop = (torch.rand(B, L, C, generator=g) < 0.2).to(torch.int32)
    drop[:, L // 2] = 1  # a row with nothing to pick
    idx, sc = route_topk_launch(q5.to(DEV), lmk.to(DEV), lse4.to(DEV), topk, 64,
                                bias4=bias4.to(DEV), drop_mask=drop.to(DEV))
    ridx, rsc, sel = O.route_topk(q5, lmk, lse4, topk, 64, drop_mask=drop, bias4=bias4)
    idx = idx.cpu().long()
    assert bool((idx[:, L // 2] == -1).all())
    bad = (idx != ridx).any(-1)
    assert int((bad & ~(O.boundary_gap(sel, topk) < NEAR_TIE)).sum()) == 0
    ok = (~bad)[..., None, None].expand_as(rsc)
    # bf16 scores of fp32 sums over 128 products: half a bf16 step (2^-9) plus
    # the sums' own difference (below 1e-3 at these magnitudes)
    torch.testing.assert_close(sc.cpu().float()[ok], rsc.bfloat16().float()[ok], atol=2e-3,
                               rtol=2.0 ** -8)


@pytest.mark.parametrize("C,Hkv,G,topk,window,valid_keys", [
    (257, 1, 7, 32, 100, True),    # one chunk past the one-pass kernels
    (271, 2, 2, 8, 319, True),     # neither a multiple of 16 nor of 64
    (304, 1, 3, 64, 0, False),     # each query's own chunk alone
    (290, 1, 1, 20, 30000, True),  # a window that hides every chunk
])
def test_route_topk_scan_derived_drop_equals_explicit(C, Hkv, G, topk, window, valid_keys):
    """The scan path's own drop mask (chunks in the window, chunks with no valid
    key) against the explicit one and the oracle."""

    print(f"[gpu-case] scan derived drop C={C} Hkv={Hkv} G={G} K={topk} W={window}", flush=True)
    g = torch.Generator().manual_seed(3000 + C)
    B, L = 2, 64 * C
    q5 = torch.randn(B, L, Hkv, G, 128, generator=g).bfloat16()
    lmk = (0.5 * torch.randn(B, C, Hkv * G, 128, generator=g)).bfloat16()
    lse4 = torch.randn(B, L, Hkv, G, generator=g) + 3.0
    bias4 = torch.randn(B, C, Hkv, G, generator=g)
    valid = torch.ones(B, L, dtype=torch.bool)
    if valid_keys:
        valid = torch.rand(B, L, generator=g) > 0.1
        dead = torch.rand(B, C, generator=g) < 0.2     # chunks with no key, the last one too
        dead[0, -1] = True
        dead = dead.repeat_interleave(64, 1)
        dead[:, 63::64] = False                        # (their landmark slots do not count)
        valid &= ~dead
    drop = O.remote_drop_mask(valid, window, 64)
    args = (q5.to(DEV), lmk.to(DEV), lse4.to(DEV), topk, 64)
    idx, sc = route_topk_launch(*args, bias4=bias4.to(DEV), derive_window=window,
                                key_valid=valid.to(DEV) if valid_keys else None)
    eidx, esc = route_topk_launch(*args, bias4=bias4.to(DEV), drop_mask=drop.to(DEV))
    assert torch.equal(idx, eidx) and torch.equal(sc, esc)
    ridx, rsc, sel = O.route_topk(q5, lmk, lse4, topk, 64, drop_mask=drop, bias4=bias4)
    bad = (idx.cpu().long() != ridx).any(-1)
    assert int((bad & ~(O.boundary_gap(sel, topk) < NEAR_TIE)).sum()) == 0


@pytest.mark.parametrize("B,Lq,C,Hkv,G,K,keep,det", [
    (1, 1, 40, 4, 7, 32, False, False),    # one query, parts of 4 steps
    (1, 33, 24, 4, 7, 32, False, False),   # 4-query tiles, the last one partial, parts
    (2, 64, 30, 2, 7, 16, True, False),    # keep rows, parts
    (1, 65, 9, 3, 8, 64, False, True),     # fixed order; tiles of 16 at most
    (1, 641, 11, 4, 7, 32, False, False),  # 16-query tiles: 8 would make 324 workgroups
    (1, 250, 7, 8, 4, 32, True, False),    # 8-query tiles: 256 workgroups
    (1, 100, 7, 4, 3, 60, False, False),   # tiles of 16, 8, 4 out of 1024 // 60 = 17 queries
])
def test_routed_tiles_and_parts_vs_oracle(B, Lq, C, Hkv, G, K, keep, det):
    print(f"[gpu-case] routed tiles B={B} Lq={Lq} C={C} Hkv={Hkv} G={G} K={K} {keep} {det}",
          flush=True)
    g = torch.Generator().manual_seed(2000 + Lq + C)
    r = lambda *s: torch.randn(*s, generator=g).bfloat16()
    q, k, v = r(B, Lq, Hkv * G, 128), r(B, C * 64, Hkv, 128), r(B, C * 64, Hkv, 128)
    w = torch.softmax(torch.randn(B, Lq, Hkv * G, K, generator=g), -1).bfloat16()
    idx = torch.rand(B, Lq, Hkv, max(C, K), generator=g).topk(K, -1).indices.int()
    idx[idx >= C] = -1                    # (K > C: lists that end early)
    valid = torch.rand(B, C * 64, generator=g) > 0.1
    tk = (torch.rand(B, Lq, Hkv, K, 64, generator=g) > 0.4).to(torch.int8) if keep else None
    want = O.selected_attention(q, k, v, w, idx, valid, token_keep=tk)
    got = selected_attention_launch(
        q.to(DEV), kv_fragments(k.to(DEV), v.to(DEV)), w.to(DEV), idx.to(DEV), valid.to(DEV), 64,
        token_keep=None if tk is None else tk.to(DEV), deterministic=det)
    # w P rounded to bf16 once per term and the output once: 2^-9 of the row's
    # absolute sum (weights sum to 1, |v| < 5) and of the output
    torch.testing.assert_close(got.cpu().float(), want, atol=5 * 2.0 ** -9, rtol=2.0 ** -8)


@pytest.mark.parametrize("C,G,K,keep", [
    (257, 7, 5, False),      # one chunk past the rule
    (300, 8, 32, True),
    (700, 3, 8, False),      # (lists with negative ends and a repeated chunk)
])
def test_routed_attention_walks_that_join_vs_oracle(C, G, K, keep):
    print(f"[gpu-case] joined walks C={C} G={G} K={K} keep={keep}", flush=True)
    g = torch.Generator().manual_seed(C)
    Lq, Hkv = 600, 2             # 8-query tiles, whole walks
    q = torch.randn(1, Lq, Hkv * G, 128, generator=g).bfloat16()
    k, v = (torch.randn(1, C * 64, Hkv, 128, generator=g).bfloat16() for _ in range(2))
    w = torch.rand(1, Lq, Hkv * G, K, generator=g).bfloat16()
    idx = torch.rand(1, Lq, Hkv, C, generator=g).topk(K, -1).indices.sort(-1).values.int()
    idx[0, 3] = -1               # a query with no chunk
    idx[0, 5, :, 2:] = -1
    # descending lists (no chunk twice: the merged slots of a repeated chunk
    # share the first one's keep row, which the oracle does not)
    idx[0, 8:16] = idx[0, 8:16].flip(-1)
    if C == 700:
        idx[0, 17, :, 1] = idx[0, 17, :, 0]
    valid = torch.rand(1, C * 64, generator=g) > 0.1
    tk = (torch.rand(1, Lq, Hkv, K, 64, generator=g) > 0.4).to(torch.int8) if keep else None
    want = O.selected_attention(q, k, v, w, idx, valid, token_keep=tk).double()
    frags = kv_fragments(k.to(DEV), v.to(DEV))
    for _ in range(3):           # each launch joins where the one before it ended
        got = selected_attention_launch(
            q.to(DEV), frags, w.to(DEV), idx.to(DEV), valid.to(DEV), 64,
            token_keep=None if tk is None else tk.to(DEV)).double().cpu()
        # P w is rounded to bf16 before its product and the output after (2^-9 each)
        assert (got - want).norm() <= 2.0 ** -8 * want.norm()
        assert torch.equal(got[0, 3], torch.zeros_like(got[0, 3]))


@pytest.mark.parametrize("mu", [2.0, 6.0, 12.0])
def test_route_scores_order_near_ties_as_well_as_the_plain_fp32_form(mu):
    """Two chunks whose scores, each another head's, lie within 1e-6: picks that
    differ from 64 bits are no more than those of x - logaddexp(LSE, m + log(sum
    of exp(x - m))) with each step rounded to fp32."""

    print(f"[gpu-case] route near ties mu={mu}", flush=True)
    L, H = 16384, 4
    g = torch.Generator().manual_seed(int(mu))
    a = (0.5 + 3.5 * torch.rand(L, H, 2, generator=g)).bfloat16()
    # head i's logits: a_i at chunk i, -8 a_i at the other (exact products)
    x = torch.stack([torch.stack([a[..., 0], -8 * a[..., 0]], -1),
                     torch.stack([-8 * a[..., 1], a[..., 1]], -1)], -2).float()
    l64 = torch.logsumexp(x.double(), -1)
    lse = torch.empty(L, H, 2)
    lse[..., 0] = mu + 0.5 * torch.randn(L, H, generator=g)
    total0 = torch.logaddexp(lse[..., 0].double(), l64[..., 0])
    total1 = a[..., 1].double() - (a[..., 0].double() - total0) \
        + 2e-6 * (torch.rand(L, H, generator=g, dtype=torch.float64) - 0.5)
    lse[..., 1] = total1 + torch.log(-torch.expm1(l64[..., 1] - total1))
    assert torch.isfinite(lse).all()

    def picks(total):  # of the larger of the heads' maxima, ties to chunk 0
        s = (x.to(total.dtype) - total[..., None]).amax(-2)
        return (s[..., 1] > s[..., 0]).int()

    exact = picks(torch.logaddexp(lse.double(), l64))
    m = x.amax(-1)
    plain = m + torch.log(torch.exp(x - m[..., None]).sum(-1))
    hi, lo = torch.maximum(lse, plain), torch.minimum(lse, plain)
    worst = int((picks(hi + torch.log1p(torch.exp(lo - hi))) != exact).sum())

    q = torch.zeros(1, L, H, 2, 128, dtype=torch.bfloat16)
    q[0, ..., 0] = a
    lmk = torch.zeros(1, 2, H * 2, 128, dtype=torch.bfloat16)
    lmk[0, 0, :, 0] = torch.tensor([1.0, -8.0]).repeat(H)
    lmk[0, 1, :, 0] = torch.tensor([-8.0, 1.0]).repeat(H)
    idx, _ = route_topk_launch(q.to(DEV), lmk.to(DEV), lse[None].to(DEV), 1, 64, sm_scale=1.0)
    got = int((idx[0, ..., 0].cpu() != exact).sum())
    print(f"picks off 64 bits: {got}, plain form {worst} of {L * H}")
    # 4000 to 14000 of 65536 differ: 10% is six standard deviations or more (the
    # totals held in base 2 give 20% to 40% more)
    assert got <= 1.1 * worst


def test_candidate_token_scores_walks_that_join_vs_oracle():
    print("[gpu-case] joined walks, token scores", flush=True)
    g = torch.Generator().manual_seed(261)
    Lq, C, Hkv, G, K = 200, 261, 2, 7, 8
    q = torch.randn(1, Lq, Hkv * G, 128, generator=g).bfloat16()
    k = torch.randn(1, C * 64, Hkv, 128, generator=g).bfloat16()
    idx = torch.rand(1, Lq, Hkv, C, generator=g).topk(K, -1).indices.sort(-1).values.int()
    idx[0, 3] = -1
    idx[0, 5, :, 2:] = -1
    valid = torch.rand(1, C * 64, generator=g) > 0.1
    want = O.candidate_token_scores(q, k, idx, valid, 64)
    fin = torch.isfinite(want)
    for _ in range(3):           # each launch joins where the one before it ended
        got = mrsa.candidate_token_scores_gqa(q.to(DEV), k.to(DEV), idx.to(DEV), valid.to(DEV),
                                              64).cpu()
        assert torch.equal(fin, torch.isfinite(got))
        # fp32 sums of 128 exact products: 128 x 2^-24 of their absolute sum, near
        # 128 x 0.64 / sqrt(128)
        torch.testing.assert_close(got[fin], want[fin], atol=1e-4, rtol=0)
