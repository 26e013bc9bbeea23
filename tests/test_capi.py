"""The C-ABI library loads, exports every declared entry point and rejects bad
arguments on the host (no GPU needed: nothing here launches a kernel)."""

import ctypes
import os
import re

import pytest

from conftest import PKG_DIR, ROOT

HEADER = os.path.join(ROOT, "include", "mrsa.h")
LIB = os.path.join(PKG_DIR, "mrsa", "libmrsa.so")


def _declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mrsa_[a-z0-9_]+)\s*\(", text)))


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        pytest.fail(f"{LIB} missing: run __graft_entry__.build() first")
    return ctypes.CDLL(LIB)


def test_header_lists_expected_entry_points():
    names = _declared()
    for expected in (
        "mrsa_chunk_attn_pool_gqa_fwd", "mrsa_remote_drop_mask", "mrsa_route_topk_fwd",
        "mrsa_route_weights_fwd", "mrsa_local_attention_fwd", "mrsa_selected_attention_fwd",
        "mrsa_fuse_hils_outputs_fwd", "mrsa_candidate_token_scores_fwd",
        "mrsa_kv_fragments", "mrsa_kv_fragments_rows",
    ):
        assert expected in names


def test_every_declared_symbol_is_exported(lib):
    missing = [n for n in _declared() if not hasattr(lib, n)]
    assert not missing, f"not exported: {missing}"


def test_python_binding_matches_header():
    import mrsa._lib as L

    assert sorted(L.SIGNATURES) == _declared()


def test_status_strings_and_version(lib):
    lib.mrsa_status_string.restype = ctypes.c_char_p
    assert lib.mrsa_status_string(0) == b"ok"
    assert b"invalid" in lib.mrsa_status_string(1)
    assert lib.mrsa_abi_version() >= 3


def test_host_side_argument_errors(lib):
    import mrsa._lib as L

    L.load()
    # Negative sizes and NULL pointers are rejected before any launch.
    assert L.call("mrsa_fuse_hils_outputs_fwd", None, None, None, None, -1, 128, None) == 1
    assert L.call("mrsa_fuse_hils_outputs_fwd", None, None, None, None, 4, 128, None) == 1
    assert L.call("mrsa_remote_drop_mask", None, None, 1, 100, 256, 64, None, None) == 1
    assert L.call("mrsa_chunk_attn_pool_gqa_fwd", None, None, None, 4, 64, 4, 17, 128,
                  1.0, 0, None, None, None, None, None) == 1
    assert L.call("mrsa_local_attention_fwd", 16, 16, None, None, 1, 64, 64, 28, 4, 96,
                  256, 0, 1.0, 16, 16, None) == 2          # head_dim 96 unsupported
    assert L.call("mrsa_selected_attention_fwd", 16, 16, 16, 16, None, 1, 64, 128, 28, 4,
                  128, 32, 32, 1, 1.0, 16, None) == 2      # chunk_size 32 unsupported
    assert L.call("mrsa_route_weights_fwd", 16, 16, 16, 16, 1, 4, 4, 4, 7, 65, 1.0, None,
                  None, 16, 16, None, None) == 2           # topk > 64
    assert L.call("mrsa_route_weights_fwd", 16, 16, 16, 16, 1, 4, 4, 4, 7, 32, 0.0, None,
                  None, 16, 16, None, None) == 1           # temperature <= 0
    assert L.call("mrsa_route_weights_bwd", 16, 16, 16, 16, 16, None, None, 1, 4, 4, 4, 7, 32,
                  1.0, 16, None, 16, 16, 16, None, None) == 1  # gate given, no d_gate
    # Walk split: parts outside 1..64, or a missing workspace, are rejected.
    assert L.call("mrsa_selected_attention_split_fwd", 16, 16, 16, 16, None, 1, 64, 128,
                  28, 4, 128, 32, 64, 1, 1.0, 0, 16, 16, None) == 1
    assert L.call("mrsa_selected_attention_split_fwd", 16, 16, 16, 16, None, 1, 64, 128,
                  28, 4, 128, 32, 64, 1, 1.0, 65, 16, 16, None) == 1
    assert L.call("mrsa_selected_attention_split_fwd", 16, 16, 16, 16, None, 1, 64, 128,
                  28, 4, 128, 32, 64, 1, 1.0, 4, None, 16, None) == 1
    assert L.call("mrsa_selected_attention_split_fwd", 16, 16, 16, 16, None, 2000, 64,
                  128, 28, 4, 128, 32, 64, 1, 1.0, 40, 16, 16, None) == 2  # batch * parts
    assert L.call("mrsa_kv_fragments_bytes", 2, 65, 4, 128) == 2 * 4 * 2 * 16384 * 2
    assert L.call("mrsa_kv_fragments_bytes", 1, 64, 4, 96) == -1
    assert L.call("mrsa_kv_fragments", 16, None, 1, 64, 4, 96, 16, None) == 2  # head_dim 96
    assert L.call("mrsa_kv_fragments", None, None, 1, 64, 4, 128, 16, None) == 1
    # Empty problems are a successful no-op.
    assert L.call("mrsa_fuse_hils_outputs_fwd", None, None, None, None, 0, 128, None) == 0


def test_key_parts_heuristic():
    from mrsa.local_attention import key_parts

    assert key_parts(1, 16384, 4, 16384, 319) == 1
    # Cached block step: 32 queries (8 workgroups), window 319 -> 8 parts.
    assert key_parts(1, 32, 4, 131072, 319) == 8
    assert key_parts(1, 32, 4, 131072, 0) == 2
    assert key_parts(0, 32, 4, 4096, 319) == 1


def test_walk_parts_heuristic():
    from mrsa.sparse_attention import walk_parts

    # Long sequences: one workgroup per walk.
    assert walk_parts(1, 16384, 4, 16384, 32) == 1
    # The cached block step (32 queries, 4 KV heads, 2048 chunks): 32 parts.
    assert walk_parts(1, 32, 4, 131072, 32) == 32
    # Parts keep >= 32 steps each: 3 queries x 4 chunks -> 12 steps -> 1.
    assert walk_parts(1, 3, 4, 131072, 4) == 1
    assert walk_parts(1, 32, 4, 4096, 32) == 2
    assert walk_parts(0, 32, 4, 4096, 32) == 1


@pytest.mark.parametrize("batch,q_len,kv_heads,chunks,topk,parts", [
    (1, 16384, 4, 256, 32, 1),     # whole walks fill the chip
    (1, 32, 4, 128, 32, 8),        # a cached block step
    (1, 32, 4, 2048, 32, 4),       # against a long cache
    (4, 32, 4, 256, 32, 2),
    (1, 3, 4, 2048, 4, 3),         # 12 steps: parts of 4
    (1, 1, 1, 1, 1, 1),
    (1, 640, 4, 10, 32, 1),
    (1, 32, 4, 64, 257, 1),        # tiles of fewer than 4 queries are not the kernel's
    (2, 100, 8, 300, 256, None),
    (1, 77, 1, 8192, 64, None),
    (1, 255, 3, 33, 20, None),
])
def test_split_parts_agree_with_the_kernels_tiles(batch, q_len, kv_heads, chunks, topk, parts):
    from mrsa.sparse_attention import _split_parts

    got = _split_parts(batch, q_len, kv_heads, 64 * chunks, topk, 64)
    assert parts is None or got == parts
    assert 1 <= got <= 64
    if got == 1:
        return

    def kernel_tile(parts):  # the launcher's rule (routed_attention.hip)
        tile = min(32, 1024 // topk // 4 * 4)
        while True:
            half = (tile // 2 + 3) // 4 * 4
            if half >= tile or batch * kv_heads * parts * -(-q_len // half) > 256:
                return tile
            tile = half

    # the parts were chosen for the tile the kernel then takes, one workgroup
    # per CU, with 4 steps or more
    assert kernel_tile(got) == kernel_tile(1)
    tile = kernel_tile(got)
    assert batch * kv_heads * got * -(-q_len // tile) <= 256
    assert got <= min(chunks, min(tile, q_len) * topk) // 4


def test_split_parts_leave_empty_and_refused_sizes_to_the_library():
    from mrsa.sparse_attention import _split_parts

    for sizes in ((1, 32, 4, 4096, 0, 64), (1, 32, 4, 4096, 32, 0), (1, 16384, 4, 16384, 32, 0),
                  (0, 32, 4, 4096, 32, 64), (1, 0, 4, 4096, 32, 64), (1, 32, 0, 4096, 32, 64)):
        assert _split_parts(*sizes) == 1


@pytest.mark.gpu
def test_selected_attention_without_slots_is_a_value_error():
    import torch

    from mrsa.sparse_attention import selected_attention_launch

    q = torch.zeros(1, 4, 7, 128, dtype=torch.bfloat16, device="cuda:0")
    frags = torch.zeros(1, 1, 2, 16384, dtype=torch.bfloat16, device="cuda:0")
    idx = torch.zeros(1, 4, 1, 0, dtype=torch.int32, device="cuda:0")
    with pytest.raises(ValueError):
        selected_attention_launch(q, frags, q[..., :0], idx, None, 64)


@pytest.mark.parametrize("use_workspace,rows,chunks,groups,limit,entry,nbytes", [
    # (4 KV heads.)  Up to the limit the path's own bytes: selection scores and
    # LSE totals of many rows, logits of few, none for up to 256 chunks.
    (None, 1024, 300, 7, 1 << 34, "ws", 4096 * (304 + 7) * 4),
    (None, 32, 300, 7, 1 << 34, "ws", 128 * 7 * 300 * 4),
    (None, 1024, 256, 7, 1 << 34, "plain", 0),
    (None, 1024, 300, 7, 1 << 20, "plain", 0),
    # past it only where asked for
    (True, 1024, 300, 7, 1 << 20, "ws", 4096 * (304 + 7) * 4),
    (True, 32, 300, 7, 1 << 17, "ws", 128 * 7 * 300 * 4),
    (False, 32, 300, 7, 1 << 34, "plain", 0),
    # one head: its logits are the smaller workspace, and alone keep the limit
    (None, 1024, 300, 1, 4096 * 300 * 4, "ws", 4096 * 300 * 4),
])
def test_route_workspace_is_the_callers_choice(monkeypatch, use_workspace, rows, chunks, groups,
                                               limit, entry, nbytes):
    import torch

    from mrsa import _lib, topk

    calls = []

    def call(name, *args):
        if name.endswith("_bytes"):
            return real(name, *args)
        calls.append((name, args))
        return 0

    real = _lib.call
    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(_lib, "stream_of", lambda t: None)
    monkeypatch.setattr(topk, "_WORKSPACE_LIMIT", limit)
    q = torch.zeros(1, rows, 4, groups, 128, dtype=torch.bfloat16)
    lmk = torch.zeros(1, chunks, 4, 128, dtype=torch.bfloat16)
    topk._route_topk_impl(q, lmk, None, None, None, None, 32, 64, -1, False, 0, 0, True, 1.0,
                          False, -1 if use_workspace is None else int(use_workspace))
    (name, args), = calls
    assert name == {"ws": "mrsa_route_topk_ws_fwd", "plain": "mrsa_route_topk_fwd"}[entry]
    if entry == "ws":
        assert args[-2] == nbytes and args[-3]


def test_layer_cache_replace_on_host_tensors():
    # fastdllm_cache.py:94-125 on CPU tensors (no tiled copy yet): rows land,
    # errors as in the reference.
    import torch

    import mrsa

    k = torch.zeros(1, 256, 4, 8, dtype=torch.bfloat16)
    v = torch.zeros_like(k)
    cache = mrsa.LayerKVCache(k, v, torch.ones(1, 256, dtype=torch.bool),
                              torch.zeros(1, 4, 4, 7, 8, dtype=torch.bfloat16),
                              torch.zeros(1, 4, 4, 7))
    pos = torch.tensor([7, 3])
    cache.replace(pos, torch.ones(1, 2, 4, 8, dtype=torch.bfloat16),
                  torch.full((1, 2, 4, 8), 2.0, dtype=torch.bfloat16))
    assert float(cache.key[0, 3].float().sum()) == 32 and float(cache.value[0, 7, 0, 0]) == 2
    assert cache.physical_length == 256
    with pytest.raises(ValueError, match="unique"):
        cache.replace(torch.tensor([1, 1]), k[:, :2], v[:, :2])
    with pytest.raises(ValueError, match="range"):
        cache.replace(torch.tensor([256]), k[:, :1], v[:, :1])
    with pytest.raises(ValueError, match="shape"):
        cache.replace(torch.tensor([1]), k[:, :2], v[:, :2])
