"""The split rule of decode attention (host-only queries): where its lines lie,
and that no shape takes more splits than its workspace bound."""
import pytest

from lite_lang_amd import _lib


def _plan(B, KVH, D, n):
    L = _lib.load()
    return (L.ll_decode_attention_split_count(B, KVH, D, n),
            L.ll_decode_attention_splits_spread(B, KVH, D, n))


@pytest.mark.parametrize("KVH,D", [(1, 128), (2, 128), (4, 128), (8, 128), (2, 64), (8, 64)])
def test_split_counts_stay_within_their_bounds(KVH, D):
    """At least what the slot table's LDS asks for; otherwise at most one split
    per eight 16-token tiles and one dispatch round, at most 16 from 8
    (sequence, KV head) units up at head_dim 128, at most 16 or one per 24 tiles
    below 8 units and at head_dim 64. A same-launch merge holds 8."""
    for B in (1, 2, 3, 4, 7, 8, 9, 16, 20, 33, 40, 64, 128, 300):
        for n in list(range(1, 3300, 61)) + [4096, 12001, 70000, 140000]:
            ns, spread = _plan(B, KVH, D, n)
            tiles, units = -(-n // 16), B * KVH
            low = max(1, -(-tiles * 16 // 4096))
            cap = min(256 * (1 if D == 128 else 2) // units, tiles // 8)
            if units >= 8 and D == 128:
                cap = min(cap, 16)
            else:
                cap = min(cap, max(16, tiles // 24))
            assert low <= ns <= max(low, cap), (B, n)
            assert spread in (0, 1) and (spread or ns <= 8) and (not spread or ns > 1), (B, n)


@pytest.mark.parametrize("B,KVH,D,n,ns,spread", [
    (1, 2, 128, 600, 4, 0), (3, 2, 128, 450, 3, 0), (1, 2, 128, 1100, 4, 0),  # few tiles
    (1, 2, 128, 1136, 4, 0), (1, 2, 128, 1137, 8, 1), (2, 2, 128, 1500, 8, 1),
    (1, 2, 128, 2032, 8, 1), (1, 2, 128, 2033, 16, 1), (1, 4, 128, 2500, 16, 1),
    (3, 2, 128, 12001, 16, 1), (1, 2, 128, 16000, 32, 1),
    (4, 8, 128, 1000, 4, 0), (4, 8, 128, 1500, 8, 1), (40, 2, 128, 600, 2, 0),
    (1, 2, 64, 2500, 8, 0), (1, 2, 64, 3057, 16, 1), (16, 2, 64, 1500, 8, 0),
    (16, 2, 64, 8192, 8, 0), (4, 2, 64, 8192, 16, 1), (1, 8, 64, 1300, 8, 1),
    (6, 8, 64, 8192, 8, 0), (20, 8, 64, 2048, 3, 0), (10, 8, 64, 4096, 6, 1),
    (12, 8, 64, 4096, 5, 1), (12, 8, 64, 1024, 4, 0)])
def test_split_rule(B, KVH, D, n, ns, spread):
    assert _plan(B, KVH, D, n) == (ns, spread)


@pytest.mark.parametrize("batch,KVH,D,max_len,dtype,bounds", [
    (1, 2, 128, 2048, "bfloat16", [1024, 2048]), (14, 2, 128, 2048, "bfloat16", [1024, 2048]),
    (3, 2, 128, 1025, "float16", [1025]), (1, 2, 128, 1500, "float16", [1024, 1500]),
    (2, 2, 64, 8192, "bfloat16", [2048, 8192]), (1, 2, 64, 2048, "bfloat16", [2048]),
    (40, 2, 128, 4096, "bfloat16", [4096]), (1, 2, 128, 8192, "float32", [8192]),
    (1, 2, 96, 8192, "bfloat16", [8192])])
def test_decode_graph_bounds(batch, KVH, D, max_len, dtype, bounds):
    """A second, shorter capture only where the plan at max_length pays a merge
    launch that the shorter bound does not."""
    import types
    import torch
    from lite_lang_amd.models.qwen2.decode_graph import decode_bounds
    cfg = types.SimpleNamespace(num_key_value_heads=KVH, head_dim=D)
    model = types.SimpleNamespace(cfg=cfg, dtype=getattr(torch, dtype))
    assert decode_bounds(model, batch, max_len) == bounds


@pytest.mark.parametrize("heads,head_dim,wide", [(8, 16, True), (16, 128, True), (8, 20, False),
                                                 (72, 128, False)])
def test_wide_fused_decode_takes_only_what_its_kernels_take(heads, head_dim, wide):
    """Batches of 65 to 256 leave the general layer only where every kernel of
    the fused one takes the shape: head_dim % 8 for the scatter of partials,
    hidden <= 8192 for the norm."""
    import torch
    from lite_lang_amd.models.qwen2.model import Qwen2Model
    from lite_lang_amd.models.qwen2.weights import Qwen2Config
    cfg = Qwen2Config(layer_nums=1, hidden_size=heads * head_dim, num_heads=heads,
                      num_key_value_heads=heads // 4, intermediate_size=256, vocab_size=32)
    assert cfg.head_dim == head_dim
    m = Qwen2Model(1, 64, cfg, 0, 1, torch.bfloat16, torch.device("cpu"))
    assert [m.fused_decode_ok(b) for b in (64, 65, 256, 257)] == [True, wide, wide, False]
