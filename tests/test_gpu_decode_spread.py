"""Decode attention whose splits are spread over all XCDs and merged by a
second launch (a few sequences with long contexts), against the oracle: one
to nine sequences, ragged lengths, empty splits, the fused RoPE form and its
quantising variant, calls of both forms sharing one workspace.
Tolerances: 2e-2 as in test_gpu_ops.py; the fused forms equal the separate
scatter, attention and quantiser bit for bit.
"""
import numpy as np
import pytest
import torch

from oracle import ops as O

pytestmark = pytest.mark.gpu


def _ops():
    from lite_lang_amd import ops
    return ops


def _case(B, H, KVH, D, lens, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    L = max(lens)
    q = torch.randn(B, H, D, generator=g).to(dtype)
    pool = torch.randn(B * L, 2 * KVH, D, generator=g).to(dtype)
    r2t = torch.from_numpy(np.random.RandomState(seed).permutation(B * L).astype(np.int32)).view(B, L)
    return q, pool, r2t


def _run(cuda, q, pool, r2t, lens, KVH, bound):
    pd = pool.to(cuda)
    B = q.shape[0]
    return _ops().decode_attention(
        q.to(cuda), r2t.to(cuda), torch.arange(B, dtype=torch.int32, device=cuda),
        torch.tensor(lens, device=cuda), bound, pd[:, :KVH], pd[:, KVH:],
        torch.empty_like(q, device=cuda)).cpu()


@pytest.mark.parametrize("B,H,KVH,D,L,dtype", [
    (1, 16, 2, 128, 4096, torch.bfloat16), (1, 12, 2, 128, 6001, torch.float16),
    (3, 16, 2, 128, 2500, torch.bfloat16), (2, 28, 4, 128, 3001, torch.float16),
    (9, 12, 2, 128, 2200, torch.bfloat16), (2, 8, 2, 64, 5000, torch.bfloat16),
    (1, 16, 2, 128, 1500, torch.bfloat16), (1, 32, 8, 64, 1300, torch.float16),
    (10, 16, 8, 64, 1800, torch.bfloat16)])
def test_spread_splits_match_oracle(cuda, B, H, KVH, D, L, dtype):
    from lite_lang_amd import _lib
    assert _lib.load().ll_decode_attention_splits_spread(B, KVH, D, L) == 1
    assert _lib.load().ll_decode_attention_splits_spread(2, KVH, D, 300) == 0
    lens = [max(1, L - (b * 1237) % L) for b in range(B)]
    lens[-1] = min(lens[-1], 40) if B > 1 else lens[-1]  # most splits of one sequence are empty
    q, pool, r2t = _case(B, H, KVH, D, lens, dtype, 61)
    print(f"case: spread decode B={B} H={H} KVH={KVH} D={D} L={L}", flush=True)
    ref = O.decode_attention(q, r2t, list(range(B)), lens, pool[:, :KVH], pool[:, KVH:])
    short = _case(2, H, KVH, D, [300, 77], dtype, 62)
    first = _run(cuda, *short, [300, 77], KVH, 300)
    for _ in range(3):  # both forms in turn on one workspace, which every call leaves at zero
        out = _run(cuda, q, pool, r2t, lens, KVH, L)
        assert float((out.double() - ref).abs().max()) <= 2e-2
        assert torch.equal(_run(cuda, *short, [300, 77], KVH, 300), first)


@pytest.mark.parametrize("quant", [False, True])
def test_spread_fused_rope_equals_separate(cuda, quant):
    ops = _ops()
    B, H, KVH, D, bound = 2, 12, 2, 128, 8192  # 16 splits for a bound far above the lengths
    g = torch.Generator().manual_seed(63)
    pool = torch.randn(7000, 2 * KVH, D, generator=g).bfloat16().to(cuda)
    r2t = torch.randperm(7000, generator=g)[:2 * 3500].view(2, 3500).to(torch.int32)
    r2t = torch.cat([r2t, r2t.flip(0)], 1).to(cuda)  # rows of 7000 entries
    lens = [3400, 17]
    from lite_lang_amd import _lib
    assert _lib.load().ll_decode_attention_splits_spread(B, KVH, D, bound) == 1
    W = (H + 2 * KVH) * D
    cos = torch.randn(bound, D // 2, generator=g).clamp(-1, 1).to(cuda)
    sin = torch.randn(bound, D // 2, generator=g).clamp(-1, 1).to(cuda)
    bias = torch.randn(W, generator=g).bfloat16().to(cuda)
    ln = torch.tensor(lens, dtype=torch.int32, device=cuda)
    pos = ln - 1
    rids = torch.arange(B, dtype=torch.int32, device=cuda)
    slots = r2t[torch.arange(B, device=cuda), pos.long()].contiguous()
    print(f"case: spread fused rope quant={quant}", flush=True)
    p1, p2 = pool.clone(), pool.clone()
    out1 = torch.empty(B, H, D, dtype=torch.bfloat16, device=cuda)
    out2, qbuf = torch.empty_like(out1), torch.empty(B, H * D, dtype=torch.bfloat16, device=cuda)
    if quant:
        part = torch.randint(-4000, 4000, (2, B, W), generator=g, dtype=torch.int32).to(cuda)
        st = (torch.rand(B, generator=g) * 0.01 + 1e-3).to(cuda)
        sc = (torch.rand(W, generator=g) * 0.05 + 1e-3).bfloat16().to(cuda)
        p = ops.I8Partials(part.view(-1), 2, st, sc)
        _, qc, qs = ops.decode_attention_rope_splitk_i32(
            p, bias, pos, cos, sin, slots, r2t, rids, ln, bound, p1[:, :KVH], p1[:, KVH:], out1,
            quant=True)
        f = torch.empty(B, W, device=cuda)
        ops.dequant_splitk(part.view(-1), 2, st, sc, f, B, W)
        ops.rope_kv_scatter_splitk(f.view(-1), 1, bias, qbuf, H, KVH, D, pos, cos, sin, slots, p2)
    else:
        part = torch.randn(3, B, W, generator=g).to(cuda)
        ops.decode_attention_rope_splitk(part.view(-1), 3, bias, pos, cos, sin, slots, r2t, rids,
                                         ln, bound, p1[:, :KVH], p1[:, KVH:], out1)
        ops.rope_kv_scatter_splitk(part.view(-1), 3, bias, qbuf, H, KVH, D, pos, cos, sin, slots, p2)
    ops.decode_attention(qbuf.view(B, H, D), r2t, rids, ln, bound, p2[:, :KVH], p2[:, KVH:], out2)
    assert torch.equal(out1, out2) and torch.equal(p1, p2)
    if quant:
        wq, ws = ops.quant_per_token(out2.view(B, H * D))
        assert torch.equal(qc, wq) and torch.equal(qs, ws)


@pytest.mark.parametrize("B,H,KVH,D,bound,same_launch", [
    (2, 40, 8, 128, 8192, True), (1, 64, 8, 128, 4096, True), (3, 33, 3, 64, 8192, True),
    (8, 40, 8, 128, 600, False), (9, 64, 8, 64, 1000, False), (3, 32, 4, 128, 8192, True),
    (4, 7, 1, 128, 4096, True)])
def test_quantising_merge_in_a_second_launch_holds_any_head_count(cuda, B, H, KVH, D, bound,
                                                                  same_launch):
    """Heads on both sides of what the merging waves keep in registers (16 and
    32), splits merged by the second launch because they are spread or because
    the same-launch merge is off: equal to the separate scatter, attention and
    quantiser bit for bit, the workspace left at zero."""
    from lite_lang_amd import _lib
    L = _lib.load()
    ops = _ops()
    assert L.ll_decode_attention_split_count(B, KVH, D, bound) > 1
    assert L.ll_decode_attention_splits_spread(B, KVH, D, bound) == same_launch
    g = torch.Generator().manual_seed(64)
    lens = [max(1, bound - b * 977) for b in range(B)]
    W, P = (H + 2 * KVH) * D, B * bound
    pool = torch.randn(P, 2 * KVH, D, generator=g).bfloat16().to(cuda)
    r2t = torch.randperm(P, generator=g).view(B, bound).to(torch.int32).to(cuda)
    cos = torch.randn(bound, D // 2, generator=g).clamp(-1, 1).to(cuda)
    sin = torch.randn(bound, D // 2, generator=g).clamp(-1, 1).to(cuda)
    bias = torch.randn(W, generator=g).bfloat16().to(cuda)
    ln = torch.tensor(lens, dtype=torch.int32, device=cuda)
    pos, rids = ln - 1, torch.arange(B, dtype=torch.int32, device=cuda)
    slots = r2t[torch.arange(B, device=cuda), pos.long()].contiguous()
    part = torch.randint(-4000, 4000, (2, B, W), generator=g, dtype=torch.int32).to(cuda)
    st = (torch.rand(B, generator=g) * 0.01 + 1e-3).to(cuda)
    sc = (torch.rand(W, generator=g) * 0.05 + 1e-3).bfloat16().to(cuda)
    static = torch.tensor([0.03], device=cuda)
    print(f"case: quantising merge B={B} H={H}/{KVH} D={D} bound={bound} {same_launch}", flush=True)
    p2 = pool.clone()
    qbuf = torch.empty(B, H * D, dtype=torch.bfloat16, device=cuda)
    want = torch.empty(B, H, D, dtype=torch.bfloat16, device=cuda)
    f = torch.empty(B, W, device=cuda)
    ops.dequant_splitk(part.view(-1), 2, st, sc, f, B, W)
    ops.rope_kv_scatter_splitk(f.view(-1), 1, bias, qbuf, H, KVH, D, pos, cos, sin, slots, p2)
    ops.decode_attention(qbuf.view(B, H, D), r2t, rids, ln, bound, p2[:, :KVH], p2[:, KVH:], want)
    prev = ops.set_same_launch_merge(same_launch)
    try:
        for scale in (None, static):
            p1 = pool.clone()
            out = torch.full((B, H, D), 9.0, dtype=torch.bfloat16, device=cuda)
            _, qc, qs = ops.decode_attention_rope_splitk_i32(
                ops.I8Partials(part.view(-1), 2, st, sc), bias, pos, cos, sin, slots, r2t, rids, ln,
                bound, p1[:, :KVH], p1[:, KVH:], out, quant=True, input_scale=scale)
            assert torch.equal(out, want) and torch.equal(p1, p2)
            wq, ws = (ops.quant_per_token(want.view(B, H * D)) if scale is None
                      else ops.quant_static(want.view(B, H * D), scale))
            assert torch.equal(qc, wq) and torch.equal(qs, ws)
            assert ops.workspace(cuda, "decode_attention", 0).count_nonzero() == 0
    finally:
        ops.set_same_launch_merge(prev)
