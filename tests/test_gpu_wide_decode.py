"""Split-K partials of the tile GEMM and the layers that read them: a decode
batch of more than 64 requests and the o_proj / down_proj of a prefill whose
products split over k.

The partials summed in split order are ll_gemm's result bit for bit (same
plan, same order). The layers are compared with the general ones (one
reduction launch per product, separate RoPE): the roundings are the same and
only the norm's sum runs in another order, so logits agree within the 2e-2 bar
of two faithful 16-bit executions on these weights (tests/model_weights.py).
"""
import pytest
import torch

from lite_lang_amd.models.qwen2.weights import Qwen2Config
from tests.model_weights import moving_state_dict

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K,dtype", [
    (65, 2560, 2048, torch.bfloat16), (128, 132, 4128, torch.float16),
    (96, 2048, 11008, torch.bfloat16), (1679, 1536, 8960, torch.float16),
    (300, 22016, 96, torch.bfloat16)])  # the last in one split
def test_partials_sum_to_the_product(cuda, M, N, K, dtype):
    from lite_lang_amd import ops
    g = torch.Generator().manual_seed(95)
    x = torch.randn(M, K + 8, generator=g).to(dtype).to(cuda)[:, :K]
    w = (torch.randn(N, K, generator=g) * 0.05).to(dtype).to(cuda)
    n = ops.gemm_tiles_splitk_count(M, N, K, dtype)
    print(f"case: tile partials M={M} N={N} K={K} splits={n}", flush=True)
    part = torch.full((n * M * N + 4,), 7.0, device=cuda)
    assert ops.gemm_tiles_splitk(x, w, part) == n
    acc = torch.zeros(M, N, device=cuda)
    for p in part[:-4].view(n, M, N):
        acc += p
    assert torch.equal(acc.to(dtype), ops.gemm(x, w))
    assert (part[-4:] == 7).all()
    with pytest.raises(RuntimeError, match="partials need"):
        ops.gemm_tiles_splitk(x, w, part[:n * M * N - 4])


def _steps(cuda, B, dtype, graph, head_dim, n_steps=2, tokens=None):
    """Logits and tokens of a prefill of B short prompts and of the decode steps
    after it, which are fed the run's own tokens or the given ones."""
    from lite_lang_amd.models.qwen2 import Qwen2ModelRunner
    from lite_lang_amd.models.runner_batch import RunnerBatch
    cfg = Qwen2Config(layer_nums=3, hidden_size=4 * head_dim, num_heads=4, num_key_value_heads=2,
                      intermediate_size=2048, vocab_size=1024)
    g = torch.Generator().manual_seed(96)
    msgs = [{"id": i, "input_tokens": torch.randint(0, 1024, (3 + i % 7,), generator=g).tolist()}
            for i in range(B)]
    r = Qwen2ModelRunner(cfg.layer_nums, B, cfg, max_length=128, mem_usage=0.5,
                         use_radix_cache=False, dtype=dtype, kv_max_size=B * 16,
                         state_dict=moving_state_dict(cfg, seed=96), device="cuda",
                         use_cuda_graph=graph)
    r.init_model()
    batch = RunnerBatch.create_batch(msgs, "wide", True, r)
    logits, outs = [], []
    for i in range(1 + n_steps):
        out = r.forward(batch)
        logits.append(r.model_ins_.last_logits.float().clone())
        outs.append(out.clone())
        batch.update_forward_message(out if tokens is None else tokens[i])
    return r, logits, outs


@pytest.mark.parametrize("B,dtype,graph,head_dim", [
    (65, torch.bfloat16, True, 128), (96, torch.float16, False, 128),
    (128, torch.bfloat16, True, 64), (129, torch.bfloat16, True, 128),  # two row tiles from 129
    (160, torch.float16, True, 64), (256, torch.float16, False, 128),
    (257, torch.float16, True, 64)])
def test_wide_decode_matches_general_layer(cuda, monkeypatch, B, dtype, graph, head_dim):
    from lite_lang_amd.models.qwen2 import model
    print(f"case: wide decode B={B} {dtype} graph={graph} D={head_dim}", flush=True)
    r, got, toks = _steps(cuda, B, dtype, graph, head_dim)
    assert r.model_ins_.fused_decode_ok(B) == (B <= model._WIDE_DECODE)
    assert r.model_ins_._norm_splits(5 * B)[1] > 1  # the prefill's down_proj splits
    if graph and not r.model_ins_.fused_decode_ok(B):
        # the captured general layer finds the workspace of its split products
        from lite_lang_amd import ops
        from lite_lang_amd.models.qwen2.decode_graph import _capture_stream
        need = r.model_ins_.norm_part_bytes(B)
        with torch.cuda.stream(_capture_stream(cuda)):
            assert 0 < need <= ops._WS[ops._ws_key(cuda, "norm_part")].numel()
    monkeypatch.setattr(model, "_WIDE_DECODE", 64)
    monkeypatch.setattr(model.Qwen2Model, "_norm_splits", lambda self, T: (1, 1))
    _, want, _ = _steps(cuda, B, dtype, graph, head_dim, tokens=toks)
    for a, b, t in zip(got, want, toks):
        assert float((a - b).abs().max()) <= 2e-2
        # the picked tokens: the largest logit of either run but for a tie within the bar
        assert float((b.amax(-1) - b.gather(-1, t).squeeze(-1)).max()) <= 4e-2
