"""Decode graphs captured for two length bounds (a small batch): steps before,
at and after the shorter bound against the eager layer, whose length bound is
each step's own. The two differ in the split of the attention's sums only, so
logits agree within the 2e-2 bar of two faithful 16-bit executions on these
weights (tests/model_weights.py); with W8A8 projections, where a moved rounding
also moves int8 codes (0.6e-2 of the logits' 2-norm at two layers), within 3e-2
of the 2-norm."""
import pytest
import torch

from lite_lang_amd.models.qwen2.weights import Qwen2Config
from tests.model_weights import moving_state_dict

pytestmark = pytest.mark.gpu


def _runner(graph, quant, cfg):
    from lite_lang_amd.models.qwen2 import Qwen2ModelRunner
    r = Qwen2ModelRunner(cfg.layer_nums, 2, cfg, max_length=2048, mem_usage=0.5,
                         use_radix_cache=False, dtype=torch.bfloat16, kv_max_size=2400,
                         state_dict=moving_state_dict(cfg, seed=97), device="cuda",
                         use_cuda_graph=graph, quant=quant)
    r.init_model()
    return r


@pytest.mark.parametrize("quant", [None, "w8a8"])
def test_steps_across_the_short_bound_match_eager(cuda, quant):
    from lite_lang_amd.models.runner_batch import RunnerBatch
    cfg = Qwen2Config(layer_nums=3, hidden_size=512, num_heads=4, num_key_value_heads=2,
                      intermediate_size=1024, vocab_size=1024)
    g = torch.Generator().manual_seed(97)
    msgs = [{"id": i, "input_tokens": torch.randint(0, 1024, (n,), generator=g).tolist()}
            for i, n in enumerate((1020, 33))]
    print(f"case: decode bounds quant={quant}", flush=True)
    got = {}
    for graph in (False, True):
        r = _runner(graph, quant, cfg)
        batch = RunnerBatch.create_batch(msgs, "b", True, r)
        got[graph] = []
        used = []
        for _ in range(1 + 8):
            out = r.forward(batch)
            got[graph].append((r.model_ins_.last_logits.float().clone(), out.clone()))
            if graph and r._graphs:
                dg = r._graphs[2]
                used.append([b for b, gr, lg in dg._graphs if gr is dg.graph and lg is dg.logits])
            batch.update_forward_message(out)
    # prefill of 1020, then decode steps at lengths 1021..1028
    assert used == [[1024]] * 4 + [[2048]] * 4
    same = torch.ones(2, dtype=torch.bool, device=cuda)
    for (a, ta), (b, tb) in zip(got[False], got[True]):
        diff = (a - b)[same]
        if quant is None:
            assert float(diff.abs().max()) <= 2e-2
        else:
            assert float(diff.norm() / a[same].norm()) <= 3e-2
        same &= (ta == tb).view(-1)
    assert bool(same.any())
