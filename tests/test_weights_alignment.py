"""Weights handed over as views into one flat buffer, at offsets that are not
16-byte aligned: the packed copy holds aligned tensors of the same values."""
import torch

from lite_lang_amd.models.qwen2.weights import DeviceWeights, Qwen2Config
from tests.model_weights import moving_state_dict


def test_views_at_odd_offsets_are_copied():
    cfg = Qwen2Config(layer_nums=2, hidden_size=96, num_heads=3, num_key_value_heads=1,
                      intermediate_size=160, vocab_size=33)
    sd = moving_state_dict(cfg, seed=5, dtype=torch.float16)
    flat = torch.empty(sum(t.numel() + 1 for t in sd.values()), dtype=torch.float16)
    views, at = {}, 0
    for i, (name, t) in enumerate(sd.items()):
        at += i % 2  # odd element offsets among them
        views[name] = flat[at:at + t.numel()].view(t.shape).copy_(t)
        at += t.numel()
    assert sum(v.data_ptr() % 16 != 0 for v in views.values()) > 4
    w = DeviceWeights(cfg, views, torch.float16, "cpu", pack=False)
    for lw, i in zip(w.layers, range(2)):
        for name, mod in (("wo", "self_attn.o_proj"), ("wdown", "mlp.down_proj")):
            assert lw[name].data_ptr() % 16 == 0
            assert torch.equal(lw[name], sd[f"model.layers.{i}.{mod}.weight"])
        assert all(t is None or t.data_ptr() % 16 == 0 for t in lw.values())
    assert w.embed.data_ptr() % 16 == 0 and torch.equal(w.embed, sd["model.embed_tokens.weight"])
