"""Calls of several threads on one stream whose two launches hand partials on
in the stream's workspace (k-split products, spread decode attention): each
thread's results are those of its calls alone, bit for bit."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _gemm(ops, g, cuda):
    x = torch.randn(96, 4096, generator=g).bfloat16().to(cuda)
    w = (torch.randn(512, 4096, generator=g) * 0.05).bfloat16().to(cuda)
    return lambda: ops.gemm(x, w)


def _gemm_i8(ops, g, cuda):
    x = torch.randint(-128, 128, (96, 4096), generator=g, dtype=torch.int8).to(cuda)
    w = torch.randint(-128, 128, (512, 4096), generator=g, dtype=torch.int8).to(cuda)
    st, sc = torch.rand(96, generator=g).to(cuda), torch.rand(512, generator=g).to(cuda)
    return lambda: ops.gemm_i8_tiled(x, st, w, sc)


def _attention(ops, g, cuda, n=3000):
    q = torch.randn(1, 12, 128, generator=g).bfloat16().to(cuda)
    pool = torch.randn(n, 4, 128, generator=g).bfloat16().to(cuda)
    r2t = torch.randperm(n, generator=g).to(torch.int32).view(1, -1).to(cuda)
    rid = torch.zeros(1, dtype=torch.int32, device=cuda)
    ln = torch.tensor([n], device=cuda)
    return lambda: ops.decode_attention(q, r2t, rid, ln, n, pool[:, :2], pool[:, 2:],
                                        torch.empty_like(q))


def _attention_mixed(ops, g, cuda):
    """The second thread's splits merge in their own launch."""
    return _attention(ops, g, cuda, 1000 if g.initial_seed() % 3 == 0 else 3000)


@pytest.mark.parametrize("make", [_gemm, _gemm_i8, _attention, _attention_mixed])
def test_threads_on_one_stream(cuda, make):
    from lite_lang_amd import _lib, ops
    L = _lib.load()
    assert L.ll_gemm_tiles_workspace_size(96, 512, 4096, 2) > 0
    assert L.ll_gemm_tiles_workspace_size(96, 512, 4096, 1) > 0
    assert L.ll_decode_attention_splits_spread(1, 2, 128, 3000) == 1
    assert L.ll_decode_attention_splits_spread(1, 2, 128, 1000) == 0
    assert L.ll_decode_attention_split_count(1, 2, 128, 1000) > 1
    print(f"case: threads {make.__name__}", flush=True)
    calls = [make(ops, torch.Generator().manual_seed(98 + i), cuda) for i in range(3)]
    want = [c() for c in calls]
    torch.cuda.synchronize()
    bad, errors = [0] * 3, []

    def work(i):
        try:
            outs = [calls[i]() for _ in range(300)]
            bad[i] = sum(not torch.equal(o, want[i]) for o in outs)
        except Exception as e:  # reported by the main thread
            errors.append(e)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors and bad == [0, 0, 0]
