"""The tile GEMM's geometries (256 x 256, 256 x 128, 128 x 128), k splits and
edges (gemm_tiles.hip) against the oracle: row counts on both sides of a tile,
K ending in half a stage, rows that allow no 16-byte stores, split products
with fewer stages in the last split. Tolerance as in test_gpu_gemm_tiles.py
(2e-2 + one bf16 ulp of |y|); int8 sums bit for bit.
"""
import pytest
import torch

from oracle import ops as O

pytestmark = pytest.mark.gpu


def _ops():
    from lite_lang_amd import ops
    return ops


def _excess(y, ref):
    return float(((y.cpu().double() - ref).abs() - (2e-2 + 2.0 ** -7 * ref.abs())).max())


@pytest.mark.parametrize("M,N,K,dtype,bias,split", [
    (65, 1536, 8960, torch.bfloat16, True, True),       # 128 x 128, many splits, last one shorter
    (128, 132, 4128, torch.float16, False, True),       # N % 8 == 4, half a stage at the end
    (100, 260, 4096, torch.float16, True, True),        # N % 8 == 4, 128 x 128 in splits
    (129, 2048, 11008, torch.bfloat16, False, True),    # one row past a tile
    (600, 2048, 11008, torch.bfloat16, True, True),     # 256 x 128 in splits
    (1679, 1536, 8960, torch.float16, False, True),     # 256 x 256 in splits
    (430, 22016, 96, torch.bfloat16, False, False),     # two stages, the last one half
    (3000, 2560, 1056, torch.bfloat16, True, False)])
def test_gemm_plans_match_oracle(cuda, M, N, K, dtype, bias, split):
    from lite_lang_amd import _lib
    assert (_lib.load().ll_gemm_tiles_workspace_size(M, N, K, 2) > 0) == split
    g = torch.Generator().manual_seed(91)
    x = torch.randn(M, K + 8, generator=g).to(dtype)[:, :K]
    w = (torch.randn(N, K, generator=g) * 0.05).to(dtype)
    b = torch.randn(N, generator=g).to(dtype) if bias else None
    print(f"case: gemm plan M={M} N={N} K={K} {dtype} bias={bias}", flush=True)
    xd, wd, bd = x.to(cuda), w.to(cuda), b.to(cuda) if bias else None
    wide = torch.zeros(M, N + 4, dtype=dtype, device=cuda)  # 8-byte aligned rows
    ref = O.linear(x, w, b)
    for y in (_ops().gemm(xd, wd, bd), _ops().gemm_tiled(xd, wd, bd),
              _ops().gemm(xd, wd, bd, out=wide[:, :N])):
        assert _excess(y, ref) <= 0
    assert not wide[:, N:].any()


@pytest.mark.parametrize("M,N,K", [(65, 2048, 11008), (600, 1536, 8960), (333, 260, 1088),
                                   (2999, 2048, 11008)])
def test_gemm_i8_splits_are_exact(cuda, M, N, K):
    g = torch.Generator().manual_seed(92)
    xq = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8)
    wq = torch.randint(-128, 128, (N, K), generator=g, dtype=torch.int8)
    st = torch.rand(M, generator=g) * 0.01 + 1e-4
    sc = (torch.rand(N, generator=g) * 0.01 + 1e-4).half()
    b = torch.randn(N, generator=g).bfloat16()
    print(f"case: gemm_i8 splits M={M} N={N} K={K}", flush=True)
    got = _ops().gemm_i8_tiled(xq.to(cuda), st.to(cuda), wq.to(cuda), sc.to(cuda), b.to(cuda)).cpu()
    acc = O.int8_gemm_i32(xq, wq)
    assert torch.equal(got, (O.dequant_int32(acc, st, sc) + b.float()).bfloat16())
    assert torch.equal(_ops().gemm_i8_i32_tiled(xq.to(cuda), wq.to(cuda)).cpu(), acc)


@pytest.mark.parametrize("M,K", [(65, 64), (129, 192), (257, 160), (700, 320), (1100, 96)])
def test_gate_up_silu_geometries_agree(cuda, M, K):
    """The fused epilogue of every geometry equals the product followed by
    silu_and_mul bit for bit (K sums run in the same order in all of them)."""
    g = torch.Generator().manual_seed(93)
    I = 8960
    x = torch.randn(M, K, generator=g).half().to(cuda)
    w = (torch.randn(2 * I, K, generator=g) * 0.1).half().to(cuda)
    ops = _ops()
    print(f"case: gate_up_silu geometry M={M} K={K}", flush=True)
    want = ops.silu_and_mul(ops.gemm_tiled(x, w), out=torch.empty(M, I, dtype=x.dtype, device=cuda))
    assert torch.equal(ops.gate_up_silu_tiled(x, ops.interleave_gate_up(w)), want)


def test_gemm_splits_inside_a_captured_graph(cuda):
    """Captured with a workspace already there the product splits; with none
    it runs one split: every replay within the bar, and the eager call's bits
    where it splits."""
    ops = _ops()
    g = torch.Generator().manual_seed(94)
    x = torch.randn(96, 4096, generator=g).bfloat16().to(cuda)
    w = (torch.randn(512, 4096, generator=g) * 0.05).bfloat16().to(cuda)
    ref = O.linear(x.cpu(), w.cpu())
    eager = ops.gemm(x, w)
    out = torch.empty_like(eager)
    print("case: gemm splits in a graph", flush=True)
    graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    for reserve in (False, True):
        if reserve:
            with torch.cuda.stream(stream):
                ops.gemm(x, w)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            ops.gemm(x, w, out=out)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert _excess(out, ref) <= 0
            assert not reserve or torch.equal(out, eager)
            ops.gemm(x, w)
