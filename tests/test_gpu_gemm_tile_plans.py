"""The tile GEMM's geometries (256 x 256, 256 x 128, 128 x 128), k splits and
edges (gemm_tiles.hip) against the oracle, every case with the plan it is meant
for: row counts on both sides of a tile, K ending in half a stage, rows that
allow no 16-byte stores, split products with fewer stages in the last split.
Tolerance as in test_gpu_gemm_tiles.py (2e-2 + one bf16 ulp of |y|); int8 sums
bit for bit.
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


# plan: (weight rows, activation rows, k splits) of the tile; one: the tile of the
# same shape in one split
@pytest.mark.parametrize("M,N,K,dtype,bias,plan,one", [
    (65, 1536, 8960, torch.bfloat16, True, (128, 128, 20), (128, 128)),
    (128, 132, 4128, torch.float16, False, (256, 256, 10), (256, 256)),  # N % 8 == 4, half a stage at the end
    (100, 260, 4096, torch.float16, True, (128, 128, 10), (128, 128)),   # N % 8 == 4
    (129, 2048, 11008, torch.bfloat16, False, (128, 128, 8), (128, 128)),  # one row past a tile
    (600, 2048, 11008, torch.bfloat16, True, (128, 128, 3), (128, 128)),
    (400, 3000, 4096, torch.bfloat16, True, (256, 128, 5), (128, 128)),
    (1679, 1536, 8960, torch.float16, False, (256, 128, 3), (128, 128)),
    (1416, 1300, 11008, torch.bfloat16, True, (256, 256, 7), (128, 128)),  # whole stages, 6 row tiles
    (1294, 2048, 8960, torch.float16, False, (256, 256, 5), (128, 128)),
    (430, 22016, 96, torch.bfloat16, False, (256, 256, 1), (256, 256)),  # two stages, the last one half
    (3000, 2560, 1056, torch.bfloat16, True, (256, 256, 1), (256, 256))])
def test_gemm_plans_match_oracle(cuda, M, N, K, dtype, bias, plan, one):
    from lite_lang_amd import _lib
    assert _ops().gemm_tiles_plan(M, N, K)[:3] == plan
    assert _ops().gemm_tiles_plan(M, N, K, split=False)[:3] == one + (1,)
    assert (_lib.load().ll_gemm_tiles_workspace_size(M, N, K, 2) > 0) == (plan[2] > 1)
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


@pytest.mark.parametrize("M,N,K,plan", [
    (65, 2048, 11008, (256, 128, 13)), (600, 1536, 8960, (256, 128, 7)),
    (333, 260, 1088, (256, 256, 1)), (2999, 2048, 11008, (256, 128, 1)),
    (2697, 1300, 8960, (256, 256, 3))])
def test_gemm_i8_splits_are_exact(cuda, M, N, K, plan):
    assert _ops().gemm_tiles_plan(M, N, K, 1)[:3] == plan
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


@pytest.mark.parametrize("M,K,tile", [
    (65, 64, (256, 128)), (129, 192, (256, 128)), (257, 160, (256, 256)), (700, 320, (256, 256)),
    (1100, 96, (256, 256)), (65, 1024, (128, 128))])
def test_gate_up_silu_geometries_agree(cuda, M, K, tile):
    """The fused epilogue of every geometry equals the product followed by
    silu_and_mul bit for bit (K sums run in the same order in all of them)."""
    g = torch.Generator().manual_seed(93)
    I = 8960
    assert _ops().gemm_tiles_plan(M, 2 * I, K, split=False)[:2] == tile
    x = torch.randn(M, K, generator=g).half().to(cuda)
    w = (torch.randn(2 * I, K, generator=g) * 0.1).half().to(cuda)
    ops = _ops()
    print(f"case: gate_up_silu geometry M={M} K={K}", flush=True)
    want = ops.silu_and_mul(ops.gemm_tiled(x, w), out=torch.empty(M, I, dtype=x.dtype, device=cuda))
    assert torch.equal(ops.gate_up_silu_tiled(x, ops.interleave_gate_up(w)), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_geometries_give_the_same_bits(cuda, dtype):
    """The same rows through all three geometries (each chosen by the row
    count): product and fused gate/up + SiLU alike, bit for bit."""
    ops = _ops()
    I, K = 8960, 1024
    g = torch.Generator().manual_seed(99)
    x = torch.randn(400, K, generator=g).to(dtype).to(cuda)
    w = (torch.randn(2 * I, K, generator=g) * 0.05).to(dtype).to(cuda)
    wil = ops.interleave_gate_up(w)
    print(f"case: geometries alike {dtype}", flush=True)
    act, y = ops.gate_up_silu_tiled(x, wil), ops.gemm_tiled(x, w)
    assert ops.gemm_tiles_plan(400, 2 * I, K, split=False)[:2] == (256, 256)
    for M, tile in ((65, (128, 128)), (129, (256, 128))):
        assert ops.gemm_tiles_plan(M, 2 * I, K, split=False)[:2] == tile
        assert torch.equal(ops.gate_up_silu_tiled(x[:M], wil), act[:M])
        assert torch.equal(ops.gemm_tiled(x[:M], w), y[:M])


@pytest.mark.parametrize("M,tile", [(200, (256, 128)), (1100, (256, 256))])
def test_i8_gate_up_silu_geometries_are_exact(cuda, M, tile):
    """The dequantising SiLU epilogue over several rounds of tiles (1100 rows:
    430 tiles of 256 x 256), bit for bit against exact int32 sums dequantised on
    the host and the separate SiLU_and_Mul."""
    ops = _ops()
    I, K = 11008, 1024
    assert ops.gemm_tiles_plan(M, 2 * I, K, 1, split=False)[:2] == tile
    g = torch.Generator().manual_seed(100)
    xq = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8).to(cuda)
    wq = torch.randint(-128, 128, (2 * I, K), generator=g, dtype=torch.int8).to(cuda)
    st = torch.rand(M, generator=g) * 0.001 + 1e-5
    sc = (torch.rand(2 * I, generator=g) * 0.001 + 1e-5).bfloat16()
    print(f"case: i8 gate_up_silu geometry M={M}", flush=True)
    got = ops.gemm_i8_gate_up_silu_tiled(xq, st.to(cuda), ops.interleave_gate_up(wq), sc.to(cuda))
    acc = ops.gemm_i8_i32_tiled(xq, wq).cpu()
    assert torch.equal(acc[:3], O.int8_gemm_i32(xq[:3].cpu(), wq.cpu()))
    gu = O.dequant_int32(acc, st, sc).bfloat16().to(cuda)
    assert torch.equal(got, ops.silu_and_mul(gu, out=torch.empty(M, I, dtype=gu.dtype, device=cuda)))


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
