"""What the edge and staged kernels store: tiles that lie whole inside C beside tiles that C ends in, rows of C on any element, every output type, scales and old
values.  Whole numbers whose sums every type holds, so every result has one right value."""
import pytest

import oracle as O

TORCH = {O.F32: "float32", O.F16: "float16", O.BF16: "bfloat16", O.I8: "int8", O.E4M3: "float8_e4m3fn", O.I32: "int32"}
OUTS = {O.F32: (O.F32,), O.F16: (O.F16, O.F32), O.BF16: (O.BF16, O.F32), O.I8: (O.I32, O.F16, O.F32), O.E4M3: (O.BF16, O.F16, O.F32)}


def check(hip, dtype, transA, transB, M, N, K, out, epilogue, clear, ldc, shift, tile=(0, 0, 0), stages=0):
    import torch
    g = torch.Generator(device="cuda").manual_seed(M * 31 + N * 7 + K)
    draw = lambda *shape: torch.randint(-2, 3, shape, device="cuda", generator=g)
    A, B = draw(M, K), draw(K, N)
    stored = lambda x, t: (x.t() if t else x).contiguous().to(getattr(torch, TORCH[dtype]))
    a, b = stored(A, transA), stored(B, transB)
    tdt = getattr(torch, TORCH[out])
    base = torch.randint(-9, 10, (shift + M * ldc,), device="cuda", generator=g).to(tdt)
    old = base.clone()
    C = base[shift:shift + M * ldc].view(M, ldc)
    sa, sb = (0.5 + torch.rand(n, device="cuda", generator=g) for n in ((M, N) if epilogue == hip.EPI_ROW_COL_SCALE else (1, 1)))
    desc = hip.make_desc(dtype, M, N, K, dtype_out=out, transA=transA, transB=transB, ldc=ldc, clear_accum=clear, epilogue=epilogue, tile=tile, stages=stages)
    need = hip.workspace_bytes(desc)
    ws = torch.full((max(need, 16),), 0xFF, dtype=torch.uint8, device="cuda")
    scales = (sa.data_ptr(), sb.data_ptr()) if epilogue else (None, None)
    hip.gemm(desc, a.data_ptr(), b.data_ptr(), C.data_ptr(), *scales, ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    want = A.float() @ B.float()  # whole numbers of at most 4 K: exact
    if epilogue:
        want = (want * (sa[:, None] if epilogue == hip.EPI_ROW_COL_SCALE else sa)) * sb
    if not clear:
        want = want + old[shift:].view(M, ldc)[:, :N].float()
    where = (O.NP_STORAGE[dtype], transA, transB, M, N, K, out, epilogue, clear, ldc, shift, hip.kernel_names()[hip.plan(desc).kernel_id])
    assert torch.equal(C[:, :N], want.to(tdt)), where
    assert torch.equal(C[:, N:], old[shift:].view(M, ldc)[:, N:]) and torch.equal(base[:shift], old[:shift]), where


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [O.F32, O.F16, O.BF16, O.I8, O.E4M3])
@pytest.mark.parametrize("transA,transB", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_whole_tiles_of_an_edge_kernel_beside_the_others(hip, dtype, transA, transB):
    """M and N of whole tiles under a partial K tile (nothing to check), one short of and one beyond them, 1 to 12 columns of a wave's tile; C packed, in odd rows and off its first 16-byte
    boundary"""
    K = {O.F32: 3 * 32 + 4, O.F16: 3 * 64 + 8, O.BF16: 3 * 64 + 8, O.I8: 3 * 128 + 16, O.E4M3: 4 * 128 + 16}[dtype]
    for M, N in ((512, 512), (511, 513), (257, 640), (130, 384), (96, 257), (300, 131), (77, 521), (260, 268)):
        for out in OUTS[dtype]:
            for epilogue in (hip.EPI_NONE, hip.EPI_ROW_COL_SCALE, hip.EPI_TENSOR_SCALE)[:1 if out == O.I32 else 3]:
                for clear, ldc, shift in ((True, N, 0), (True, N + 3, 1), (False, N, 0), (False, N + 3, 1)):
                    check(hip, dtype, transA, transB, M, N, K, out, epilogue, clear, ldc, shift)
                if dtype != O.F32 and M > 256:
                    for tile in (128, 256):
                        check(hip, dtype, transA, transB, M, N, K, out, epilogue, False, N + 3, 1, tile=(tile, tile, 0))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [O.F16, O.BF16])
@pytest.mark.parametrize("stages", [2, 3])
def test_old_values_fetched_beside_the_k_tiles(hip, dtype, stages):
    """A weight gradient on 128x128 tiles into float32: from one K tile, whose old values come at once, over four and two pieces a K tile to loops that go on behind them, whole and
    with a partial last tile; wave tiles inside C and beyond it"""
    for tiles in (1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 19):
        for K in (tiles * 64, tiles * 64 - 8, tiles * 64 - 3):
            if K % 64 == 0:
                check(hip, dtype, 1, 0, 256, 128, K, O.F32, hip.EPI_NONE, False, 128, 0, tile=(128, 128, 0), stages=stages)
            if stages == 2:
                check(hip, dtype, 1, 0, 200, 320, K, O.F32, hip.EPI_NONE, False, 323, 1, tile=(128, 128, 0), stages=2)
            else:  # (the planner's own choice: no descriptor names the ring of 3 off the tile)
                check(hip, dtype, 1, 0, 2600, 1027, K, O.F32, hip.EPI_NONE, False, 1030, 1)
    p = hip.plan(hip.make_desc(dtype, 2600, 1027, 715, dtype_out=O.F32, transA=True, clear_accum=False))
    assert (p.tile_m, p.tile_n, p.stages) == (128, 128, 3)
    check(hip, dtype, 1, 0, 2304, 1289, 712, O.F32, hip.EPI_NONE, False, 1289, 0)
