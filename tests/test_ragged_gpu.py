"""Problems off the tiles on the device: a K that is no multiple of the K tile on the edge kernels, rows off 16-byte boundaries staged
through registers (no workspace) and copied to aligned rows first (workspace).  Operands end with their last element, and the
bytes around C are checked for stray writes."""
import re

import numpy as np
import pytest

import oracle as O
from helpers import DEFAULT_OUT, TOL, from_dev, make_operand, run_gemm, stored_shapes, to_dev

BK = {O.F32: 32, O.F16: 64, O.BF16: 64, O.I8: 128, O.E4M3: 128}
ES = {O.F32: 4, O.F16: 2, O.BF16: 2, O.I8: 1, O.E4M3: 1}
OUT_NP = {O.F32: np.float32, O.F16: np.uint16, O.BF16: np.uint16, O.I32: np.int32}


def launch(hip, dtype, A, B, M, N, K, transA, transB, aligned, workspace=True, ldc_extra=0, **kw):
    """A and B as stored, each row padded to a multiple of 16 bytes (`aligned`) or followed by one more element"""
    import torch
    per = 16 // ES[dtype]

    def rows(x):
        cols = x.shape[1]
        ld = (cols + per - 1) // per * per if aligned else cols + 1 - (cols & 1)  # odd: no row but the first on a boundary
        buf = np.zeros((x.shape[0], ld), x.dtype)
        buf[:, :cols] = x
        return to_dev(buf.reshape(-1)[:(x.shape[0] - 1) * ld + cols]), ld

    (dA, lda), (dB, ldb) = rows(A), rows(B)
    out = DEFAULT_OUT[dtype]
    ldc = N + ldc_extra
    guard = np.full(64 + M * ldc, 0x55, dtype=np.uint8).astype(OUT_NP[out])
    dC = to_dev(guard)
    d = hip.make_desc(dtype, M, N, K, dtype_out=out, transA=bool(transA), transB=bool(transB), lda=lda, ldb=ldb, ldc=ldc, **kw)
    need = hip.workspace_bytes(d) if workspace else 0
    ws = torch.full((max(need, 16),), 0xFF, dtype=torch.uint8, device="cuda")  # NaNs of every float type
    hip.gemm(d, dA.data_ptr(), dB.data_ptr(), dC.data_ptr() + 32 * guard.itemsize, None, None, ws.data_ptr() if need else None, need,
             torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = from_dev(dC, OUT_NP[out], (64 + M * ldc,))
    inner = got[32:32 + M * ldc].reshape(M, ldc)
    assert np.array_equal(got[:32], guard[:32]) and np.array_equal(got[32 + M * ldc:], guard[32 + M * ldc:]), "write outside C"
    assert np.array_equal(inner[:, N:], guard[:M * ldc_extra].reshape(M, ldc_extra)), "write between the rows of C"
    return inner[:, :N], hip.kernel_names()[hip.plan(d).kernel_id], need


def verify(dtype, got, A, B, transA, transB):
    if dtype == O.I8:
        assert np.array_equal(got, O.gemm_i32(A, B, transA, transB))
    else:
        r = O.compare(DEFAULT_OUT[dtype], np.ascontiguousarray(got), O.gemm_f64(dtype, A, B, transA, transB))
        assert r["nonfinite"] == 0 and r["max_rel"] <= TOL[dtype] and r["fro_rel"] <= TOL[dtype], r


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.I8, O.E4M3, O.F32])
@pytest.mark.parametrize("transA,transB", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_a_partial_last_k_tile_on_the_edge_kernels(hip, dtype, transA, transB):
    """one to eight K tiles (every path through the prologue, the unrolled loop and the drain), the last one of 1 element up to all
    but one, on both edge tiles; C rows off 16-byte boundaries"""
    bk, big = BK[dtype], 128 if dtype == O.F32 else 256
    M, N = 150, 301
    for tile, ks in (((big, big, 0), (1, bk - 1, bk + 1, 2 * bk - 3, 2 * bk + 1, 3 * bk + 5, 8 * bk - 1)), ((big // 2, big // 2, 0), (7, bk + 3, 2 * bk + bk // 2, 4 * bk - 1))):
        for K in ks:
            A = make_operand(dtype, *stored_shapes(M, N, K, transA, transB)[0], seed=81, tensor=0, scale=0.5)
            B = make_operand(dtype, *stored_shapes(M, N, K, transA, transB)[1], seed=81, tensor=1, scale=0.5)
            got, name, need = launch(hip, dtype, A, B, M, N, K, transA, transB, True, ldc_extra=1, tile=tile, stages=2 if tile[0] != 256 else 3)
            assert name.endswith("_guard") and need == 0, name
            verify(dtype, got, A, B, transA, transB)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [O.F16, O.F32])
def test_infinities_before_k_do_not_leak_into_the_cleared_part_of_a_k_tile(hip, dtype):
    """the chunks fetched in place of those beyond K repeat values of the operand: an infinity among them must not meet a zero"""
    M, N, K = 64, 64, BK[dtype] + 5
    A = make_operand(dtype, M, K, seed=82, tensor=0, scale=0.5)
    B = make_operand(dtype, K, N, seed=82, tensor=1, scale=0.5)
    A[3, K - 1] = O.encode(dtype, np.array([np.inf], np.float32))[0]
    B[K - 1, :] = O.encode(dtype, np.full(N, 0.25, np.float32))
    got, _, _ = launch(hip, dtype, A, B, M, N, K, 0, 0, True)
    f = got.astype(np.float32) if dtype == O.F32 else got.view(np.float16).astype(np.float32)
    assert np.all(np.isposinf(f[3])) and np.all(np.isfinite(np.delete(f, 3, axis=0)))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.I8, O.E4M3, O.F32])
@pytest.mark.parametrize("transA,transB", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_rows_off_16_byte_boundaries(hip, dtype, transA, transB):
    """sizes around a chunk, a tile and a K tile; once without a workspace (staged through registers) and once with (copied first)"""
    bk = BK[dtype]
    for (M, N, K) in ((1, 3, 5), (3, 130, 1), (17, 9, bk + 1), (129, 127, 2 * bk), (255, 131, 3 * bk - 1), (301, 515, 5 * bk + 7)):
        A = make_operand(dtype, *stored_shapes(M, N, K, transA, transB)[0], seed=83, tensor=0, scale=0.5)
        B = make_operand(dtype, *stored_shapes(M, N, K, transA, transB)[1], seed=83, tensor=1, scale=0.5)
        for kw in (dict(workspace=False), dict(split_k=1), dict(tile=(128, 128, 0) if dtype == O.F32 else (256, 256, 0))):
            got, name, need = launch(hip, dtype, A, B, M, N, K, transA, transB, False, **kw)
            assert name.endswith("_guard") and (need > 0) == ("tile" in kw), (name, need)
            verify(dtype, got, A, B, transA, transB)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,transA,transB,aligned", [(O.F16, 0, 0, True), (O.BF16, 1, 0, True), (O.I8, 0, 1, False), (O.E4M3, 0, 1, True)])
def test_tail_split_of_an_edge_kernel(hip, dtype, transA, transB, aligned):
    """257 to 272 tiles of 256 x 256: the tiles behind the first round are computed in slices of K of unequal length (the last one
    partial), their sums and the checked stores in the second kernel"""
    bk = BK[dtype]
    M, N, K = 16 * 256 + 3, 15 * 256 + 17, (8 if bk == 64 else 16) * bk * 4 - bk - 8
    A = make_operand(dtype, *stored_shapes(M, N, K, transA, transB)[0], seed=84, tensor=0, scale=0.5)
    B = make_operand(dtype, *stored_shapes(M, N, K, transA, transB)[1], seed=84, tensor=1, scale=0.5)
    got, name, need = launch(hip, dtype, A, B, M, N, K, transA, transB, aligned, ldc_extra=1)
    tiles = 16  # 17 x 16 tiles
    assert "256x256" in name and need >= 2 * tiles * 256 * 256 * 4, (name, need)
    verify(dtype, got, A, B, transA, transB)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.I8, O.E4M3])
@pytest.mark.parametrize("M", [1, 17, 33, 63])
def test_tiles_that_stream_b_take_any_rows_and_any_k(hip, dtype, M):
    """32x32 and 64x32 tiles whose waves split K: one to seven K tiles (every path through the prologue and the drain), whole and partial,
    every work-group starting its walk over the whole ones at another of them; N ending inside a tile and inside a chunk"""
    bk, names = 4 * BK[dtype], set()
    cases = [(1040, bk - 56), (1037, bk + 7), (2056, 2 * bk - 24), (2056, 3 * bk), (4104, 3 * bk + 48), (4101, 4 * bk - 40), (4104, 6 * bk + 8)]
    cases += [(8328, bk), (8328, 2 * bk + 8), (8328, 4 * bk - 8)] if M <= 32 else []  # more than 256 tiles: the ring of 2
    for N, K in cases:
        A = make_operand(dtype, M, K, seed=85, tensor=0, scale=0.5)
        B = make_operand(dtype, N, K, seed=85, tensor=1, scale=0.5)
        got, name, _ = launch(hip, dtype, A, B, M, N, K, 0, 1, True, ldc_extra=1)
        names |= {name.split("_")[2], "s2" if "_s2" in name else "s4" if "_s4" in name else "s3"}
        verify(dtype, got, A, B, 0, 1)
    assert names >= ({"32x32x%d" % bk, "s2", "s4"} if M <= 32 else {"32x32x%d" % bk, "64x32x%d" % bk}), names
    assert names <= {"32x32x%d" % bk, "64x32x%d" % bk, "s2", "s3", "s4"}, names


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.I8, O.E4M3])
@pytest.mark.parametrize("transB", [0, 1])
def test_192_row_tiles(hip, dtype, transB):
    """one to eight K tiles, whole and partial, M and N ending inside a tile, inside a wave's 96 rows and at their end"""
    bk = BK[dtype]
    for M, N, K in ((3001, 2999, bk - 24), (2976, 3072, 2 * bk + 1), (2881, 3080, 3 * bk), (2900, 2999, 3 * bk + 8), (2880, 3072, 8 * bk + 40)):
        A = make_operand(dtype, *stored_shapes(M, N, K, 0, transB)[0], seed=86, tensor=0, scale=0.5)
        B = make_operand(dtype, *stored_shapes(M, N, K, 0, transB)[1], seed=86, tensor=1, scale=0.5)
        got, name, _ = launch(hip, dtype, A, B, M, N, K, 0, transB, True, ldc_extra=1)
        assert "192x256" in name, (M, N, K, name)
        verify(dtype, got, A, B, 0, transB)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,transB", [(O.F16, 0), (O.BF16, 0), (O.F16, 1), (O.I8, 1), (O.E4M3, 1)])
def test_few_rows_on_64_column_tiles(hip, dtype, transB):
    """a few rows to 64 of them (B stored along K: below 32), N ending inside a tile, eight to eleven K tiles of 256 bytes, whole and partial"""
    bk, few = 2 * BK[dtype], 9 if transB and dtype == O.F16 else 1
    for M, N, K in ((few, 8256, 8 * bk), (17, 9544, 8 * bk + 32), (31, 16320, 9 * bk), (12 if transB else 64, 12296, 10 * bk), (16 if transB else 33, 8264, 11 * bk - 64)):
        A = make_operand(dtype, M, K, seed=94, tensor=0, scale=0.5)
        B = make_operand(dtype, *stored_shapes(M, N, K, 0, transB)[1], seed=94, tensor=1, scale=0.5)
        got, name, need = launch(hip, dtype, A, B, M, N, K, 0, transB, True)
        assert "64x64x" in name and need == 0, (M, N, K, name, need)
        verify(dtype, got, A, B, 0, transB)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.I8])
@pytest.mark.parametrize("transB", [0, 1])
def test_160_and_224_row_tiles(hip, dtype, transB):
    """whole tiles, M and N ending inside a tile, inside a wave's 80 and 112 rows and inside an atom; whole K tiles and partial ones of a chunk and of an element"""
    bk = BK[dtype]
    for M, N, K, tile in ((2400, 3584, 12 * bk, "160x256"), (2399, 3583, 12 * bk + 1, "160x256"), (2321, 3592, 15 * bk + 8, "160x256"), (3584, 4095, 14 * bk, "224x256"),
                          (3473, 3900, 13 * bk + 3, "224x256")):
        A = make_operand(dtype, *stored_shapes(M, N, K, 0, transB)[0], seed=91, tensor=0, scale=0.5)
        B = make_operand(dtype, *stored_shapes(M, N, K, 0, transB)[1], seed=91, tensor=1, scale=0.5)
        got, name, need = launch(hip, dtype, A, B, M, N, K, 0, transB, True, ldc_extra=int(M != 2400))
        assert tile in name and need == 0, (M, N, K, name, need)
        verify(dtype, got, A, B, 0, transB)


@pytest.mark.gpu
def test_160_row_tiles_apply_scales_and_accumulate(hip):
    """int8 with per-row and per-column scales (bit for bit) and into old int32 values, fp16 into old fp32 ones; rows off 16-byte boundaries behind copies"""
    M, N, K8, K16 = 2399, 3581, 1537, 772
    Ai, Bi = make_operand(O.I8, M, K8, 92, 0), make_operand(O.I8, N, K8, 92, 1)
    sA, sB = O.uniform(M, 92, 2, 0.001, 0.02), O.uniform(N, 92, 3, 0.001, 0.02)
    acc = O.gemm_i32(Ai, Bi, 0, 1)
    got = run_gemm(hip, O.I8, Ai, Bi, 0, 1, O.F16, M, N, K8, epilogue=hip.EPI_ROW_COL_SCALE, sA=sA, sB=sB, pad_c=0)
    assert np.array_equal(got, O.epilogue_rowcol_f16(acc, sA, sB))
    C0 = (np.arange(M * N, dtype=np.int64).reshape(M, N) % 91 - 45).astype(np.int32)
    assert np.array_equal(run_gemm(hip, O.I8, Ai, Bi, 0, 1, O.I32, M, N, K8, C_init=C0, clear_accum=False), acc + C0)
    Ah, Bh = make_operand(O.F16, M, K16, 93, 0, scale=0.5), make_operand(O.F16, K16, N, 93, 1, scale=0.5)
    Cf = O.uniform(M * N, 93, 2, -1.0, 1.0).reshape(M, N).astype(np.float32)
    assert "160x256" in hip.kernel_names()[hip.plan(hip.make_desc(O.F16, M, N, K16, dtype_out=O.F16)).kernel_id]
    got = run_gemm(hip, O.F16, Ah, Bh, 0, 0, O.F32, M, N, K16, C_init=Cf, clear_accum=False)
    r = O.compare(O.F32, np.ascontiguousarray(got), O.gemm_f64(O.F16, Ah, Bh) + Cf.astype(np.float64))
    assert r["nonfinite"] == 0 and r["max_rel"] <= TOL[O.F32] and r["fro_rel"] <= TOL[O.F32], r


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,transA,transB,aligned,size", [
    (O.F16, 0, 0, True, (1001, 1003, 4001)),   # 64 tiles of 128 x 128 in 4 slices
    (O.BF16, 1, 0, True, (17, 4096, 4096)),    # one row of tiles in 8 slices
    (O.I8, 1, 0, True, (300, 1088, 130 * 48 + 5)),  # 49 K tiles: 3 slices, the last one shorter and its last K tile partial
    (O.E4M3, 1, 1, True, (704, 512, 5760)),
    (O.F16, 0, 1, False, (1000, 1000, 4000 - 9)),   # behind the copies of both operands
    (O.F16, 0, 1, True, (2500, 1664, 4040)),   # 70 tiles of 256 x 256 in 3 slices
    (O.F16, 0, 0, True, (1500, 2816, 3016)),   # 88 tiles of 192 x 256 in 2
])
def test_edge_kernels_split_on_grids_of_half_a_round(hip, dtype, transA, transB, aligned, size):
    """every tile of the grid in slices of K of unequal length, and the same problem with no workspace in one pass"""
    M, N, K = size
    A = make_operand(dtype, *stored_shapes(M, N, K, transA, transB)[0], seed=87, tensor=0, scale=0.5)
    B = make_operand(dtype, *stored_shapes(M, N, K, transA, transB)[1], seed=87, tensor=1, scale=0.5)
    for workspace in (True, False):
        got, name, need = launch(hip, dtype, A, B, M, N, K, transA, transB, aligned, workspace=workspace, ldc_extra=1)
        if workspace:
            bm, bn = map(int, name.split("_")[2].split("x")[:2])
            tiles = -(-M // bm) * -(-N // bn)
            assert bm >= 128 and tiles <= 128 and need >= 2 * tiles * bm * bn * 4, (name, need)
        verify(dtype, got, A, B, transA, transB)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,tail", [(500, 1501, False), (500, 1503, False), (16 * 256 + 3, 15 * 256 + 17, True)])
def test_summed_edge_tiles_apply_scales_and_accumulate(hip, M, N, tail):
    """the second kernel of split edge tiles at ragged M and N: column scales of exactly N entries with N ending inside a quad of columns, rows of
    C off 16-byte boundaries, the tensor scale and the old values of C; int8 bit for bit"""
    K8, K16 = 8048, 4024 if not tail else 2008

    def split(*a, **kw):
        p = hip.plan(hip.make_desc(*a, transB=True, **kw))
        tiles = p.grid_x * p.grid_y % 256 if tail else p.grid_x * p.grid_y
        assert "_guard" in hip.kernel_names()[p.kernel_id] and p.workspace_bytes >= 2 * tiles * p.tile_m * p.tile_n * 4, (hip.kernel_names()[p.kernel_id], p.workspace_bytes)

    Ai, Bi = make_operand(O.I8, M, K8, 88, 0), make_operand(O.I8, N, K8, 88, 1)
    sA, sB = O.uniform(M, 88, 2, 0.001, 0.02), O.uniform(N, 88, 3, 0.001, 0.02)
    acc = O.gemm_i32(Ai, Bi, 0, 1)
    split(O.I8, M, N, K8, dtype_out=O.F16, epilogue=hip.EPI_ROW_COL_SCALE)
    got = run_gemm(hip, O.I8, Ai, Bi, 0, 1, O.F16, M, N, K8, epilogue=hip.EPI_ROW_COL_SCALE, sA=sA, sB=sB, pad_c=0)
    assert np.array_equal(got, O.epilogue_rowcol_f16(acc, sA, sB))
    C0 = (np.arange(M * N, dtype=np.int64).reshape(M, N) % 91 - 45).astype(np.int32)
    assert np.array_equal(run_gemm(hip, O.I8, Ai, Bi, 0, 1, O.I32, M, N, K8, C_init=C0, clear_accum=False), acc + C0)
    Ah, Bh = make_operand(O.F16, M, K16, 89, 0, scale=0.5), make_operand(O.F16, N, K16, 89, 1, scale=0.5)
    Cf = O.uniform(M * N, 89, 2, -1.0, 1.0).reshape(M, N).astype(np.float32)
    split(O.F16, M, N, K16, dtype_out=O.F32, clear_accum=False)
    got = run_gemm(hip, O.F16, Ah, Bh, 0, 1, O.F32, M, N, K16, C_init=Cf, clear_accum=False)
    r = O.compare(O.F32, np.ascontiguousarray(got), O.gemm_f64(O.F16, Ah, Bh, False, True) + Cf.astype(np.float64))
    assert r["nonfinite"] == 0 and r["max_rel"] <= TOL[O.F32] and r["fro_rel"] <= TOL[O.F32], r
    if not tail:
        A8, B8 = make_operand(O.E4M3, M, K8, 90, 0, scale=0.5), make_operand(O.E4M3, N, K8, 90, 1, scale=0.5)
        split(O.E4M3, M, N, K8, dtype_out=O.BF16, epilogue=hip.EPI_TENSOR_SCALE)
        got = run_gemm(hip, O.E4M3, A8, B8, 0, 1, O.BF16, M, N, K8, epilogue=hip.EPI_TENSOR_SCALE, sA=[0.25], sB=[0.02])
        r = O.compare(O.BF16, np.ascontiguousarray(got), O.epilogue_tensor(O.gemm_f64(O.E4M3, A8, B8, False, True), np.float32(0.25), np.float32(0.02)))
        assert r["nonfinite"] == 0 and r["max_rel"] <= TOL[O.BF16] and r["fro_rel"] <= TOL[O.BF16], r


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,transA,transB,tile", [(O.F16, 0, 0, "64x64"), (O.F16, 0, 1, "64x64"), (O.BF16, 0, 0, "64x64"), (O.BF16, 0, 1, "64x64"), (O.I8, 0, 1, "64x64"), (O.E4M3, 0, 1, "64x64"),
                                                      (O.F16, 1, 1, "128x128"), (O.BF16, 1, 0, "128x128"), (O.I8, 0, 0, "128x128"), (O.E4M3, 1, 0, "128x128"), (O.E4M3, 0, 0, "128x128"),
                                                      (O.F32, 0, 0, "32x32"), (O.F32, 0, 1, "32x32"), (O.F32, 1, 0, "32x32"), (O.F32, 1, 1, "32x32")])
def test_tiles_that_follow_up_on_few_larger_ones(hip, dtype, transA, transB, tile):
    """64x64 and 32x32 tiles whose waves share a K tile and the 128x128 edge tile in a ring of 3: one to seven K tiles, whole and partial; M and N
    at the end of a tile, one beyond it, and inside a chunk; rows on 16-byte boundaries and copied there; accumulation into C"""
    per = {"64x64": 128, "128x128": 64, "32x32": 128}[tile] * (1 if tile == "32x32" else 2 // ES[dtype])  # the K tile
    tiles = {"64x64": (1, 2, 3, 4, 7), "128x128": (13, 14, 16), "32x32": (1, 2, 3, 5)}[tile]
    ms = {"64x64": (128, 129, 255), "128x128": (130, 257, 383), "32x32": (96, 97, 127)}[tile]
    seen, cases = set(), []
    for n in tiles:
        for M, N, K in ((ms[0], 256, n * per), (ms[1], 200, n * per - 16), (ms[2], 333, n * per + 9)):
            cases += [(M, N, K, True), (M, N, K, False)]
    if tile == "64x64":  # whole tiles
        cases += [(576, 576, 4 * per, True), (960, 704, 8 * per, True)]
    for i, (M, N, K, aligned) in enumerate(cases):
        A = make_operand(dtype, *stored_shapes(M, N, K, transA, transB)[0], seed=91 + i, tensor=0, scale=0.5)
        B = make_operand(dtype, *stored_shapes(M, N, K, transA, transB)[1], seed=91 + i, tensor=1, scale=0.5)
        got, name, _ = launch(hip, dtype, A, B, M, N, K, transA, transB, aligned, ldc_extra=0 if M % 32 == 0 and aligned else 1)
        verify(dtype, got, A, B, transA, transB)
        if "_%sx" % tile in name and ("_s3" in name or tile == "32x32"):
            seen |= {-(-K // per), "plain" if re.search("_s[23]$", name) else "partial K" if K % per else "whole K", "aligned" if aligned else "copied"}
    assert seen >= set(tiles[1:]) | {"partial K", "aligned", "copied"} | ({"plain"} if tile == "64x64" or (tile == "32x32" and not transA and not transB) else set()), seen
    M, N, K = ms[1], 264, tiles[-1] * per - 16
    A = make_operand(dtype, *stored_shapes(M, N, K, transA, transB)[0], seed=99, tensor=0, scale=0.5)
    B = make_operand(dtype, *stored_shapes(M, N, K, transA, transB)[1], seed=99, tensor=1, scale=0.5)
    if dtype != O.I8:
        C0 = O.uniform(M * N, 99, 2, -1.0, 1.0).reshape(M, N).astype(np.float32)
        got = run_gemm(hip, dtype, A, B, transA, transB, O.F32, M, N, K, C_init=C0, clear_accum=False)
        r = O.compare(O.F32, np.ascontiguousarray(got), O.gemm_f64(dtype, A, B, transA, transB) + C0.astype(np.float64))
        assert r["nonfinite"] == 0 and r["max_rel"] <= TOL[O.F32] and r["fro_rel"] <= TOL[O.F32], r
