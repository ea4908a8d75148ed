"""Deep products of up to two rounds of 128x128 tiles, which run on 256x256 edge tiles in slices of K: which ones, and what they give."""
import pytest

import oracle as O
from frisk_amd import runtime as R

# (M, N, K, slices of the 256x256 tiles that `workspace_bytes` is for; 0: another tile)
ROUTES = [(1777, 1216, 7488, 7), (2043, 1144, 9024, 6), (1213, 2370, 9984, 5), (2669, 1256, 7424, 0), (2560, 1025, 7488, 5), (1137, 2880, 11968, 4), (511, 2264, 10496, 8), (511, 2264, 10432, 0),
          (600, 5214, 8192, 4), (600, 5214, 8128, 0), (1777, 1216, 7424, 0), (1512, 2624, 10368, 0), (2095, 1856, 9472, 0), (250, 6400, 9024, 0), (2048, 2048, 8192, 0), (3000, 4096, 8192, 0),
          (1019, 5408, 6912, 2), (1347, 4288, 6080, 0), (1012, 4640, 4352, 3), (1012, 4640, 4288, 0), (700, 1216, 9024, 0)]


def routed(p):
    return "256x256x64_w2x2_s2x3_a16_edge" in R.kernel_names()[p.kernel_id]


@pytest.mark.parametrize("dtype", [O.F16, O.BF16])
@pytest.mark.parametrize("transB", [0, 1])
@pytest.mark.parametrize("M,N,K,slices", ROUTES)
def test_which_problems(dtype, transB, M, N, K, slices):
    ld = (N + 7) // 8 * 8
    d = R.make_desc(dtype, M, N, K, transB=transB, ldb=K if transB else ld, ldc=ld)
    p = R.plan(d)
    where = (R.kernel_names()[p.kernel_id], p.workspace_bytes)
    if slices:
        assert routed(p) and p.workspace_bytes == slices * p.grid_x * p.grid_y * 256 * 256 * 4 == R.workspace_bytes(d), where
    else:
        assert not routed(p) or p.workspace_bytes == 0, where  # (whole grids of 256x256 tiles may be the planner's choice in one pass)


@pytest.mark.parametrize("dtype,M,N,K,slices", [(O.E4M3, 944, 3472, 16384, (4, 0)), (O.E4M3, 944, 3472, 16256, (0, 0)), (O.E4M3, 944, 3472, 18304, (4, 0)), (O.E4M3, 944, 3472, 18432, (4, 4)),
                                                (O.I8, 1333, 2200, 16256, (0, 0)), (O.I8, 1333, 2200, 18304, (4, 0)), (O.I8, 1333, 2200, 18432, (4, 4))])
def test_four_slices_of_8_bit_types_by_the_layout_of_B(dtype, M, N, K, slices):
    """against B [N][K], which the 128x128 tiles read faster, two K tiles in seven later: at 16384 it was slower from memory too"""
    for transB in (0, 1):
        ld = (N + 15) // 16 * 16
        p = R.plan(R.make_desc(dtype, M, N, K, transB=transB, ldb=K if transB else ld, ldc=ld, dtype_out={O.I8: O.I32, O.E4M3: O.BF16}[dtype]))
        got = p.workspace_bytes // (p.grid_x * p.grid_y * 256 * 256 * 4) if p.tile_m == p.tile_n == 256 else 0
        assert got == slices[transB], (transB, R.kernel_names()[p.kernel_id], p.workspace_bytes)


@pytest.mark.parametrize("dtype", [O.I8, O.E4M3])
@pytest.mark.parametrize("M,N,K,sliced", [(1249, 1520, 16512, 1), (1152, 2368, 14592, 1), (1152, 2368, 14464, 0), (944, 3472, 18432, 1), (1921, 2848, 12032, 1), (1921, 2848, 11904, 0), (1196, 4320, 8576, 1)])
def test_which_problems_of_8_bit_types(dtype, M, N, K, sliced):
    for transB in (0, 1):
        ld = (N + 15) // 16 * 16
        p = R.plan(R.make_desc(dtype, M, N, K, transB=transB, ldb=K if transB else ld, ldc=ld, dtype_out={O.I8: O.I32, O.E4M3: O.BF16}[dtype]))
        assert sliced == (p.tile_m == p.tile_n == 256 and p.workspace_bytes > 0), (transB, R.kernel_names()[p.kernel_id], p.workspace_bytes)


@pytest.mark.parametrize("change", [dict(tile=(128, 128, 0)), dict(split_k=1), dict(policy=R.POLICY_FULL_ROW)])
def test_what_a_descriptor_asks_for_stays(change):
    """a tile, a number of slices or a wave policy that the descriptor names"""
    assert routed(R.plan(R.make_desc(O.F16, 1777, 1216, 7488)))
    try:
        p = R.plan(R.make_desc(O.F16, 1777, 1216, 7488, **change))
    except R.FriskHipError:
        assert "policy" in change  # (no kernel under that wave policy)
        return
    assert not routed(p), R.kernel_names()[p.kernel_id]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [O.F16, O.BF16])
@pytest.mark.parametrize("transA,transB", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_their_results(hip, dtype, transA, transB):
    """whole numbers, exact in any order: C off its tiles and packed, old values, scales, 16- and 32-bit C"""
    from test_edge_stores_gpu import check
    for M, N, K in ((1784, 1216, 7488), (1336, 1736, 8192), (2208, 904, 9024), (512, 2264, 10496), (1016, 4640, 4352), (1016, 5408, 6912)):
        for out in (dtype, O.F32):
            p = hip.plan(hip.make_desc(dtype, M, N, K, dtype_out=out, transA=transA, transB=transB, ldc=(N + 7) // 8 * 8 + 8, clear_accum=False))
            assert routed(p) and p.workspace_bytes, (M, N, K, out)
            check(hip, dtype, transA, transB, M, N, K, out, hip.EPI_NONE, False, (N + 7) // 8 * 8 + 8, 0)
            check(hip, dtype, transA, transB, M, N, K, out, hip.EPI_ROW_COL_SCALE, True, N, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [O.I8, O.E4M3])
@pytest.mark.parametrize("transB", [0, 1])
def test_their_results_in_8_bit_types(hip, dtype, transB):
    from test_edge_stores_gpu import check
    for M, N, K in ((1249, 1520, 16512), (944, 3472, 18432), (1200, 4320, 8576), (1921, 2848, 12032)):
        for out in ((O.I32, O.F32) if dtype == O.I8 else (O.BF16, O.F32)):
            p = hip.plan(hip.make_desc(dtype, M, N, K, dtype_out=out, transB=transB, ldc=(N + 15) // 8 * 8, clear_accum=False))
            assert p.tile_m == p.tile_n == 256 and p.workspace_bytes, (M, N, K, out)
            check(hip, dtype, 0, transB, M, N, K, out, hip.EPI_NONE, False, (N + 15) // 8 * 8, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("share", [0, 3, 4, 5, 7])
def test_with_less_workspace(hip, share):
    """slices that the workspace does not hold fall away; below five another tile takes the problem (test_launches.py says which)"""
    import torch
    M, N, K = 1777, 1216, 7488
    g = torch.Generator(device="cuda").manual_seed(share)
    A, B = (torch.randint(-2, 3, s, device="cuda", generator=g).half() for s in ((M, K), (K, N)))
    C = torch.full((M, N), 7.0, device="cuda")
    d = hip.make_desc(O.F16, M, N, K, dtype_out=O.F32)
    need = share * 35 * 256 * 256 * 4
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    hip.gemm(d, A.data_ptr(), B.data_ptr(), C.data_ptr(), None, None, ws.data_ptr() if need else None, need, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(C, A.float() @ B.float())
