"""Where one row of tiles runs in launch order instead of regrouped by XCD: B stored [K][N] with rows a multiple of 2 KiB apart."""
import pytest

import oracle as O
from frisk_amd import runtime as R


@pytest.mark.parametrize("dtype,M,N,K,transB,ldb,regrouped", [
    (O.F16, 48, 8192, 8192, 0, 8192, 0), (O.I8, 16, 8192, 2048, 0, 8192, 0), (O.F16, 48, 8000, 8192, 0, 8192, 0), (O.F16, 48, 8192, 8192, 0, 8200, 1), (O.F16, 48, 8192, 8192, 1, 8192, 1),
    (O.F16, 300, 8192, 1024, 0, 8192, 1), (O.F32, 30, 4096, 512, 0, 4096, 0), (O.E4M3, 8, 5184, 4096, 0, 5184, 1)])
def test_which_grids_stay_in_launch_order(dtype, M, N, K, transB, ldb, regrouped):
    p = R.plan(R.make_desc(dtype, M, N, K, transB=transB, ldb=ldb, dtype_out={O.I8: O.I32, O.E4M3: O.BF16}.get(dtype)))
    assert p.xcd_remap == regrouped and (not regrouped or p.grid_x * p.grid_y >= 8)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [O.F16, O.BF16, O.I8, O.E4M3, O.F32])
def test_products_in_launch_order(hip, dtype):
    """whole numbers: exact on every tile, in one pass and in slices, in grids of 8 columns or fewer and more"""
    from test_edge_stores_gpu import check
    for M in (1, 32, 48):
        for N, K in ((1024, 512), (2048, 640), (4096, 2048), (4000, 2048)):
            check(hip, dtype, 0, 0, M, N, K, {O.I8: O.I32, O.E4M3: O.BF16}.get(dtype, dtype) if dtype == O.I8 else O.F32, hip.EPI_NONE, True, N, 0)
