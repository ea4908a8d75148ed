"""The passes beside the products at the edges of their loops: the sums of split-K slices and of split edge tiles."""
or in one launch, and the last group of a row in block bodies."""
import numpy as np
import pytest

import oracle as O
from helpers import make_operand, run_gemm


@pytest.mark.gpu
@pytest.mark.parametrize("split", [2, 3, 5, 6, 7, 8, 9, 15, 16])
def test_the_sum_of_any_number_of_slices_is_exact(hip, split):
    """int8 products are whole numbers: every slice once, whole quads and a row's last one; into int32 on old values, into fp16 with scales"""
    M, N, K = 40, 130, 128 * 2 * split
    A, B = make_operand(O.I8, M, K, 61, 0), make_operand(O.I8, K, N, 61, 1)
    want = O.gemm_i32(A, B)
    C0 = (np.arange(M * N, dtype=np.int32).reshape(M, N) * 7919) % 100003
    got = run_gemm(hip, O.I8, A, np.pad(B, ((0, 0), (0, 14))), 0, 0, O.I32, M, N, K, C_init=C0, clear_accum=False, split_k=split, pad_c=2)
    assert np.array_equal(got, want + C0)
    sA, sB = O.uniform(M, 61, 2, 0.001, 0.02), O.uniform(N, 61, 3, 0.001, 0.02)
    got = run_gemm(hip, O.I8, A, np.pad(B, ((0, 0), (0, 14))), 0, 0, O.F16, M, N, K, epilogue=hip.EPI_ROW_COL_SCALE, sA=sA, sB=sB, split_k=split, pad_c=6)
    assert np.array_equal(got, O.epilogue_rowcol_f16(want, sA, sB))


@pytest.mark.gpu
@pytest.mark.parametrize("columns", [64, 42, 32, 25, 21, 18, 16])
def test_the_sum_of_split_edge_tiles_is_exact(hip, columns):
    """two rows of 128x128 edge tiles over K tiles enough for 2 to 8 slices, in place of as many work-groups as there are CUs"""
    M, N, K = 193, 128 * columns - 5, 128 * 16 * 8
    A, B = make_operand(O.I8, M, K, 62, 0), make_operand(O.I8, K, N, 62, 1)
    assert np.array_equal(run_gemm(hip, O.I8, A, B, 0, 0, O.I32, M, N, K), O.gemm_i32(A, B))
