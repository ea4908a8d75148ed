"""The passes beside the products at the edges of their loops: the sums of split-K slices, reductions whose loads are under way several at a time
or in one launch, and the last group of a row in block bodies."""
import numpy as np
import pytest

import oracle as O
from helpers import TOL, make_operand, run_gemm
from oracle import tile_ops as T


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
@pytest.mark.parametrize("M,N,K,tile,slices", [
    (193, 123, 4608, 128, 2), (193, 123, 6144, 128, 3), (193, 128 * 32 - 5, 16384, 128, 4), (193, 128 * 25 - 5, 16384, 128, 5), (193, 128 * 21 - 5, 16384, 128, 6),
    (193, 128 * 18 - 5, 16384, 128, 7), (193, 128 * 16 - 5, 16384, 128, 8), (513, 6651, 4608, 192, 2), (513, 6651, 8192, 192, 3), (193, 128 * 64 - 5, 16384, 256, 7),
    (193, 128 * 42 - 5, 16384, 256, 8)])
def test_the_sum_of_split_edge_tiles_is_exact(hip, M, N, K, tile, slices):
    """2 to 8 slices of edge tiles, in place of as many work-groups as there are CUs; B's rows are copied to aligned ones first, the sums lie behind them"""
    p = hip.plan(hip.make_desc(O.I8, M, N, K, dtype_out=O.I32))
    copies = -(-K * (-(-N // 16) * 16) // 256) * 256
    assert p.tile_m == tile and p.workspace_bytes - copies == slices * p.grid_x * p.grid_y * p.tile_m * p.tile_n * 4
    A, B = make_operand(O.I8, M, K, 62, 0), make_operand(O.I8, K, N, 62, 1)
    assert np.array_equal(run_gemm(hip, O.I8, A, B, 0, 0, O.I32, M, N, K), O.gemm_i32(A, B))


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [O.F32, O.F16, O.BF16])
@pytest.mark.parametrize("rows,cols,dim", [
    (129, 8, 0), (1023, 40, 0), (1024, 65, 0), (1025, 500, 0), (1535, 9, 0), (1536, 64, 0), (1537, 64, 0), (1200, 16384, 0), (1200, 16385, 0), (1500, 3, 0),  # one launch, and beyond it
    (3, 2049, 1), (3, 4096, 1), (2, 8191, 1), (2, 8192, 1), (5, 8193, 1), (3, 10248, 1), (2, 40000, 1), (1, 65543, 1)])                                        # 1 to 5 groups a lane, slices
def test_reductions_with_several_loads_under_way(hip, dt, rows, cols, dim):
    import torch
    ld, st = cols + 3, O.NP_STORAGE[dt]
    vals = O.encode(dt, O.normal(rows * cols, 63, 0, 1.0)).reshape(rows, cols)
    src = np.zeros((rows, ld), st)
    src[:, :cols] = vals
    x = torch.from_numpy(src.view(np.uint8).reshape(-1).copy()).cuda()
    kept = rows if dim == 1 else cols
    old = O.encode(dt, O.normal(kept, 63, 1, 0.5))
    need = hip.reduce_workspace_bytes(dt, rows, cols, dim)
    ws = torch.full((max(need, 4),), 0xFF, dtype=torch.uint8, device="cuda")
    for kind, clear in (("max", True), ("min", False), ("add", True), ("add", False)):
        d = torch.from_numpy(old.view(np.uint8).reshape(-1).copy()).cuda()
        hip.reduce(dt, x.data_ptr(), rows, cols, ld, dim, kind, clear, d.data_ptr(), ws.data_ptr() if need else None, need, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        got = d.cpu().numpy().view(st)
        if kind != "add":
            assert np.array_equal(got, T.reduce(dt, vals, dim, kind, None if clear else old)), (kind, clear)
            continue
        want = T.reduce_f64(dt, vals, dim, kind, None if clear else old).astype(np.float64).reshape(-1)
        # one rounding to the element type of |sum| <= sum of |x|, and fp32 sums of at most 64 + 10 additions in a row each
        size = np.abs(O.decode(dt, vals).astype(np.float64)).sum(axis=dim).reshape(-1) + np.abs(O.decode(dt, old).astype(np.float64))
        bound = {O.F32: 2.0 ** -24, O.F16: 2.0 ** -11, O.BF16: 2.0 ** -8}[dt] * np.abs(want) + 2.0 ** -24 * 80 * size
        assert np.all(np.abs(O.decode(dt, got).astype(np.float64) - want) <= bound)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [O.F32, O.F16, O.BF16])
@pytest.mark.parametrize("pitch", ["dense", "lines", "odd"])
def test_the_last_group_of_columns_reduced_in_one_launch(hip, dt, pitch):
    """a last group of 1 to all but one columns, alone in its strip, with others and behind whole strips, of rows that start on 128-byte lines or anywhere; what
    lies between the rows is no number.  Whole numbers whose sums every type holds: the same bits in any order."""
    import torch
    es, G = O.NP_STORAGE[dt]().itemsize, 16 // O.NP_STORAGE[dt]().itemsize
    tdt = {O.F32: torch.float32, O.F16: torch.float16, O.BF16: torch.bfloat16}[dt]
    g = torch.Generator(device="cuda").manual_seed(6)
    for rows in (120, 1152, 1153, 1536):
        for cols in [G - 1, G, 2 * G + 1] + [8 * G * k + r for k in (1, 3) for r in (0, 1, G - 1, G + 2, 8 * G - 1)]:
            ld = {"dense": cols, "lines": -(-cols * es // 128) * 128 // es, "odd": cols + 1 + (cols & 1)}[pitch]
            x = torch.full((rows, ld), float("nan"), device="cuda", dtype=tdt)
            x[:, :cols] = (torch.rand(rows, cols, device="cuda", generator=g) < 0.06).to(tdt) * (2 * torch.randint(0, 2, (rows, cols), device="cuda", generator=g) - 1).to(tdt)
            need = hip.reduce_workspace_bytes(dt, rows, cols, 0)
            ws = torch.full((max(need, 4),), 0xFF, dtype=torch.uint8, device="cuda")
            for with_ws in (True, False):
                d = torch.full((cols + 1,), 7.0, device="cuda", dtype=tdt)
                hip.reduce(dt, x.data_ptr(), rows, cols, ld, 0, "add", True, d.data_ptr(), ws.data_ptr() if need and with_ws else None, need if with_ws else 0, torch.cuda.current_stream().cuda_stream)
                torch.cuda.synchronize()
                assert torch.equal(d[:cols].float(), x[:, :cols].float().sum(0)) and float(d[cols]) == 7.0, (rows, cols, ld, with_ws)


@pytest.mark.gpu
@pytest.mark.parametrize("dt,tdt", [(O.F32, "float32"), (O.F16, "float16"), (O.BF16, "bfloat16")])
@pytest.mark.parametrize("rows", [1, 5, 2600])
def test_the_last_group_of_a_row(hip, dt, tdt, rows):
    """rows of a whole number of groups of 8 columns and of 1 to 7 columns more, shorter than a group, than a wave, than a work-group and longer; into
    another matrix and into its own operand.  Every operation rounds to fp32 once, as torch's do: the same bits."""
    import torch
    tdt = getattr(torch, tdt)
    g = torch.Generator(device="cuda").manual_seed(5)
    stream = torch.cuda.current_stream().cuda_stream
    for cols in (1, 5, 7, 8, 9, 12, 15, 17, 127, 131, 511, 513, 518, 2047, 2054) + ((20003,) if rows < 100 else ()):
        ld = cols + 1
        x, z = (torch.randn(rows, ld, device="cuda", generator=g).to(tdt) for _ in range(2))
        r, c = torch.randn(rows, device="cuda", generator=g).to(tdt), torch.randn(cols, device="cuda", generator=g).to(tdt)
        body = [("input", 0), ("input", 1), "sub", ("input", 2), "mul", ("input", 3), "add"]
        for operands, program, want in (
                ([x, r, c, z], body, (x.float()[:, :cols] - r.float()[:, None]) * c.float() + z.float()[:, :cols]),
                ([x, z], [("input", 0), ("input", 1), "add"], x.float()[:, :cols] + z.float()[:, :cols]),
                ([x], [("input", 0), ("const", 0.75), "mul"], x.float()[:, :cols] * 0.75)):
            strides = [(dt, ld, 1) if t is x or t is z else (dt, 1, 0) if t is r else (dt, 0, 1) for t in operands]
            desc = hip.make_elementwise_desc(program, strides, dt, rows, cols, out_ld=ld)
            for out in (torch.full_like(x, 3.0), x.clone()):
                beside = out[:, cols:].clone()
                ins = [out if t is x and bool((out == x).all()) else t for t in operands]
                hip.elementwise(desc, [t.data_ptr() for t in ins], out.data_ptr(), stream)
                torch.cuda.synchronize()
                assert torch.equal(out[:, :cols], want.to(tdt)) and torch.equal(out[:, cols:], beside), (rows, cols, len(operands))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,transA,transB", [(O.F16, 0, 0), (O.F16, 1, 0), (O.BF16, 0, 1), (O.I8, 0, 0), (O.I8, 0, 1), (O.E4M3, 0, 0), (O.E4M3, 0, 1)])
def test_slices_of_unequal_length(hip, dtype, transA, transB):
    """numbers of K tiles that no number of slices divides, a few rows to a few hundred, off the tiles and on them: the last slice is the shorter one"""
    bk, seen = {O.F16: 64, O.BF16: 64, O.I8: 128, O.E4M3: 128}[dtype], 0
    for M, N, tiles in ((4, 576, 53), (32, 512, 59), (58, 2240, 59), (64, 1024, 53), (128, 512, 31), (198, 896, 59), (256, 768, 43)):
        if (transA and M % 32) or (transB and M <= 64):
            continue
        K = bk * tiles * (2 if transB else 1)
        p = hip.plan(hip.make_desc(dtype, M, N, K, transA=transA, transB=transB, dtype_out={O.I8: O.I32, O.E4M3: O.BF16}.get(dtype, dtype)))
        seen += (K // p.tile_k) % p.split_k != 0
        A = make_operand(dtype, *((K, M) if transA else (M, K)), 64, 0, scale=0.5)
        B = make_operand(dtype, *((N, K) if transB else (K, N)), 64, 1, scale=0.5)
        out = {O.I8: O.I32, O.E4M3: O.BF16}.get(dtype, dtype)
        got = run_gemm(hip, dtype, A, B, transA, transB, out, M, N, K)
        if dtype == O.I8:
            assert np.array_equal(got, O.gemm_i32(A, B, transA, transB)), (M, N, K)
        else:
            r = O.compare(out, np.ascontiguousarray(got), O.gemm_f64(dtype, A, B, transA, transB))
            assert r["nonfinite"] == 0 and r["max_rel"] <= TOL[dtype] and r["fro_rel"] <= TOL[dtype], (M, N, K, r)
    assert seen


@pytest.mark.gpu
@pytest.mark.parametrize("dt,tdt", [(O.F32, "float32"), (O.F16, "float16"), (O.BF16, "bfloat16")])
def test_the_last_group_of_a_row_reduced(hip, dt, tdt):
    """rows shared by lanes of a wave, of 256 and 512 lanes and of several work-groups, with a last group of 1 to all but one elements; what lies between the rows is no
    number.  Whole numbers whose sums every type holds: the same bits in any order."""
    import torch
    tdt = getattr(torch, tdt)
    G = 16 // torch.empty(0, dtype=tdt).element_size()
    g = torch.Generator(device="cuda").manual_seed(7)
    stream = torch.cuda.current_stream().cuda_stream
    for cols in (1, G - 1, G, G + 1, 63 * G + 1, 64 * G - 1, 128 * G + 1, 256 * G - 1, 256 * G + 1, 1024 * G - 1, 1024 * G + 3, 2049 * G, 4096 * G - 1, 4096 * G + 1, 9000 * G + 5):
        for rows in (1, 3, 700 if cols < 300 * G else 5) + ((16600,) if cols in (256 * G + 1, 1024 * G + 3) else ()):
            x = torch.full((rows, cols + 1), float("nan"), device="cuda", dtype=tdt)
            x[:, :cols] = (torch.rand(rows, cols, device="cuda", generator=g) < 0.06).to(tdt) * (2 * torch.randint(0, 2, (rows, cols), device="cuda", generator=g) - 1).to(tdt)
            need = hip.reduce_workspace_bytes(dt, rows, cols, 1)
            ws = torch.full((max(need, 4),), 0xFF, dtype=torch.uint8, device="cuda")
            for kind, clear in (("add", True), ("add", False), ("max", True)):
                d = torch.full((rows + 1,), 7.0, device="cuda", dtype=tdt)
                hip.reduce(dt, x.data_ptr(), rows, cols, cols + 1, 1, kind, clear, d.data_ptr(), ws.data_ptr() if need else None, need, stream)
                torch.cuda.synchronize()
                want = x[:, :cols].float().sum(1) + (0 if clear else 7.0) if kind == "add" else x[:, :cols].float().amax(1)
                assert torch.equal(d[:rows].float(), want) and float(d[rows]) == 7.0, (rows, cols, kind, clear)


@pytest.mark.gpu
@pytest.mark.parametrize("dt,tdt,tol", [(O.F32, "float32", 2e-5), (O.F16, "float16", 2e-3), (O.BF16, "bfloat16", 8e-3)])
def test_softmax_of_rows_held_in_registers(hip, dt, tdt, tol):
    """rows at the edges of what a number of groups per lane holds, starting on any element, in matrices that the caches are read through and past (from 112 MiB on, where the
    first group is a part too); what lies between the rows is no number and stays as it is.  Bar: that of the other softmax tests."""
    import torch
    tdt = getattr(torch, tdt)
    es = torch.empty(0, dtype=tdt).element_size()
    G = 16 // es
    g = torch.Generator(device="cuda").manual_seed(8)
    stream = torch.cuda.current_stream().cuda_stream
    edges = [G * k + r for k in (256, 512, 768, 1024, 1536, 2048, 3072, 4096) for r in (-1, 0, 1)]
    many = [(-(-(112 << 20) // (cols * es)) + 1, cols) for cols in (256 * G + 1, 512 * G, 512 * G - 1, 4096 * G - 1, 4096 * G)]
    for rows, cols in [(3, c) for c in edges + [1, G - 1, G + 1, 64 * G + 3, 129 * G - 1]] + many:
        for ld, shift in ((cols + 1, 0), (cols + 3, 1), (-(-cols // G) * G + G, G - 1)) if rows == 3 else ((cols + 1, 1),):
            base = torch.full((shift + rows * ld,), float("nan"), device="cuda", dtype=tdt)
            x = base[shift:].view(rows, ld)
            x[:, :cols] = (torch.randn(rows, cols, device="cuda", generator=g) * 3).to(tdt)
            out = torch.full_like(base, 5.0)
            y, lse = out[shift:].view(rows, ld), torch.full((rows,), float("nan"), device="cuda")
            hip.softmax(dt, x.data_ptr(), ld, y.data_ptr(), ld, rows, cols, 1.25, lse.data_ptr(), stream)
            torch.cuda.synchronize()
            z = x[:, :cols].double() * (1.25 * 0.6931471805599453)
            want, want_lse = torch.softmax(z, 1), torch.logsumexp(z, 1) / 0.6931471805599453
            scale = torch.maximum(want, want.square().mean().sqrt())
            assert bool(((y[:, :cols].double() - want).abs() <= tol * scale + (2.0 ** -25 if dt == O.F16 else 0)).all()), (rows, cols, ld, shift)
            assert float((lse.double() - want_lse).abs().max()) <= 1e-4 * max(1.0, float(want_lse.abs().max())), (rows, cols, ld, shift)
            assert bool((y[:, cols:] == 5.0).all()) and bool((out[:shift] == 5.0).all()), (rows, cols, ld, shift)
            del z, want, scale


@pytest.mark.gpu
@pytest.mark.parametrize("dt,tdt", [(O.F32, "float32"), (O.F16, "float16"), (O.BF16, "bfloat16")])
def test_columns_of_long_rows_in_one_launch_and_beyond(hip, dt, tdt):
    """both sides of the numbers of rows up to which rows of 14 and 20 KiB on 128-byte lines are summed in one launch; the same rows off lines and without a workspace.  Whole numbers
    whose sums every type holds"""
    import torch
    tdt = getattr(torch, tdt)
    es = torch.empty(0, dtype=tdt).element_size()
    g = torch.Generator(device="cuda").manual_seed(10)
    for kib, rows in ((14, 2048), (14, 2049), (20, 3072), (20, 3073)):
        for cols in (kib * 1024 // es, kib * 1024 // es - 64, kib * 1024 // es + 3):
            for ld in (-(-cols * es // 128) * 128 // es, cols + 1 + (cols & 1)):
                x = torch.full((rows, ld), float("nan"), device="cuda", dtype=tdt)
                x[:, :cols] = ((torch.rand(rows, cols, device="cuda", generator=g) < 0.03).float() * (2 * torch.randint(0, 2, (rows, cols), device="cuda", generator=g) - 1).float()).to(tdt)
                need = hip.reduce_workspace_bytes(dt, rows, cols, 0)
                ws = torch.full((max(need, 4),), 0xFF, dtype=torch.uint8, device="cuda")
                for with_ws in (True, False):
                    d = torch.full((cols + 1,), 7.0, device="cuda", dtype=tdt)
                    hip.reduce(dt, x.data_ptr(), rows, cols, ld, 0, "add", False, d.data_ptr(), ws.data_ptr() if with_ws else None, need if with_ws else 0, torch.cuda.current_stream().cuda_stream)
                    torch.cuda.synchronize()
                    assert torch.equal(d[:cols].float(), x[:, :cols].float().sum(0) + 7) and float(d[cols]) == 7.0, (rows, cols, ld, with_ws)


@pytest.mark.gpu
@pytest.mark.parametrize("dt,tdt", [(O.F32, "float32"), (O.F16, "float16"), (O.BF16, "bfloat16")])
def test_row_reductions_on_and_off_boundaries(hip, dt, tdt):
    """rows of whole groups and not, on 16-byte boundaries and off them, on 256 and 512 lanes and on lanes of a wave with one, two and four groups each; what lies between the rows is no number.  Whole
    numbers whose sums every type holds: the same bits in any order"""
    import torch
    tdt = getattr(torch, tdt)
    G = 16 // torch.empty(0, dtype=tdt).element_size()
    g = torch.Generator(device="cuda").manual_seed(11)
    stream = torch.cuda.current_stream().cuda_stream
    for rows, cols in ((1030, 1300 * G), (1030, 1300 * G + 1), (1030, 1536 * G - 1), (1030, 1537 * G), (1024, 1025 * G), (1030, 1024 * G), (1030, 257 * G - 1), (2000, 256 * G), (2000, 129 * G), (2000, 128 * G - 1), (2000, 65 * G - 1),
                       (2000, 64 * G), (5000, 3 * G), (5000, 3 * G + 1), (5000, G), (5000, G - 1)):
        for ld, shift in ((-(-cols // G) * G, 0), (-(-cols // G) * G + G, 0), (cols + 1, 0), (-(-cols // G) * G, 1)):
            base = torch.full((shift + rows * ld,), float("nan"), device="cuda", dtype=tdt)
            x = base[shift:].view(rows, ld)
            x[:, :cols] = (torch.rand(rows, cols, device="cuda", generator=g) < 0.06).to(tdt) * (2 * torch.randint(0, 2, (rows, cols), device="cuda", generator=g) - 1).to(tdt)
            for kind in ("add", "min"):
                d = torch.full((rows + 1,), 7.0, device="cuda", dtype=tdt)
                hip.reduce(dt, x.data_ptr(), rows, cols, ld, 1, kind, True, d.data_ptr(), None, 0, stream)
                torch.cuda.synchronize()
                want = x[:, :cols].float().sum(1) if kind == "add" else x[:, :cols].float().amin(1)
                assert torch.equal(d[:rows].float(), want) and float(d[rows]) == 7.0, (rows, cols, ld, shift, kind)


@pytest.mark.gpu
@pytest.mark.parametrize("dt,tdt,tol", [(O.F32, "float32", 2e-5), (O.F16, "float16", 2e-3), (O.BF16, "bfloat16", 8e-3)])
def test_softmax_of_whole_groups(hip, dt, tdt, tol):
    """rows of whole groups, on 128-byte lines and off them, at the edges of what a number of groups per lane holds, up to 56 MiB and beyond, into another matrix and in place; what lies between
    the rows stays as it is.  Bar: that of the other softmax tests."""
    import torch
    tdt = getattr(torch, tdt)
    es = torch.empty(0, dtype=tdt).element_size()
    G = 16 // es
    g = torch.Generator(device="cuda").manual_seed(13)
    stream = torch.cuda.current_stream().cuda_stream
    views = [(5, G * k, pad) for k in (1, 3, 64, 65, 128, 129, 256, 257, 512, 513, 768, 769, 1024, 1025, 1536, 1537, 2048, 2049, 3072, 3073, 4096) for pad in (0, G)]
    views += [(1000, 24, 0), (1000, G, G), (-(-(56 << 20) // (512 * 16)) + 1, 512 * G, 0), (-(-(120 << 20) // (600 * 16)), 600 * G, 0)]
    for rows, cols, pad in views:
        ld = cols + pad
        x = torch.full((rows, ld), float("nan"), device="cuda", dtype=tdt)
        x[:, :cols] = (torch.randn(rows, cols, device="cuda", generator=g) * 3).to(tdt)
        z = x[:, :cols].double() * (1.25 * 0.6931471805599453)
        want = torch.softmax(z, 1)
        scale = torch.maximum(want, want.square().mean().sqrt())
        for y in (torch.full_like(x, 5.0), x):
            beside = y[:, cols:].clone()
            hip.softmax(dt, x.data_ptr(), ld, y.data_ptr(), ld, rows, cols, 1.25, None, stream)
            torch.cuda.synchronize()
            assert bool(((y[:, :cols].double() - want).abs() <= tol * scale + (2.0 ** -25 if dt == O.F16 else 0)).all()), (rows, cols, ld)
            assert torch.equal(y[:, cols:].nan_to_num(3.0), beside.nan_to_num(3.0)), (rows, cols, ld)
        del z, want, scale


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [4100, 5003, 6144])
def test_sums_of_rows_on_256_lanes_are_no_further_from_the_exact_ones_than_on_512(hip, cols):
    """fp32 rows of 1025 to 1536 groups, more than 1024 of them, against the error of 512 lanes that add their elements one after the other, then in pairs"""
    import torch
    rows, lanes = 2000, 512
    vals = O.normal(rows * cols, 65, 0, 1.0).astype(np.float32).reshape(rows, cols)
    exact = vals.astype(np.float64).sum(1)
    chains = np.zeros((rows, lanes), np.float32)
    for c in range(0, cols, 4 * lanes):
        for e in range(4):
            part = vals[:, c + e:min(c + 4 * lanes, cols):4]
            chains[:, :part.shape[1]] += part
    while chains.shape[1] > 1:
        half = chains.shape[1] // 2
        chains = chains[:, :half] + chains[:, half:]
    x, d = torch.from_numpy(vals).cuda(), torch.empty(rows, device="cuda")
    hip.reduce(O.F32, x.data_ptr(), rows, cols, cols, 1, "add", True, d.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert np.linalg.norm(d.cpu().numpy().astype(np.float64) - exact) <= np.linalg.norm(chains[:, 0].astype(np.float64) - exact)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(4100, 4096), (4097, 4097), (8, 2097153), (50000, 400), (45003, 403), (600000, 33), (600000, 31), (9000, 7500)])
def test_32_bit_bodies_of_views_on_either_side_of_64_and_256_mib(hip, rows, cols):
    """stores through the caches and past them, of rows of whole groups and not, longer than a wave and shorter, into another matrix and into its own operand; every operation rounds once, as torch's do"""
    import torch
    g, ld, stream = torch.Generator(device="cuda").manual_seed(14), cols + 1, torch.cuda.current_stream().cuda_stream
    x = torch.randn(rows, ld, device="cuda", generator=g)
    r, c = torch.randn(rows, device="cuda", generator=g), torch.randn(cols, device="cuda", generator=g)
    desc = hip.make_elementwise_desc([("input", 0), ("input", 1), ("const", 0.5), "mul", "sub", ("input", 2), "mul"], [(O.F32, ld, 1), (O.F32, 1, 0), (O.F32, 0, 1)], O.F32, rows, cols, out_ld=ld)
    want = (x[:, :cols] - r[:, None] * 0.5) * c
    for out in (torch.full_like(x, 3.0), x):
        beside = out[:, cols:].clone()
        hip.elementwise(desc, [x.data_ptr(), r.data_ptr(), c.data_ptr()], out.data_ptr(), stream)
        torch.cuda.synchronize()
        assert torch.equal(out[:, :cols], want) and torch.equal(out[:, cols:], beside)
