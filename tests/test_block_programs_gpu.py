"""The interpreter of frisk.block bodies at the edges of its step machine: programs of more than one chunk of steps, the deepest stack,
every operation with its right operand a constant, a value of the row, a value of the column, a second walking operand or a
value from below, more broadcast operands than there are slots, mixed element types, rows of any length and alignment."""
import numpy as np
import pytest

import oracle as O
from oracle import tile_ops as T

ES = {O.F32: 4, O.F16: 2, O.BF16: 2}
TOL = {O.F32: 3e-6, O.F16: 1e-3, O.BF16: 8e-3}
BINARY = ["add", "sub", "mul", "div", "max", "min"]


def run(hip, prog, operands, out_dt, rows, cols, in_place=None):
    """operands: (dtype, kind, values as float) with kind walk | row | col | one; walking rows are one element longer than cols"""
    import torch
    bufs, ins, refs = [], [], []
    for dt, kind, vals in operands:
        st = O.encode(dt, np.ascontiguousarray(vals, dtype=np.float32).reshape(-1))
        dec = O.decode(dt, st).astype(np.float64)
        if kind == "walk":
            padded = np.zeros((rows, cols + 1), st.dtype)
            padded[:, :cols] = st.reshape(rows, cols)
            bufs.append(torch.from_numpy(padded.view(np.uint8).reshape(-1).copy()).cuda())
            ins.append((dt, cols + 1, 1))
            refs.append(dec.reshape(rows, cols))
        else:
            bufs.append(torch.from_numpy(st.view(np.uint8).reshape(-1).copy()).cuda())
            ins.append({"row": (dt, 1, 0), "col": (dt, 0, 1), "one": (dt, 0, 0)}[kind])
            refs.append(dec.reshape({"row": (rows, 1), "col": (1, cols), "one": (1, 1)}[kind]))
    want = T.elementwise(prog, refs, rows, cols)
    out = torch.full((rows * (cols + 1) * ES[out_dt],), 0xEE, dtype=torch.uint8, device="cuda") if in_place is None else bufs[in_place]
    before = out.cpu().numpy().view(O.NP_STORAGE[out_dt]).reshape(rows, cols + 1)[:, cols].copy()
    hip.elementwise(hip.make_elementwise_desc(prog, ins, out_dt, rows, cols, out_ld=cols + 1), [b.data_ptr() for b in bufs], out.data_ptr(),
                    torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    full = out.cpu().numpy().view(O.NP_STORAGE[out_dt]).reshape(rows, cols + 1)
    assert np.array_equal(full[:, cols], before), "written between the rows"
    got = O.decode(out_dt, np.ascontiguousarray(full[:, :cols])).astype(np.float64).reshape(rows, cols)
    err = np.abs(got - want) / np.maximum(np.abs(want), 1.0)  # the operands are of the order of 1: so are the fp32 roundings inside
    assert np.all(np.isfinite(want)) and err.max() <= TOL[out_dt], (prog, rows, cols, err.max())


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [O.F32, O.F16, O.BF16])
@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 7), (5, 64), (130, 513), (4, 20001)])
def test_every_operation_with_every_kind_of_right_operand(hip, dt, rows, cols):
    u = lambda n, t: O.uniform(n, 101, t, 0.5, 2.0)
    ops = [(dt, "walk", u(rows * cols, 0)), (O.F32, "row", u(rows, 1)), (dt, "row", u(rows, 2)), (dt, "col", u(cols, 3)), (O.F32, "col", u(cols, 4)), (dt, "walk", u(rows * cols, 5)),
           (dt, "one", u(1, 6)), (dt, "col", u(cols, 7))]
    x = ("input", 0)
    for op in BINARY:
        for right in ([("const", 1.25)], *[[("input", k)] for k in range(8)], [x, ("const", 0.5), "add"]):
            run(hip, [x] + right + [op], ops, dt, rows, cols)
    run(hip, [x, "neg", "exp2", "log2", ("input", 5), "max"], ops, dt, rows, cols, in_place=0)


@pytest.mark.gpu
def test_long_and_deep_programs_and_mixed_types(hip):
    rows, cols = 37, 300
    u = lambda n, t: O.uniform(n, 102, t, 0.5, 1.5)
    same = [(O.F16, "walk", u(rows * cols, 0)), (O.F16, "col", u(cols, 1)), (O.F16, "row", u(rows, 2)), (O.F16, "walk", u(rows * cols, 3)), (O.F16, "walk", u(rows * cols, 4))]
    mixed = [(O.F32, "walk", u(rows * cols, 0)), (O.F16, "col", u(cols, 1)), (O.BF16, "row", u(rows, 2)), (O.BF16, "walk", u(rows * cols, 3)), (O.F16, "walk", u(rows * cols, 4))]
    inputs = [("input", k) for k in range(5)]
    # six values, folded from the top down; the divisor is at least 0.5 + 0.5 * 0.5, so that no rounding is magnified by more than 3 (a first
    # form divided by a difference that came within 1e-5 of zero)
    deep = inputs + [("input", 0)] + ["mul", "add", "div", "sub", "max"]
    long_ = inputs[:4] + ["mul", "add", "sub"]                                               # then 40 more steps: 47 of 48
    long_ += [s for k in range(20) for s in (("input", k % 5), ("add", "mul", "max", "min")[k % 4])]
    unfused = [("input", 3)]                                                                # values saved, fetched, loaded and combined from below: two chunks
    for k in range(11):
        unfused += [("input", 4), "neg", "neg", "max" if k % 2 else "mul"]
    for ops in (same, mixed):
        for out in (O.F16, O.F32):
            for prog in (deep, long_, unfused):
                run(hip, prog, ops, out, rows, cols)


@pytest.mark.gpu
@pytest.mark.parametrize("dt,rows,cols", [(O.F16, 4099, 2056), (O.F32, 4099, 2056), (O.BF16, 70001, 72), (O.F16, 70001, 71)])
def test_lanes_that_walk_down_several_rows(hip, dt, rows, cols):
    """more rows than the grid covers at once: two slabs of columns, and 16 lanes a row whose last row block is incomplete; operands held
    ahead, fetched in place (more of a kind than there are slots) and mixed types"""
    u = lambda n, t: O.uniform(n, 103, t, 0.5, 1.5)
    other = O.F32 if dt != O.F32 else O.F16
    ops = [(dt, "walk", u(rows * cols, 0)), (dt, "row", u(rows, 1)), (other, "row", u(rows, 2)), (dt, "row", u(rows, 3)), (dt, "col", u(cols, 4)), (dt, "col", u(cols, 5)),
           (dt, "col", u(cols, 6)), (dt, "walk", u(rows * cols, 7))]
    prog = [("input", 0)]
    for k, op in zip((1, 4, 7, 2, 5, 3, 6), ("sub", "mul", "add", "max", "add", "min", "mul")):
        prog += [("input", k), op]
    run(hip, prog, ops, dt, rows, cols)
    run(hip, prog, ops, dt, rows, cols, in_place=0)
    run(hip, prog, [(other, "walk", u(rows * cols, 0))] + ops[1:], dt, rows, cols)


def on_device(hip, prog, dt, rows, cols, kinds, want, ld=None, in_place=False):
    """operands of `kinds` (walk, row, col, one) drawn on the device; `want` computes the reference from them in float64"""
    import torch
    t = {O.F32: torch.float32, O.F16: torch.float16, O.BF16: torch.bfloat16}[dt]
    ld = ld or cols
    g = torch.Generator(device="cuda").manual_seed(104)
    draw = lambda *shape: (torch.rand(*shape, device="cuda", generator=g) * 1.5 + 0.5).to(t)
    shape = {"walk": (rows, ld), "row": (rows, 1), "col": (1, cols), "one": (1, 1)}
    stride = {"walk": (dt, ld, 1), "row": (dt, 1, 0), "col": (dt, 0, 1), "one": (dt, 0, 0)}
    ops = [draw(*shape[k]) for k in kinds]
    ref = want(*[o.double()[:, :cols] for o in ops]).expand(rows, cols).clone()
    out = ops[0] if in_place else torch.full((rows, ld), 7.0, device="cuda", dtype=t)
    beyond = out[:, cols:].clone()
    hip.elementwise(hip.make_elementwise_desc(prog, [stride[k] for k in kinds], dt, rows, cols, out_ld=ld), [o.data_ptr() for o in ops], out.data_ptr(),
                    torch.cuda.current_stream().cuda_stream)
    err = ((out[:, :cols].double() - ref).abs() / ref.abs().clamp(min=1.0)).max().item()
    assert err <= TOL[dt] and torch.equal(out[:, cols:], beyond), (prog, rows, cols, err)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [O.F32, O.F16, O.BF16])
@pytest.mark.parametrize("rows,cols", [(8200, 520), (2051, 2059)])
def test_broadcast_operands_held_while_a_lane_walks_down(hip, dt, rows, cols):
    """every operation on an operand held for the rows a lane walks: one value per row, per column, and one in all (the smaller views above hold none)"""
    import torch
    does = {"add": torch.add, "sub": torch.sub, "mul": torch.mul, "div": torch.div, "max": torch.maximum, "min": torch.minimum}
    for op in BINARY:
        for kind in ("row", "col", "one"):
            on_device(hip, [("input", 0), ("input", 1), op], dt, rows, cols, ["walk", kind], does[op], ld=cols + 1)


@pytest.mark.gpu
@pytest.mark.parametrize("dt", [O.F32, O.F16, O.BF16])
@pytest.mark.parametrize("rows,cols", [(1, 4097 * 2048), (1, 4097 * 2048 - 8), (3073, 8192), (4096, 2048)], ids=["folded", "one_row", "three_groups_a_lane", "one_group_a_lane"])
def test_dense_views_of_several_groups_a_lane(hip, dt, rows, cols):
    """dense views just above and below the sizes at which 16-bit ones are folded and f32 ones change kernel; in place too"""
    gated = [("input", 0), ("input", 1), "mul", ("input", 2), "add"]
    on_device(hip, gated, dt, rows, cols, ["walk", "walk", "walk"], lambda x, y, z: x * y + z)
    on_device(hip, [("input", 0), ("input", 1), "add"], dt, rows, cols, ["walk", "walk"], lambda x, y: x + y, in_place=True)
    on_device(hip, [("input", 0), ("const", 1.0), "add", "log2"], dt, rows, cols, ["walk"], lambda x: (x + 1).log2(), in_place=True)


@pytest.mark.gpu
@pytest.mark.parametrize("dt,tdt", [(O.F32, "float32"), (O.F16, "float16"), (O.BF16, "bfloat16")])
@pytest.mark.parametrize("rows,cols", [(3, 40), (4100, 520), (6200, 259)])
def test_a_value_of_the_row_combined_with_a_constant(hip, dt, tdt, rows, cols):
    """either way round, once and for both slots, as a right operand, before everything else and with the operand mentioned again; zeros of either sign and infinities among the
    values.  One rounding to fp32 per operation, as torch's do: the same bits."""
    import torch
    tdt, g = getattr(torch, tdt), torch.Generator(device="cuda").manual_seed(9)
    x = torch.randn(rows, cols, device="cuda", generator=g).to(tdt)
    r, s = (torch.randn(rows, device="cuda", generator=g).to(tdt) for _ in range(2))
    col = (torch.rand(cols, device="cuda", generator=g) + 0.5).to(tdt)
    r[0], r[1], r[2] = 0.0, -0.0, float("inf")
    X, Rv, Sv, Cv = x.float(), r.float()[:, None], s.float()[:, None], col.float()
    does = {"add": torch.add, "sub": torch.sub, "mul": torch.mul}
    programs = []
    for name, f in does.items():
        for c in (0.75, -3.0):
            k = torch.tensor(c, device="cuda")
            programs += [([("input", 0), ("input", 1), ("const", c), name, "sub", ("input", 3), "mul"], (X - f(Rv, k)) * Cv),
                         ([("input", 0), ("const", c), ("input", 1), name, "max"], torch.maximum(X, f(k, Rv))),
                         ([("input", 1), ("const", c), name, ("input", 0), "add"], f(Rv, k) + X),
                         ([("input", 0), ("input", 1), ("const", c), name, "neg", "add"], X + (-f(Rv, k))),
                         ([("input", 0), ("input", 1), ("const", c), name, "add", ("const", 2.0), ("input", 2), name, "mul"], (X + f(Rv, k)) * f(torch.tensor(2.0, device="cuda"), Sv)),
                         ([("input", 0), ("input", 2), ("const", c), name, "add", ("input", 2), "mul"], (X + f(Sv, k)) * Sv),
                         ([("input", 0), ("input", 2), ("const", c), "div", "add"], X + Sv / k)]
    for program, want in programs:
        desc = hip.make_elementwise_desc(program, [(dt, cols, 1), (dt, 1, 0), (dt, 1, 0), (dt, 0, 1)], dt, rows, cols)
        out = torch.full_like(x, 7.0)
        hip.elementwise(desc, [t.data_ptr() for t in (x, r, s, col)], out.data_ptr(), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(out, want.to(tdt)), program


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [3, 1100, 5000])
def test_halves_of_a_lanes_columns_with_operands_of_other_types(hip, rows):
    """32-bit rows of 8 columns to more than a slab of 2048 beside f16 and bf16 operands of one value per column and per row, held and fetched in place; packed and one element
    apart, into another matrix and in place.  One rounding to fp32 per operation, as torch's do: the same bits."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(12)
    stream = torch.cuda.current_stream().cuda_stream
    for cols in (8, 9, 11, 12, 13, 31, 33, 35, 36, 64, 67, 259, 511, 512, 513, 1026) + ((2047, 2048, 2049, 2051, 2052, 4101) if rows < 5000 else ()):
        for ld in (cols, cols + 1):
            x = torch.randn(rows, ld, device="cuda", generator=g)
            c1, c2 = torch.randn(cols, device="cuda", generator=g).half(), torch.randn(cols, device="cuda", generator=g).bfloat16()
            r1, c3 = torch.randn(rows, device="cuda", generator=g).half(), torch.randn(cols, device="cuda", generator=g)
            X = x[:, :cols]
            for program, want in (
                    ([("input", 0), ("input", 1), "mul", ("input", 2), "add"], X * c1.float() + c2.float()),
                    ([("input", 0), ("input", 3), "sub", ("input", 1), "mul", ("input", 2), "add", ("input", 4), "max"], torch.maximum((X - r1.float()[:, None]) * c1.float() + c2.float(), c3)),
                    ([("input", 0), ("const", 2.5), "mul"], X * 2.5)):
                desc = hip.make_elementwise_desc(program, [(O.F32, ld, 1), (O.F16, 0, 1), (O.BF16, 0, 1), (O.F16, 1, 0), (O.F32, 0, 1)], O.F32, rows, cols, out_ld=ld)
                for out in (torch.full_like(x, 3.0), x.clone()):
                    beside = out[:, cols:].clone()
                    first = out if bool((out == x).all()) else x
                    hip.elementwise(desc, [t.data_ptr() for t in (first, c1, c2, r1, c3)], out.data_ptr(), stream)
                    torch.cuda.synchronize()
                    assert torch.equal(out[:, :cols], want) and torch.equal(out[:, cols:], beside), (rows, cols, ld, len(program))
