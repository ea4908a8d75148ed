"""Host-only: whatever the planner picks must be a kernel that may run on the problem.  A fast kernel moves whole tiles with
16-byte transfers, an edge kernel clamps M and N but not K, the chunk-wise guarded kernel needs whole 16-byte chunks along K, and
a split needs whole K tiles per slice: a plan that breaks one of these would send a kernel beyond its operands."""
import random
import re

import pytest

from frisk_amd import runtime as R

ES = {R.F32: 4, R.F16: 2, R.BF16: 2, R.I8: 1, R.E4M3: 1}
OUT = {R.F32: R.F32, R.F16: R.F16, R.BF16: R.BF16, R.I8: R.I32, R.E4M3: R.BF16}
OS = {R.F32: 4, R.F16: 2, R.BF16: 2, R.I32: 4}
NAME = re.compile(r"(\w+?)_(n|t)(n|t)_(\d+)x(\d+)x(\d+)_w(\d+)x(\d+)(?:x(\d+))?_s(\d+)(?:x(\d+))?(_a16)?(_guard_chunks|_guard)?(_splitk)?(_edge)?")


def shapes(rng, n):
    for _ in range(n):
        kind = rng.choice(["whole", "edge", "ragged_k", "any", "skinny", "big"])
        if kind == "whole":
            yield rng.choice([32, 64, 128, 256, 512, 1024, 4096]), rng.choice([32, 128, 256, 1024, 4096, 8192]), rng.choice([128, 512, 1024, 4096, 8192])
        elif kind == "edge":
            yield rng.randint(1, 5000), 16 * rng.randint(1, 700), 128 * rng.randint(1, 64)
        elif kind == "ragged_k":
            yield rng.randint(1, 3000), 16 * rng.randint(1, 300), 16 * rng.randint(1, 500)
        elif kind == "skinny":
            yield rng.randint(1, 300), 128 * rng.randint(1, 128), 128 * rng.randint(8, 128)
        elif kind == "big":
            yield 256 * rng.randint(8, 40), 256 * rng.randint(8, 40), 128 * rng.randint(8, 64)
        else:
            yield rng.randint(1, 2000), rng.randint(1, 2000), rng.randint(1, 2000)


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_every_plan_is_a_kernel_that_may_run_on_the_problem(seed):
    rng = random.Random(seed)
    names = R.kernel_names()
    seen = set()
    for M, N, K in shapes(rng, 1500):
        dt = rng.choice([R.F32, R.F16, R.BF16, R.I8, R.E4M3])
        tA, tB = rng.random() < 0.3, rng.random() < 0.5
        split = rng.choice([0, 0, 0, 1, 2, 4])
        d = R.make_desc(dt, M, N, K, dtype_out=OUT[dt], transA=tA, transB=tB, split_k=split)
        try:
            p = R.plan(d)
        except R.FriskHipError as ex:
            assert ex.status in (R.ERR_TILE, R.ERR_SHAPE), (M, N, K, str(ex))
            continue
        name = names[p.kernel_id]
        m = NAME.fullmatch(name)
        assert m, name
        bm, bn, bk = int(m.group(4)), int(m.group(5)), int(m.group(6))
        guard, splitk, edge = m.group(13), bool(m.group(14)), bool(m.group(15))
        es, osz = ES[dt], OS[OUT[dt]]
        what = (name, M, N, K, tA, tB, split)
        seen.add((guard or "") + ("_splitk" if splitk else "") + ("_edge" if edge else ""))
        assert (m.group(2) == "t") == tA and (m.group(3) == "t") == tB and (bm, bn, bk) == (p.tile_m, p.tile_n, p.tile_k), what
        assert p.grid_x == -(-N // bn) and p.grid_y == -(-M // bm), what
        rows_aligned = (d.lda * es) % 16 == 0 and (d.ldb * es) % 16 == 0 and (d.ldc * osz) % 16 == 0
        if guard is None:
            assert rows_aligned and K % bk == 0, what
            if edge:
                assert M % bm or N % bn, what
            else:
                assert M % bm == 0 and N % bn == 0, what
        elif guard == "_guard_chunks":
            assert rows_aligned and K % (16 // es) == 0, what
        assert bool(p.guarded) == (guard is not None), what
        if p.split_k > 1:
            # slices of equal length but the last, which holds at least one K tile; those of a split that the descriptor names divide the K tiles
            per = -(-(K // bk) // p.split_k)
            assert splitk and K % bk == 0 and (p.split_k - 1) * per < K // bk and p.workspace_bytes == p.split_k * M * N * 4, what
            assert split in (0, p.split_k) and (split == 0 or (K // bk) % split == 0), what
        else:
            assert p.split_k == 1, what
        if p.tail_split > 1:
            assert splitk and not edge and p.tail_tiles == (p.grid_x * p.grid_y) % 256 and (K // bk) % p.tail_split == 0, what
            assert p.workspace_bytes == p.tail_split * p.tail_tiles * bm * bn * 4, what
        if splitk and p.workspace_bytes:
            assert p.split_k > 1 or p.tail_split > 1, what
        if split == 1:
            assert p.split_k == 1 and p.tail_split == 1 and p.workspace_bytes == 0, what
    # the walk reached every kind of kernel
    assert {"", "_edge", "_splitk", "_splitk_edge", "_guard", "_guard_chunks"} <= seen, seen


def test_kept_plans_are_those_of_their_descriptor():
    """workspace_bytes looks its plan up among those that the thread keeps, plan() works it out anew: the same for more descriptors than are kept, met
    in any order and from several threads"""
    import random
    import threading
    rng = random.Random(17)
    dts = [rng.choice([R.F16, R.BF16, R.I8, R.E4M3, R.F32]) for _ in range(300)]
    descs = [R.make_desc(dt, rng.randrange(1, 700), rng.randrange(1, 700) * rng.choice([1, 8]), rng.randrange(1, 9000),
                         dtype_out=OUT[dt], transA=rng.random() < 0.5, transB=rng.random() < 0.5, clear_accum=rng.random() < 0.5) for dt in dts]
    want = [R.plan(d).workspace_bytes for d in descs]
    assert len(set(want)) > 50

    def walk(seed, wrong):
        order = random.Random(seed).choices(range(len(descs)), k=2000)
        wrong.extend(i for i in order if R.workspace_bytes(descs[i]) != want[i])

    wrong = []
    threads = [threading.Thread(target=walk, args=(s, wrong)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    walk(9, wrong)
    assert not wrong


def test_slices_of_unequal_length_leave_the_last_one_its_k_tiles():
    """a split in slices of unequal length: the plan says how many, every slice holds K tiles, the last one at least as many as the kernel's loop is
    written for (16x16x128 atoms: four); a split that the caller names still has to divide them"""
    uneven = 0
    for dt in (R.F16, R.I8, R.E4M3):
        for tb in (0, 1):
            for M, N in ((4, 576), (58, 2240), (200, 896), (512, 512), (2048, 2048), (2304, 1280)):
                for K in range(2048, 9000, 128):
                    d = R.make_desc(dt, M, N, K, transB=tb, dtype_out={R.F16: R.F16, R.I8: R.F16, R.E4M3: R.BF16}[dt],
                                    epilogue={R.F16: R.EPI_NONE, R.I8: R.EPI_ROW_COL_SCALE, R.E4M3: R.EPI_TENSOR_SCALE}[dt])
                    p = R.plan(d)
                    kt, slices = K // p.tile_k, p.split_k
                    if kt % slices == 0:
                        continue
                    per = -(-kt // slices)
                    last = kt - (slices - 1) * per
                    assert K % p.tile_k == 0 and p.workspace_bytes == slices * M * N * 4 and slices > 1 and p.tail_split == 1, (dt, M, N, K)
                    assert (4 if dt == R.E4M3 and p.mfma_m == 16 else 1) <= last < per, (dt, M, N, K, slices)
                    assert R.plan(R.make_desc(dt, M, N, K, transB=tb, dtype_out=d.dtype_out, epilogue=d.epilogue, split_k=1)).workspace_bytes == 0
                    uneven += 1
    assert uneven > 50
    with pytest.raises(R.FriskHipError):
        R.plan(R.make_desc(R.F16, 256, 256, 64 * 7, split_k=2))
