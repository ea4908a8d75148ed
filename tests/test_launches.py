"""What a call launches, recorded on the CPU: an executable whose own definitions of the HIP runtime's calls come before the runtime's prints them."""
import os
import re
import subprocess

import pytest

from frisk_amd import runtime as R

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.fixture(scope="module")
def recorded(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("launches") / "launch_recorder")
    rocm, lib = os.environ.get("ROCM_PATH", "/opt/rocm"), os.path.dirname(R.LIB_PATH)
    subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(rocm, "include"), "-I" + os.path.join(ROOT, "include"),
                    os.path.join(HERE, "launch_recorder.cpp"), "-o", exe, "-L" + lib, "-lfrisk_hip", "-L" + os.path.join(rocm, "lib"), "-lamdhip64",
                    "-Wl,-rpath," + lib, "-Wl,-rpath," + os.path.join(rocm, "lib")], check=True)

    def run(*args):
        """(status, [(kernel, grid x, grid y, lanes)]), or the lines of "kept" """
        out = subprocess.run([exe] + [str(a) for a in args], check=True, capture_output=True, text=True).stdout.split("\n")
        if args == ("kept",):
            return {l.split()[0]: float(l.split()[1]) for l in out if l}
        launches = [l.split()[1:] for l in out if l.startswith("launch ")]
        return int([l for l in out if l.startswith("status ")][0].split()[1]), [(n, int(x), int(y), int(lanes)) for n, x, y, _, lanes in launches]
    return run


@pytest.mark.parametrize("keep", ["keep", "nokeep"])
@pytest.mark.parametrize("dt,M,N,K,transA,transB", [(R.F16, 1999, 4099, 3001, 0, 0), (R.F16, 1589, 3072, 9600, 0, 0), (R.F16, 4, 576, 6784, 0, 0), (R.I8, 58, 2240, 7680, 0, 0)])
def test_a_call_without_workspace_uses_none_of_the_plan_that_needs_one(recorded, dt, M, N, K, transA, transB, keep):
    """copies, split edge tiles, slices of K: planned again without a workspace, nothing of the first plan is left, also where the thread has no storage for the
    plans it keeps"""
    need = R.workspace_bytes(R.make_desc(dt, M, N, K, transA=transA, transB=transB, dtype_out=R.I32 if dt == R.I8 else None))
    assert need > 0
    status, with_it = recorded("gemm", keep, dt, M, N, K, transA, transB, need)
    assert status == 0 and len(with_it) >= 2
    for too_small in (0, 16):
        status, launches = recorded("gemm", keep, dt, M, N, K, transA, transB, too_small)
        assert status == 0 and len(launches) == 1 and "gemm_kernel" in launches[0][0] and launches[0][2] == 1, launches


@pytest.mark.parametrize("slices,tile", [(7, "ELi256ELi256E"), (5, "ELi256ELi256E"), (4, None), (3, None), (0, None)])
def test_slices_of_a_deep_product_that_the_workspace_does_not_hold_fall_away(recorded, slices, tile):
    """35 tiles of 256x256 under 117 K tiles: five slices and more; below that line another tile takes the product"""
    status, launches = recorded("gemm", "keep", R.F16, 1777, 1216, 7488, 0, 0, slices * 35 * 256 * 256 * 4)
    assert status == 0 and ("ELi256ELi256E" in launches[0][0]) == bool(tile), launches
    assert not tile or (launches[0][1] == 35 * slices and "tail_reduce_kernel" in launches[1][0]), launches


@pytest.mark.parametrize("dt,M,N,K,transA,transB", [(R.E4M3, 2410, 865, 1222, 1, 0), (R.E4M3, 2511, 2241, 536, 1, 1), (R.BF16, 2321, 2172, 1978, 0, 1), (R.F16, 1524, 1901, 861, 0, 0),
                                                    (R.I8, 445, 2933, 150, 0, 0), (R.F16, 157, 23, 32, 1, 1)])
def test_rows_off_16_bytes_are_staged_through_registers_without_a_workspace(recorded, dt, M, N, K, transA, transB):
    """the 128x128 kernel whose flag for it (the first of two after the wave grid and the ring) is set"""
    status, launches = recorded("gemm", "keep", dt, M, N, K, transA, transB, 0)
    (name, *_), = launches
    assert status == 0 and "gemm_kernel" in name and "ELi128ELi128E" in name and "ELi2ELi2ELi2ELb1ELb0E" in name, name


def test_kept_plans_tell_leading_dimensions_types_and_alignments_apart(recorded):
    """one shape in turn on two of them finds both plans kept: nearer to the time of a repeated call (0.06 us) than to that of a new one (2 us)"""
    ns = recorded("kept")
    for what in ("lda", "ldb", "ldc", "dtype_out", "alignment"):
        assert ns[what] < (ns["again"] * ns["new"]) ** 0.5, ns


@pytest.mark.parametrize("dt", [R.F16, R.BF16, R.F32])
@pytest.mark.parametrize("cols", [2048, 4097, 5000, 11008, 20000, 16384])
def test_block_bodies_with_held_operands_are_one_round_of_work_groups(recorded, dt, cols):
    """as many work-groups as the chip holds at once, 4 a CU, also where a row's slabs of 2048 columns do not divide their number: a few more would run alone"""
    for operands in ("mc", "mr", "mrc", "mcc"):
        status, launches = recorded("block", dt, 6000 // -(-cols // 2048), cols, operands)
        (_, x, y, lanes), = launches
        assert status == 0 and lanes == 256 and x == -(-cols // 2048) and 1024 - x < x * y <= 1024, (operands, x, y)


@pytest.mark.parametrize("dt,rows,cols,operands,groups", [
    (R.F16, 7, 300000, "mc", 1029), (R.BF16, 640, 4096, "mrcc", 1280), (R.F16, 641, 4096, "mrcc", 1024), (R.F32, 640, 4096, "mmc", 1280),    # five work-groups a CU in one round
    (R.F16, 768, 4096, "mr", 1536), (R.F16, 769, 4096, "mr", 1024), (R.F32, 513, 4096, "mr", 1024), (R.F32, 1024, 4096, "mc", 2048),          # one broadcast operand
    (R.F16, 131072, 24, "mc", 2048), (R.F16, 100000, 24, "mcm", 1024),
    (R.F16, 7168, 8192, "mcm", 1024), (R.F16, 7169, 8192, "mcm", 4096), (R.F16, 7169, 8192, "mcc", 1024)])                                    # a second operand that walks long rows
def test_grids_of_block_bodies_with_few_or_many_groups_a_lane(recorded, dt, rows, cols, operands, groups):
    """one group a lane where the kernels that hold no broadcast operand take all of them at once; 16 work-groups a CU again from 28 groups a lane beside a second walking operand"""
    status, launches = recorded("block", dt, rows, cols, operands)
    (_, x, y, _), = launches
    assert status == 0 and groups - x < x * y <= groups, (x, y)


@pytest.mark.parametrize("rows,cols,operands,groups", [
    (2048, 4096, "mm", 1024), (3000, 4096, "mm", 4096), (4096, 4096, "mm", 4096), (4096, 4096, "mcm", 4096), (20000, 300, "mcm", 1024),  # a second operand that walks the rows
    (1500, 7000, "mr", 1024), (4096, 4096, "mr", 4096), (4096, 4096, "mrcc", 1024), (6200, 4096, "mrcc", 4096),                        # held operands alone
    (100000, 24, "mr", 1563), (200000, 24, "mrc", 3125), (800000, 24, "mrc", 4096), (200000, 24, "mrcc", 1024), (120000, 24, "mrcc", 1875), (350000, 24, "mcm", 4096)])  # rows shorter than a wave
def test_grids_of_f32_block_bodies(recorded, rows, cols, operands, groups):
    """4 work-groups a CU up to 5, 7 or 12 groups a lane, 16 beyond; in rows shorter than a wave 16 where nothing is held"""
    status, launches = recorded("block", R.F32, rows, cols, operands)
    (_, x, y, _), = launches
    assert status == 0 and groups - x < x * y <= groups, (x, y)


@pytest.mark.parametrize("dt", [R.F16, R.BF16, R.F32])
@pytest.mark.parametrize("rows,cols", [(4000, 5000), (1000000, 24), (4000000, 7)])
def test_only_bodies_with_a_constant_on_a_rows_value_run_on_the_kernels_that_apply_one(recorded, dt, rows, cols):
    """as an argument of all kernels that hold operands, the constant made the bodies without one 1 to 2 % slower"""
    held = {}
    for operands in ("mrcc", "mcc", "mrrc", "mscc", "mcs", "mrsc", "mssc"):
        status, launches = recorded("block", dt, rows, cols, operands)
        (name, *_), = launches
        held[operands] = re.search(r"elementwise_kernelILi(\d)ELi(\d)E", name).groups()
        assert status == 0 and held[operands][0] == str(dt), name
    assert {held[o] for o in held if "s" not in o} == {(str(dt), "2")} and {held[o] for o in held if "s" in o} == {(str(dt), "3")}, held


@pytest.mark.parametrize("dt,rows,cols,ld,off,one", [
    (R.F16, 1152, 1495, 1495, 0, True), (R.F16, 1153, 1495, 1495, 0, False), (R.F16, 1435, 1495, 1536, 0, True), (R.F16, 1435, 1495, 1536, 16, False),  # rows anywhere, on 128-byte lines, off by a chunk
    (R.F16, 1536, 128, 131, 0, True), (R.F16, 1536, 129, 131, 0, False), (R.F32, 1452, 460, 460, 0, False), (R.F32, 1452, 480, 480, 0, True),            # 256 bytes of a row and more
    (R.BF16, 1537, 1536, 1536, 0, False), (R.BF16, 1000, 16384, 16385, 0, True), (R.BF16, 1000, 16385, 16385, 0, False)])
def test_column_reductions_in_one_launch_or_in_slices(recorded, dt, rows, cols, ld, off, one):
    """work-groups of 1024 lanes up to 1152 rows, on 128-byte lines or of 256 bytes at most up to 1536, else slices and their sums; without a workspace always one launch"""
    status, launches = recorded("reduce", dt, rows, cols, ld, 0, off, 1)
    assert status == 0 and [lanes for _, _, _, lanes in launches] == ([1024] if one else [256, 256]), launches
    status, launches = recorded("reduce", dt, rows, cols, ld, 0, off, 0)
    assert status == 0 and [lanes for _, _, _, lanes in launches] == [1024 if rows <= 1536 and cols < 16385 else 256], launches


@pytest.mark.parametrize("dt,rows,cols,ld,off,kernel", [
    # <groups a lane, rows of whole groups 0 / a part 1 / less than a group 2>
    (R.F16, 20000, 1000, 1000, 0, "short 2 0"), (R.F16, 20000, 1003, 1003, 0, "short 2 1"), (R.BF16, 5878, 864, 865, 2, "short 2 0"), (R.F32, 7313, 464, 464, 0, "short 2 0"), (R.F16, 100000, 24, 24, 0, "short 1 0"),
    (R.F16, 100000, 27, 27, 0, "short 1 1"), (R.F16, 100000, 7, 8, 0, "short 1 2"), (R.F32, 300000, 3, 3, 0, "short 1 2"), (R.F32, 5000, 1023, 1024, 0, "short 4 1"), (R.F32, 5000, 1024, 1024, 0, "short 4 0"),
    # <lanes, through the caches 0 / past them 1 / past them from a row's first boundary on 2>
    (R.F16, 4096, 8192, 8192, 0, "rows 256 0"), (R.F32, 3000, 4096, 4096, 0, "rows 256 0"), (R.F16, 8192, 8192, 8192, 0, "rows 256 1"), (R.F16, 8200, 4095, 4096, 0, "rows 256 1"), (R.F16, 3000, 4095, 4095, 0, "rows 256 0"),
    (R.F16, 10069, 4946, 4946, 0, "rows 256 2"), (R.F16, 8192, 8192, 8192, 2, "rows 256 2"), (R.F16, 2177, 8944, 8944, 0, "rows 256 0"), (R.BF16, 1024, 9000, 9000, 0, "rows 512 0"),
    (R.BF16, 1025, 9000, 9000, 0, "rows 256 0"), (R.F32, 4000, 6144, 6144, 0, "rows 256 1"), (R.F32, 4000, 6148, 6148, 0, "rows 512 1"), (R.F16, 4426, 15161, 15161, 0, "rows 512 2"), (R.F32, 394, 9229, 9229, 0, "rows 512 0")])
def test_row_reductions_by_what_their_rows_are(recorded, dt, rows, cols, ld, off, kernel):
    """rows of whole groups on kernels that know of no others; past the caches beyond 64 MiB; 512 lanes where they have work"""
    status, launches = recorded("reduce", dt, rows, cols, ld, 1, off, 1)
    (name, *_), = launches
    which, a, b = kernel.split()
    got = re.search(r"reduce_short_rows_kernelILi%dELi0ELi(\d+)ELi(\d+)E" % dt if which == "short" else r"reduce_rows_kernelILi%dELi0ELi(\d+)ELi(\d+)E" % dt, name)
    assert status == 0 and got and got.groups() == (a, b), name


@pytest.mark.parametrize("dt,rows,cols,ld,off,kernel", [
    # <groups a lane, rows of whole groups 0 / a part 1 / less than a group 2>
    (R.F16, 32768, 512, 512, 0, "short 1 0"), (R.F16, 100000, 27, 27, 0, "short 1 1"), (R.F16, 100000, 7, 8, 0, "short 1 2"), (R.F32, 300000, 3, 3, 0, "short 1 2"), (R.F16, 8192, 1024, 1025, 2, "short 2 0"),
    (R.BF16, 14242, 790, 790, 0, "short 2 1"), (R.F32, 8192, 1024, 1024, 0, "short 4 0"), (R.F32, 8192, 1023, 1024, 0, "short 4 1"),
    # <groups a lane, lanes, whole groups past the caches 0 / through them 1 / any through them 2 / any past them from a row's first boundary on 3>
    (R.F16, 4096, 4096, 4096, 0, "held 2 256 0"), (R.F32, 3000, 4096, 4096, 0, "held 2 512 0"), (R.F16, 3584, 8192, 8192, 0, "held 2 512 0"), (R.F16, 3585, 8192, 8192, 0, "held 2 512 1"), (R.F16, 7168, 8192, 8192, 0, "held 2 512 1"), (R.F16, 7169, 8192, 8192, 0, "held 2 512 0"), (R.F16, 8192, 8192, 8200, 0, "held 2 512 0"),
    (R.F16, 4096, 4000, 4000, 0, "held 2 256 1"), (R.F16, 4096, 4096, 4096, 16, "held 2 256 1"), (R.F16, 4096, 4096, 4096, 2, "held 2 256 2"), (R.F16, 4096, 4095, 4096, 0, "held 2 256 2"), (R.F16, 8192, 8192, 8193, 0, "held 3 512 3"),
    (R.F16, 870, 16370, 16370, 0, "held 4 512 2"), (R.F16, 4426, 15161, 15161, 0, "held 4 512 3"), (R.F16, 64, 32768, 32768, 0, "held 9 512 0")])
def test_softmax_by_what_its_rows_are(recorded, dt, rows, cols, ld, off, kernel):
    """rows of whole groups on kernels that know of no others; past the caches where that was the faster way"""
    status, launches = recorded("softmax", dt, rows, cols, ld, off)
    (name, *_), = launches
    which, *want = kernel.split()
    got = re.search(r"softmax_%s_rows_kernelILi%d" % (which, dt) + r"ELi(\d+)" * len(want) + "E", name)
    assert status == 0 and got and list(got.groups()) == want, name
