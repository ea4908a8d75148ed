"""The 16-row MFMA atoms are written as inline assembly (gemm_kernel.hip.inc: Mma<*, 16>), so the compiler places none of the
wait states an MFMA needs around them.  This test compiles a few of those kernels to gfx950 ISA (no GPU needed) and
checks the two patterns that would be wrong: a vector instruction writing a register that an MFMA reads within the next
few instructions (accumulator initialisation right before the first MFMA), and a vector instruction reading an MFMA
result too soon after it (before the drain the kernel issues ahead of the epilogue)."""
import concurrent.futures
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "frisk_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

KERNELS = [
    "template __global__ void gemm_kernel<GemmCfg<FRISK_F16, 0, 1, 256, 256, 64, 2, 2, 2, false, false, 1, 3, 16>>(GemmParams);",
    "template __global__ void gemm_kernel<GemmCfg<FRISK_F16, 0, 0, 256, 256, 64, 2, 2, 2, false, true, 1, 3, 16>>(GemmParams);",
    "template __global__ void gemm_kernel<GemmCfg<FRISK_BF16, 1, 1, 256, 256, 64, 2, 2, 2, false, false, 1, 3, 16>>(GemmParams);",
    "template __global__ void gemm_kernel<GemmCfg<FRISK_I8, 1, 0, 256, 256, 128, 2, 2, 2, false, false, 1, 3, 16>>(GemmParams);",
    "template __global__ void gemm_kernel<GemmCfg<FRISK_E4M3, 0, 1, 256, 256, 128, 2, 2, 2, false, false, 1, 3, 16>>(GemmParams);",
    "template __global__ void gemm_kernel<GemmCfg<FRISK_F16, 0, 0, 160, 256, 64, 2, 2, 2, false, false, 1, 3, 16, true>>(GemmParams);",
    "template __global__ void gemm_kernel<GemmCfg<FRISK_BF16, 0, 1, 192, 256, 64, 2, 2, 2, false, false, 1, 3, 16, true>>(GemmParams);",
    "template __global__ void gemm_kernel<GemmCfg<FRISK_BF16, 0, 0, 224, 256, 64, 2, 2, 2, false, false, 1, 3, 16, true>>(GemmParams);",
    "template __global__ void gemm_kernel<GemmCfg<FRISK_I8, 0, 1, 160, 256, 128, 2, 2, 2, false, false, 1, 3, 16, true>>(GemmParams);",
    "template __global__ void gemm_kernel<GemmCfg<FRISK_I8, 0, 0, 224, 256, 128, 2, 2, 2, false, false, 1, 3, 16, true>>(GemmParams);",
]


def _registers(text):
    out = set()
    for kind, lo, hi in re.findall(r"\b([av])\[(\d+):(\d+)\]", text):
        out.update(kind + str(r) for r in range(int(lo), int(hi) + 1))
    out.update(kind + n for kind, n in re.findall(r"\b([av])(\d+)\b", text))
    return out


def _operands(line):
    parts = line.split(None, 1)
    return parts[1].split(",") if len(parts) > 1 else []


def hazards(listing, window_before=8, window_after=12):
    found = []
    for kernel in re.split(r"\n\t\.globl\t", listing)[1:]:
        name = kernel.split("\n")[0]
        lines = [l.strip() for l in kernel.split("\n") if l.startswith("\t") and not l.strip().startswith((".", ";"))]
        for i, line in enumerate(lines):
            if not line.startswith("v_mfma"):
                continue
            ops = _operands(line)
            reads, result = _registers(",".join(ops)), _registers(ops[0])
            multiplicands = _registers(",".join(ops[1:3])) - result
            for back in range(1, window_before + 1):
                prev = lines[i - back] if i - back >= 0 else ""
                if prev.startswith("v_") and not prev.startswith("v_mfma"):
                    written = _registers((_operands(prev) or [""])[0]) & reads
                    # a multiplicand written by an ordinary vector instruction is interlocked by the hardware (only the accumulator
                    # operand needs wait states); keep two instructions of distance anyway
                    if written - multiplicands or (written and back <= 2):
                        found.append((name, prev, line))
            for fwd in range(1, window_after + 1):
                nxt = lines[i + fwd] if i + fwd < len(lines) else ""
                if nxt.startswith("v_") and not nxt.startswith("v_mfma") and _registers(",".join(_operands(nxt)[1:])) & result:
                    found.append((name, line, nxt))
    return found


def foreign_m0_uses(listing, reach=6):
    """lines that name M0 outside the transfers the kernels write themselves: s_add_u32 m0 followed, within a few
    instructions that do not name M0 (an MFMA and scalar address arithmetic may sit between the two halves of a transfer), by
    its global_load_lds_dwordx4.  The transfer writes M0 without telling the compiler, which is only sound while the
    compiler has no use of M0 of its own in the kernel."""
    lines = [l.strip() for l in listing.split("\n") if l.startswith("\t") and not l.strip().startswith((".", ";"))]
    found = []
    for i, line in enumerate(lines):
        if not re.search(r"\bm0\b", line):
            continue
        own = False
        if line.startswith("s_add_u32 m0, "):
            for nxt in lines[i + 1:i + 1 + reach]:
                if nxt.startswith("global_load_lds_dwordx4"):
                    own = True
                    break
                if re.search(r"\bm0\b", nxt):
                    break
        if not own:
            found.append(line)
    return found


def test_scanner_sees_both_patterns():
    listing = "\n\t.globl\tk\nk:\n\tv_accvgpr_mov_b32 a5, a1\n\ts_nop 0\n\tv_mfma_f32_16x16x32_f16 a[4:7], v[0:3], v[4:7], a[4:7]\n\tv_accvgpr_read_b32 v9, a6\n"
    got = hazards(listing)
    assert len(got) == 2 and got[0][1].startswith("v_accvgpr_mov") and got[1][2].startswith("v_accvgpr_read")
    assert foreign_m0_uses("\ts_add_u32 m0, s4, 0x400\n\ts_nop 0\n\tglobal_load_lds_dwordx4 v1, s[2:3]\n\ts_mov_b32 m0, s7\n\tds_read_b32 v1, v2\n") == ["s_mov_b32 m0, s7"]
    split = "\ts_add_u32 m0, s4, 0x400\n\tv_mfma_f32_16x16x32_f16 a[4:7], v[0:3], v[4:7], a[4:7]\n\ts_add_u32 s8, s8, s0\n\tglobal_load_lds_dwordx4 v1, s[8:9]\n"
    assert foreign_m0_uses(split) == [] and foreign_m0_uses(split.replace("s_add_u32 s8, s8, s0", "s_add_u32 m0, s4, 0x800")) == ["s_add_u32 m0, s4, 0x400"]
    clean = "\n\t.globl\tk\nk:\n\tv_mfma_f32_16x16x32_f16 a[4:7], v[0:3], v[4:7], a[4:7]\n\tv_mfma_f32_16x16x32_f16 a[8:11], v[0:3], v[4:7], a[8:11]\n"
    assert hazards(clean) == []


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which("hipcc")), reason="needs hipcc to produce the ISA listing")
def test_inline_assembly_mfma_kernels_keep_their_wait_states(tmp_path):
    def compiled(i, kernel):  # (a unit each, side by side: one kernel takes half a minute)
        src, out = tmp_path / ("atoms16_%d.hip" % i), tmp_path / ("atoms16_%d.s" % i)
        src.write_text('#include "gemm_kernel.hip.inc"\nnamespace frisk {\n%s\n}\n' % kernel)
        cmd = [HIPCC if os.path.exists(HIPCC) else "hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
               "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-Wno-unused-command-line-argument", "--cuda-device-only", "-S", str(src), "-o", str(out)]
        r = subprocess.run(cmd, capture_output=True, text=True)
        assert r.returncode == 0, r.stderr[-2000:]
        return out.read_text()

    with concurrent.futures.ThreadPoolExecutor(min(8, os.cpu_count() or 1)) as pool:
        listing = "\n".join(pool.map(compiled, range(len(KERNELS)), KERNELS))
    assert listing.count("v_mfma_f32_16x16x32_f16") > 300 and "v_mfma_i32_16x16x64_i8" in listing and "v_mfma_f32_16x16x32_bf16" in listing
    assert listing.count("v_mfma_f32_16x16x128_f8f6f4") >= 64 * 7 and "scratch_" not in listing  # seven tile bodies, no spills
    bad = hazards(listing)
    assert not bad, "\n".join("%s: %s  ->  %s" % (n[:60], a, b) for n, a, b in bad[:10])
    assert listing.count("global_load_lds_dwordx4") > 100 and foreign_m0_uses(listing) == []


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which("hipcc")), reason="needs hipcc to produce the ISA listing")
def test_attention_kernel_has_no_use_of_m0_besides_its_transfers(tmp_path):
    """the attention kernel stages K and V with the same transfers (csrc/attention.hip: SK / SV issue_one): M0 is written by inline
    assembly without a clobber, so the compiler must have no use of M0 of its own in that kernel either"""
    out = tmp_path / "attention.s"
    cmd = [HIPCC if os.path.exists(HIPCC) else "hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-Wno-unused-command-line-argument", "--cuda-device-only", "-S", os.path.join(CSRC, "attention.hip"), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    listing = out.read_text()
    assert listing.count("global_load_lds_dwordx4") >= 4 * 16 and listing.count("v_mfma_f32_32x32x16") >= 4 * 32  # four kernels (f16 / bf16, two K layouts)
    assert foreign_m0_uses(listing) == [] and "scratch_" not in listing


def test_the_interpreter_of_block_bodies_declares_every_scalar_register_it_writes():
    """csrc/elementwise.hip runs its steps in inline assembly: what its scalar instructions write must be an output or a clobber, else the
    compiler may keep a value there (M0, a reserved register, cannot be declared: the listing is checked below)"""
    source = open(os.path.join(CSRC, "elementwise.hip")).read()
    text = source[source.index("#define EW_EACH"):source.index("#define EW_CLOBBERS")].replace("\\n", "\n")
    written = set("s%s" % r for r in re.findall(r"\bv_readlane_b32 s(\d+)", text))
    for lo, hi in re.findall(r"\bs_getpc_b64 s\[(\d+):(\d+)\]", text):
        written.update("s%d" % r for r in range(int(lo), int(hi) + 1))
    written.update(re.findall(r"\bs_(?:add|addc|addk|lshr|lshl|mov|and|or|sub|subb)\w* (s\d+)", text))
    assert {"s48", "s49", "s50", "s51", "s52", "s54", "s55", "s56"} <= written
    clobbers = set(re.findall(r'"(\w+)"', re.search(r"#define EW_CLOBBERS (.*)", source).group(1)))
    outputs = set(re.findall(r'"[=+]\{(s\d+)\}"', source))
    assert written <= clobbers | outputs, written - clobbers - outputs


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which("hipcc")), reason="needs hipcc to produce the ISA listing")
def test_kernels_of_block_bodies_have_no_use_of_m0_besides_the_index_mode(tmp_path):
    out = tmp_path / "elementwise.s"
    cmd = [HIPCC if os.path.exists(HIPCC) else "hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-Wno-unused-command-line-argument", "--cuda-device-only", "-S", os.path.join(CSRC, "elementwise.hip"), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    listing = out.read_text()
    assert listing.count("s_set_gpr_idx_on") > 28 * 10 and foreign_m0_uses(listing) == [] and "scratch_" not in listing
    # instructions that read M0 without naming it
    assert not re.search(r"^\s+(s_movrel|v_movrel|s_sendmsg|ds_gws|ds_append|ds_consume|buffer_load\w* .* lds|global_load_lds)", listing, re.M)


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which("hipcc")), reason="needs hipcc to produce the ISA listing")
def test_what_stands_in_front_of_a_16_bit_body(tmp_path):
    """the 16-bit kernels that hold all operands place their columns in 32 bits: 1780 instructions in all, 1801 with the 64 that the halves of 32-bit rows ask for"""
    out = tmp_path / "elementwise.s"
    cmd = [HIPCC if os.path.exists(HIPCC) else "hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-Wno-unused-command-line-argument", "--cuda-device-only", "-S", os.path.join(CSRC, "elementwise.hip"), "-o", str(out)]
    assert subprocess.run(cmd, capture_output=True).returncode == 0
    body = re.search(r"^_ZN5frisk\S*elementwise_kernelILi1ELi2ELi1ELi1E\S*:.*?\n(.*?)s_endpgm", out.read_text(), re.S | re.M).group(1)
    assert 1000 < len(re.findall(r"^\s+(?:[sv]|global|flat|ds|scratch)_", body, re.M)) <= 1790


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which("hipcc")), reason="needs hipcc to produce the ISA listing")
def test_stores_under_a_condition_do_not_wait_for_everything_under_way(tmp_path):
    """The tiles that C ends in accumulate with counted waits: loads and the knowledge that there are any stand under no condition of their own, else the compiler puts a wait for all that is under way, stores
    included, in front of every store (312 such waits in this kernel, 170 so; 19 us of 77 in a weight gradient of one round)"""
    src, out = tmp_path / "edge.hip", tmp_path / "edge.s"
    src.write_text('#include "gemm_kernel.hip.inc"\nnamespace frisk {\n'
                   "template __global__ void gemm_kernel<GemmCfg<FRISK_BF16, 1, 0, 256, 256, 64, 2, 2, 2, false, false, 1, 3, 16, true>>(GemmParams);\n}\n")
    cmd = [HIPCC if os.path.exists(HIPCC) else "hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-Wno-unused-command-line-argument", "--cuda-device-only", "-S", str(src), "-o", str(out)]
    assert subprocess.run(cmd, capture_output=True).returncode == 0
    listing = out.read_text()
    assert "scratch_" not in listing and listing.count("global_store_dwordx4") > 400 and len(re.findall(r"vmcnt\(0\)", listing)) < 200


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which("hipcc")), reason="needs hipcc to produce the ISA listing")
def test_the_smallest_fp32_products_have_one_body(tmp_path):
    """the fp32 edge tiles whose waves split K: 2184 instructions, 2508 with bodies of their own for whole tiles, those that C ends in and a few columns"""
    src, out = tmp_path / "edge.hip", tmp_path / "edge.s"
    src.write_text('#include "gemm_kernel.hip.inc"\nnamespace frisk {\n'
                   "template __global__ void gemm_kernel<GemmCfg<FRISK_F32, 0, 0, 32, 32, 128, 1, 1, 2, false, false, 4, 2, 32, true>>(GemmParams);\n}\n")
    cmd = [HIPCC if os.path.exists(HIPCC) else "hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
           "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-Wno-unused-command-line-argument", "--cuda-device-only", "-S", str(src), "-o", str(out)]
    assert subprocess.run(cmd, capture_output=True).returncode == 0
    listing = out.read_text()
    assert "scratch_" not in listing and 1500 < len(re.findall(r"^\s+(?:[sv]|global|flat|ds|buffer)_", listing, re.M)) <= 2300
