"""`python -m frisk_amd.build --if-missing` on trees that hold some of what the package loads"""
import os
import shutil
import subprocess
import sys
import sysconfig

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SUFFIX = sysconfig.get_config_var("EXT_SUFFIX")
LIBRARY = "frisk_amd/lib/libfrisk_hip.so"


@pytest.mark.parametrize("missing", [(), ("frisk_amd/frisk_launch" + SUFFIX,), ("frisk_amd/frisk_launch" + SUFFIX, "frisk_amd/frisk/frisk_ffi" + SUFFIX)])
def test_what_is_missing_is_built_and_nothing_else(tmp_path, missing):
    """a tree from before an extension was added, or built under another Python: the library is there and the extension for this interpreter is not"""
    for part in ("frisk_amd", "include"):
        shutil.copytree(os.path.join(ROOT, part), tmp_path / part, ignore=shutil.ignore_patterns("build", "__pycache__"))
    for path in missing:
        (tmp_path / path).unlink()
    present = {p: p.stat().st_mtime_ns for p in tmp_path.rglob("*.so")}
    env = dict(os.environ, HIPCC="/bin/false", PYTHONPATH=str(tmp_path))  # (a device compilation would fail)
    subprocess.run([sys.executable, "-m", "frisk_amd.build", "--if-missing"], cwd=tmp_path, env=env, check=True, capture_output=True, text=True)
    assert {p: p.stat().st_mtime_ns for p in present} == present and all((tmp_path / p).exists() for p in missing)
    out = subprocess.run([sys.executable, "-c", "from frisk_amd import runtime as R; import frisk; print(R.lib()._name, R.plan(R.make_desc(R.F16, 128, 128, 128)).tile_m > 0)"], cwd=tmp_path, env=env,
                         check=True, capture_output=True, text=True).stdout.split()
    assert out == [str(tmp_path / LIBRARY), "True"], out
