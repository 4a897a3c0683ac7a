"""The library's build stands on its own: no test program, missing or broken, fails it."""
import os
import shutil
import subprocess
import sys

import pytest

from tests.conftest import ROOT

PROGRAMS = ("dropin_check", "core_emulation", "packed_emulation")


@pytest.mark.parametrize("programs", ["missing", "broken"])
def test_build_needs_no_test_program(tmp_path, programs):
    skip = shutil.ignore_patterns("*.so", "*.o", "_build", "_ref", "__pycache__")
    for d in ("cubiquity_amd", "include", "oracle"):
        shutil.copytree(os.path.join(ROOT, d), tmp_path / d, ignore=skip)
    shutil.copy(os.path.join(ROOT, "__graft_entry__.py"), tmp_path)
    cpp = tmp_path / "tests" / "cpp"
    if programs == "broken":
        cpp.mkdir(parents=True)
        for name in PROGRAMS:
            (cpp / f"{name}.cpp").write_text("#error a test program that does not compile\n")
            (cpp / name).write_text("of an older source\n")
        (cpp / "in_the_way").mkdir()
        (cpp / PROGRAMS[1]).unlink()
        (cpp / "in_the_way").rename(cpp / PROGRAMS[1])  # one that cannot be removed as a file
    r = subprocess.run([sys.executable, "-c", "import __graft_entry__ as g; g.build()"], cwd=tmp_path, timeout=300,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert r.returncode == 0, r.stdout
    assert (tmp_path / "cubiquity_amd" / "libcqx.so").exists() and (tmp_path / "oracle" / "liboracle.so").exists()
    for name in PROGRAMS:
        assert not (cpp / name).is_file()
        assert programs == "missing" or f"test program {name} not built" in r.stdout
