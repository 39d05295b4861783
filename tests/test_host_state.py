"""Host checks of engine state, as C++ programs over the library's own headers (no GPU)."""
import os
import subprocess

import pytest

from hmglib_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


# state: the states that captured products are compared with differ between successive H-matrices
# options: the near field's LDS reservation is set and given back
# kept: a kept buffer is not freed or handed on before its stream was waited for
@pytest.mark.parametrize("name", ["state", "options", "kept"])
def test_host_program(tmp_path, name):
    exe = str(tmp_path / name)
    subprocess.run([build.hipcc()] + build.FLAGS +
                   ["-I", build.CSRC, os.path.join(HERE, "host", name + ".cpp"), "-L", os.path.dirname(build.LIB),
                    "-l:libhmglib.so", "-Wl,-rpath," + os.path.dirname(build.LIB), "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
