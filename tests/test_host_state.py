"""Host checks of engine state, as a C++ program over the library's own headers (no GPU)."""
import os
import subprocess

from hmglib_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


def test_states_of_successive_h_matrices_differ(tmp_path):
    exe = str(tmp_path / "state")
    subprocess.run([build.hipcc()] + build.FLAGS +
                   ["-I", build.CSRC, os.path.join(HERE, "host", "state.cpp"), "-L", os.path.dirname(build.LIB), "-l:libhmglib.so",
                    "-Wl,-rpath," + os.path.dirname(build.LIB), "-o", exe], check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
