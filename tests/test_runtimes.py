"""The count of loaded HIP runtimes against the process's maps, with torch loaded before and after
the library."""
import subprocess
import sys

import pytest

CODE = """
%s
from dmtz_amd import _native
n = _native.lib().dmtz_hip_runtimes()
%s
m = _native.lib().dmtz_hip_runtimes()
paths = {l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64.so" in l}
assert m == len(paths), (m, paths)
assert n == 1, n
"""


@pytest.mark.parametrize("order", [("import torch", ""), ("", "import torch"), ("", "")])
def test_runtimes_equal_the_maps(order):
    r = subprocess.run([sys.executable, "-c", CODE % order], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
