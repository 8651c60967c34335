"""Host-side parts of the library tested in C++: each program of tests/cpp
named here is compiled against csrc/ and the built library and run.  No GPU."""
import os
import subprocess

import pytest

from ecl_wavelet_amd import build

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("name", ["test_host_pipes", "test_pass_params"])
def test_cpp_host(tmp_path, name):
    exe = str(tmp_path / name)
    cmd = [build.hipcc(), *build.common_flags(), "-x", "hip",
           os.path.join(HERE, "cpp", name + ".cpp"), "-o", exe, "-L", build.PKG,
           "-lecl_wavelet_hip", "-Wl,-rpath," + build.PKG]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "ALL OK" in r.stdout, r.stdout[-3000:] + r.stderr[-2000:]
