"""The site buffers' buddy allocator on host memory, under the address and undefined-behaviour sanitizers:
once with room for everything and once with an allocator that often fails."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.parametrize("limit_mib,refuses", [(16384, False), (96, True)])
def test_site_pool(tmp_path, limit_mib, refuses):
    exe = str(tmp_path / "pool")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=address,undefined", "-o", exe,
                    os.path.join(HERE, "cpp", "site_pool_test.cpp")], check=True)
    r = subprocess.run([exe, str(limit_mib)], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:]
    assert r.stdout.startswith("ok") and (r.stdout != "ok, 0 refused\n") == refuses
