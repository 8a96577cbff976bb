"""The site buffers' allocator takes from the device what it is asked for, and an eighth more at most at the ends of
its slabs: the HBM budget counts the bytes asked for."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_held_is_what_was_asked(tmp_path):
    exe = str(tmp_path / "pool")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=address,undefined", "-o", exe,
                    os.path.join(HERE, "cpp", "site_pool_bytes_test.cpp")], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-2000:]
