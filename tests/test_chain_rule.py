"""The rule that chooses how a measurement's environments are formed, against measured times of both ways."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_the_way_taken_is_the_faster_one(tmp_path):
    exe = str(tmp_path / "rule")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=address,undefined", "-o", exe,
                    os.path.join(HERE, "cpp", "chain_rule_test.cpp")], check=True)
    r = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
