"""The rules for the memory of the large products' decoded weights
(fh3_fragments.h), run against a runtime that only keeps books: no GPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_rules(tmp_path):
    exe = str(tmp_path / "weight_fragments")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror",
                    "-I" + os.path.join(ROOT, "fasth3inc_amd", "csrc"),
                    os.path.join(ROOT, "tests", "c", "weight_fragments.cpp"), "-o", exe], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout
