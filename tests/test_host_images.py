"""Which calls write their host arrays in order (host_images.hpp), compiled for
the host, against a map of the written bytes (host_images_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_overlap_rule_matches_written_bytes(tmp_path):
    exe = tmp_path / "host_images_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-o", str(exe),
                    os.path.join(HERE, "host_images_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
