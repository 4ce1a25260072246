"""Parts of the runtime that need no device, compiled for the host: which calls
write their host arrays in order (host_images.hpp), against a map of the written
bytes, and the cache of device blocks (block_cache.hpp) over a limited memory."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("check", ["host_images_check", "block_cache_check"])
def test_check_program(tmp_path, check):
    exe = tmp_path / check
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-o", str(exe),
                    os.path.join(HERE, check + ".cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout + out.stderr
