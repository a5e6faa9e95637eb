"""The rule that gives a flat call its kernel (csrc/routes.h), over every shape,
compiled for the host."""
import os
import subprocess

from conftest import ROOT


def test_flat_routes(tmp_path):
    exe = str(tmp_path / "routes")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "megatron-lm_amd", "csrc"),
                    os.path.join(ROOT, "tests", "routes_driver.cpp"), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stdout[-2000:]
    assert "routes driver ok" in out.stdout
