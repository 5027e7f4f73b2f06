"""The staggered tile on the CPU: which places of its box a tile reads, for the even extents on both
sides of every tile boundary, and its stored faces against plain half sweeps, bit for bit.  Built
with bounds checks on every array (AddressSanitizer, host code only)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_tile_stays_in_its_box(tmp_path):
    src = os.path.join(HERE, "host", "tile_sweeps.cpp")
    exe = str(tmp_path / "tile_sweeps")
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-fsanitize=address", "-static-libasan",
                    "-DLMFHD_HOST_DEBUG", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", exe, src], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, (res.stdout + res.stderr)[-4000:]
