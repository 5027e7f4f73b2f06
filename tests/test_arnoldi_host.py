"""The Arnoldi steps on the CPU (host form of the sources): a step that loses w is repaired, the steps
after it, those past the fused sweeps' 15 vectors among them, are not."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_lost_step_is_repaired_once(tmp_path):
    src = os.path.join(HERE, "host", "arnoldi_steps.cpp")
    exe = str(tmp_path / "arnoldi_steps")
    subprocess.run(["g++", "-O0", "-std=c++17", "-ffp-contract=off", "-DLMFHD_HOST_DEBUG", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-o", exe, src], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, (res.stdout + res.stderr)[-4000:]
