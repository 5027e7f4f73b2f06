"""The on-device noise's map from words to N(0,1) on the CPU (host form of the sources), at both ends of
a word's range."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_extreme_words(tmp_path):
    src = os.path.join(HERE, "host", "noise_words.cpp")
    exe = str(tmp_path / "noise_words")
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-o", exe, src], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, (res.stdout + res.stderr)[-4000:]
