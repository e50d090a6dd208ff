"""The places of small models' loops (csrc/small_place.h), on the CPU."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_places_under_threads(tmp_path):
    exe = str(tmp_path / "small_place")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", os.path.join(HERE, "..", "simplellminference_amd", "csrc"),
                    os.path.join(HERE, "cpp", "small_place.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
