"""The block codec's forms for planes with many runs against its step-per-run forms, on the CPU."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_planes_with_many_runs_come_out_the_same_in_both_forms(tmp_path):
    exe = str(tmp_path / "plane_forms")
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-o", exe,
                    os.path.join(HERE, "cpp_plane_forms.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
