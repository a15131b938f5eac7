"""The wave-per-row norms' ordered sums against the plain left-to-right f32 sum, on the host.  No GPU needed."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_ordered_sums_are_the_plain_sums(tmp_path):
    exe = tmp_path / "ordered_sums_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-I", os.path.join(ROOT, "ratchet_amd", "csrc"), os.path.join(ROOT, "tests", "ordered_sums_check.cpp"),
                    "-o", str(exe)], check=True)
    run = subprocess.run([str(exe), "300"], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout + run.stderr
    assert int(run.stdout.split()[-1]) > 3000, run.stdout
