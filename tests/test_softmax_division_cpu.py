"""The short divisions of the 16-bit softmax kernels against the rounded f32 division, on the host.  No GPU needed."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_short_divisions_round_as_the_division_does(tmp_path):
    exe = tmp_path / "softmax_division_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", "-I", os.path.join(ROOT, "ratchet_amd", "csrc"), os.path.join(ROOT, "tests", "softmax_division_check.cpp"),
                    "-o", str(exe)], check=True)
    run = subprocess.run([str(exe), "1"], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout + run.stderr
    fields = run.stdout.split()
    counts = dict(zip(fields[0::2], (int(v) for v in fields[1::2])))
    assert counts["f16"] == 0 and counts["bf16"] == 0 and counts["checked"] > 1_845_000_000, run.stdout
