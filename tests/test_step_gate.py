"""The counters that decide whether a decode step takes its layers in one launch, by themselves on the CPU
(csrc/step_gate.h has no device code)."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_threads_count_down_to_zero_and_no_further(tmp_path):
    exe = str(tmp_path / "step_gate")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-pthread", "-o", exe, os.path.join(HERE, "step_gate.cpp")])
    run = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert run.returncode == 0 and run.stdout == "wrong 0\n", run.stdout
