"""The excluded-volume entry points that the kernels call are the combined form's values bit for bit
(tests/cpp/exvol_entry_check.cpp, FP64 path, on the host), so the accuracy measured on that form is theirs."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_separate_calls_are_the_combined_form(tmp_path):
    hipcc = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")
    exe = str(tmp_path / "exvol_entry_check")
    subprocess.run([hipcc, "--offload-host-only", "-O2", "-std=c++17", "-ffp-contract=off", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "exvol_entry_check.cpp")], check=True, capture_output=True)
    n, deferred, bad = (int(v) for v in subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split())
    assert n == 60000 and deferred > 1000 and bad == 0
