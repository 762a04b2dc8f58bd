"""cd_bvh_first_hit_order when allocations fail, in a host program of its own
(tests/plan/order_oom.cpp): an error code or the order, never the process's end."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_failing_allocations_end_in_a_status(tmp_path):
    exe = str(tmp_path / "order_oom")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-I" + os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "plan", "order_oom.cpp"),
                    os.path.join(ROOT, "poisson_caustic_design_amd", "csrc", "cd_bvh_order.cpp"),
                    "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
