"""bench.py's command line on the CPU: it measures one GPU only and says so,
before it touches a device, when asked for more; and the HBM traffic it prints
is that of the kernel and the workload it was measured on."""
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_more_than_one_gpu_is_refused_with_a_message():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], cwd=ROOT,
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 2
    assert "one GPU only" in r.stderr
    assert r.stdout == ""


def test_traffic_is_that_of_the_measured_workload():
    sys.path.insert(0, ROOT)
    import bench
    with open(os.path.join(ROOT, "profiles", "pmc_traffic.json")) as fh:
        kernels = json.load(fh)["kernels"]
    name = "k_gmres_coopw<2, 13>"  # nf = 800: 13 columns of 64 per lane
    assert bench.traffic_for(bench.KCLASS[4], "airfoil_flap") == (round(kernels[name]["bytes_per_launch"]), name)
    assert bench.traffic_for(bench.KCLASS[4], "plate") == (None, None)
