"""bench.py without a GPU: the one-GPU contract (more GPUs exit with a message), the launch-variant
kernel names, and the HBM traffic read back from the committed rocprofv3 summary."""
import json
import os
import re
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import bench  # noqa: E402


def test_more_than_one_gpu_exits_with_a_message():
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True,
                       text=True, timeout=120, cwd=ROOT)
    assert r.returncode == 2
    msg = json.loads(r.stdout.strip().splitlines()[-1])
    assert msg["n_gpus"] == 2 and "one GPU" in msg["error"]


def test_kernel_names_follow_the_launch_variants():
    assert bench.kernel_name("hex", "double", 0) == "k_hex_forces<double, double, 256, 2, false>"
    assert bench.kernel_name("q4", "float", 3) == "k_q4_forces<float, float, 256, 3, false>"


def test_traffic_of_the_chosen_hex_variant_is_in_the_committed_profile():
    t = bench.measured_traffic(bench.kernel_name("hex", "double", 0))
    assert t is not None and 1.5e9 < t < 4.0e9
    assert bench.measured_traffic("k_not_a_kernel<double>") is None


def test_every_variant_has_the_name_of_a_kernel_that_is_built_and_profiled():
    built = {"k_hex_forces<double, double, 256, 2, false>", "k_hex_forces<float, float, 256, 2, false>",
             "k_hex_forces<float, float, 256, 3, false>", "k_q4_forces<double, double, 256, 2, false>",
             "k_q4_forces<float, float, 256, 2, false>", "k_q4_forces<float, float, 256, 3, false>"}
    names = {bench.kernel_name(f, r, v) for f in ("hex", "q4") for r in ("double", "float") for v in range(4)}
    assert names == built
    assert bench.kernel_name("hex", "float", 1) == bench.kernel_name("hex", "float", 0)
    text = open(os.path.join(ROOT, "profiles", "block160_plate1000_hbm_traffic.md")).read()
    listed = set(re.findall(r"`(k_(?:hex|q4)_forces<[^`]*>)`", text))
    assert listed == built
    for n in built:
        t = bench.measured_traffic(n)
        assert t is not None and 0.5e9 < t < 2.0e9, (n, t)
