"""The ordered pass's default launch shape against the timings shipped with the library: the rule
may cost a size at most 5% of the shape that was fastest there (timings of one size in
different runs differ by 2%)."""
import json
import os
import re
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.join(HERE, "..", "spacelab_amd")


def test_default_shape_is_near_the_fastest_shipped(tmp_path):
    with open(os.path.join(PKG, "data", "tune.json")) as f:
        timed = {k: v["ms"] for k, v in json.load(f).items() if k.startswith("ordered:")}
    assert len(timed) >= 4
    sizes = [re.search(r":n(\d+):", k).group(1) for k in timed]
    exe = str(tmp_path / "ordered_rule")
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I" + os.path.join(PKG, "csrc"), "-o", exe,
                    os.path.join(HERE, "c", "ordered_rule.cpp")], check=True)
    shapes = subprocess.run([exe] + sizes, capture_output=True, text=True, check=True).stdout.split()
    for (key, ms), shape in zip(timed.items(), shapes):
        assert len(ms) == 9
        assert ms[int(shape) - 1] <= 1.05 * min(ms), (key, shape, ms)
