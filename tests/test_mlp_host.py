"""Host rules of the surrogate network that a machine without a GPU can check: which nets one
launch may carry, and that passes sent ahead are waited for when one of them fails."""
import os
import subprocess

import spacelab_amd as sl

HERE = os.path.dirname(os.path.abspath(__file__))


def test_host_rules(tmp_path):
    exe = str(tmp_path / "mlp_host_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I" + os.path.join(HERE, "..", "spacelab_amd", "csrc"),
                    "-o", exe, os.path.join(HERE, "c", "mlp_host_check.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, check=True)
    assert r.stdout == ""


def _net(**change):
    m = sl.MLP.__new__(sl.MLP)     # no GPU: the attributes alone
    for k, v in {**dict(_m=None, device=0, n_in=21, n_out=9, width=256, max_batch=4096), **change}.items():
        setattr(m, k, v)
    return m


def test_nets_of_two_devices_are_not_alike():
    assert sl.mlp_alike([_net(), _net()])
    for change in (dict(device=1), dict(width=128), dict(max_batch=64), dict(n_in=20), dict(n_out=8)):
        assert not sl.mlp_alike([_net(), _net(**change)]), change
