"""The host's side of the counters against a stand-in for the device: what it keeps
of them where calls, readers and failures meet at the worst moment, which a real
device only does now and then."""
import inspect
import os
import shutil
import subprocess
import sys

import pytest

import host_scenarios

HERE = os.path.dirname(os.path.abspath(__file__))
SCENARIOS = [name for name, f in vars(host_scenarios).items()
             if inspect.isfunction(f) and f.__module__ == "host_scenarios" and not name.startswith("_")]


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("stand_in") / "libstand_in.so")
    subprocess.check_call([shutil.which("gcc") or "gcc", "-O1", "-fPIC", "-shared", "-Wall",
                           os.path.join(HERE, "stand_in_runtime.c"), "-o", out])
    return out


@pytest.mark.parametrize("scenario", SCENARIOS)
def test_counters_on_the_host(stand_in, scenario):
    done = subprocess.run([sys.executable, os.path.join(HERE, "stand_in_device.py"), stand_in, scenario],
                          capture_output=True, text=True, timeout=120, cwd=HERE)
    assert done.returncode == 0 and "as it should be" in done.stdout, done.stdout + done.stderr
