"""Which kernels a call of the C ABI takes, and what it does where memory
cannot be had, checked on the CPU: each scenario of host_routes.py runs the
library's host code in a child process over a stand-in of the HIP runtime."""
import os
import re
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
DRIVER = os.path.join(HERE, "host_routes.py")
NAMES = re.search(r"^SCENARIOS = \[(.*?)\]", open(DRIVER).read(), re.M | re.S).group(1).replace(",", " ").split()


@pytest.mark.parametrize("name", NAMES)
def test_route(name):
    assert os.path.exists(os.path.join(HERE, "cpp", "bin", "libfakehip.so")), "run __graft_entry__.build()"
    r = subprocess.run([sys.executable, DRIVER, name], capture_output=True, text=True, timeout=120)
    print(r.stdout[-3000:])
    assert r.returncode == 0, r.stderr[-3000:]
