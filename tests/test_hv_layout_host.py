"""Host checks of what the H.v kernels read of a layout
(tests/cpp/hv_layout_host.cpp, no device)."""
import os
import subprocess

import pytest

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "_build", "hv_layout_host")
CHECKS = ["shared_low_table", "segment_order", "page_positions", "cross_stages", "many_cross_bonds"]


@pytest.fixture(scope="module")
def report():
    out = subprocess.run([BIN], capture_output=True, text=True, check=True, timeout=120).stdout
    return {f[0]: (int(f[1]), int(f[2])) for f in (line.split() for line in out.splitlines())}


@pytest.mark.parametrize("name", CHECKS)
def test_layout(report, name):
    bad, checked = report[name]
    assert bad == 0 and checked > 0
