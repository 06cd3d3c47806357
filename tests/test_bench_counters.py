"""bench.py's counter patterns against the kernels that libvgi.so holds: a kernel that is renamed,
or gains a template argument, would drop out of the counters without a word."""
import os
import re
import shutil
import subprocess

import pytest

import bench

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def kernels():
    if shutil.which("nm") is None:
        pytest.skip("nm not found")
    out = subprocess.run(["nm", "-C", os.path.join(ROOT, "final184_amd", "libvgi.so")], check=True, capture_output=True,
                         text=True).stdout
    return sorted(set(re.findall(r"__device_stub__(k_\w+(?:<[^>]*>)?)\(", out)))


def test_every_counter_pattern_names_a_kernel(kernels):
    assert len(kernels) > 20
    for key, rx in bench.COUNTER_KERNELS:
        assert any(re.search(rx, k) for k in kernels), f"{key}: {rx} names no kernel"


def test_every_trace_and_plain_mip_kernel_is_counted(kernels):
    """Whichever of a precision's kernels a call's size picks, its counters go to one key."""
    rx = dict(bench.COUNTER_KERNELS)
    for prec, number in (("fp32", 0), ("fp16", 1), ("fp16x2", 3)):
        traces = [k for k in kernels if re.match(rf"k_trace\w*<{number}\b", k)]
        assert len(traces) > 1
        assert [k for k in kernels if re.search(rx[f"trace_{prec}"], k)] == traces
        mips = [k for k in kernels if re.match(rf"k_mips<{number}, \w+, 0>", k)]
        got = [k for k in kernels if any(re.search(rx[f"mips_{prec}_{part}"], k) for part in ("first", "rest"))]
        assert got == mips and len(mips) == 2
