"""bench.py reads the profiler's rows by kernel name: every pattern of its
counter sets names kernels of the built library, and the dense, causal,
default and exact softmax rows name different ones."""
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


def kernel_names():
    lib = os.path.join(ROOT, "chelis_amd", "libchelis_hip.so")
    out = subprocess.run(["nm", "-C", lib], capture_output=True, text=True, check=True).stdout
    return [ln.split(" ", 2)[2] for ln in out.splitlines() if "_kernel" in ln and "__device_stub__" not in ln]


@pytest.mark.parametrize("set_name", ["BW_SET", "MFMA_SET", "TRANSFORMER_SET", "VALU_SET"])
def test_counter_patterns_name_built_kernels(set_name):
    names, seen = kernel_names(), {}
    for entry in getattr(bench, set_name):
        matched = frozenset(n for n in names if re.search(entry[1], n))
        assert matched, entry[0]
        if "softmax_kernel" in entry[1]:
            assert all(not (matched & other) for other in seen.values()), entry[0]
            seen[entry[0]] = matched


def test_dense_softmax_pattern_is_the_headline_kernel():
    pattern = dict((e[0], e[1]) for e in bench.BW_SET)["softmax_f32_16384x1024"]
    assert re.search(pattern, "void chelis::softmax_kernel<float, 4, 2, 2, 1, 64, true, false, false>(float const*)")
