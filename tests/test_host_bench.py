"""bench.py reports counter measurements only for the kernel sources they were taken
on: its hash covers every source of a measured kernel and the headers these include."""
import os
import re

import bench


def test_traffic_hash_covers_sources_and_headers():
    root = os.path.dirname(os.path.abspath(bench.__file__))
    text = {p: open(os.path.join(root, p)).read() for p in bench.KERNEL_SOURCES}
    for path, src in text.items():
        for header in re.findall(r'#include "([^"]+)"', src):
            name = os.path.normpath(os.path.join(os.path.dirname(path), header))
            assert name in bench.KERNEL_SOURCES or not name.startswith("usaf_amd/"), f"{path} includes {name}"
    with open(bench.TRAFFIC_FILE.replace(".json", ".md")) as f:
        kernels = re.findall(r"\(`(\w+_kernel)\b", f.read())
    assert kernels
    for name in kernels:
        assert any(re.search(rf"__global__[^;{{]*\b{name}\(", src) for src in text.values()), name
