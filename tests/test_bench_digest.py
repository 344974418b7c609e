"""The counter traffic that bench.py quotes is in force only for the kernels it was measured with:
the digest covers the per-step kernels' source and every header of this repository it includes."""
import os
import re

import bench

CSRC = "pannde_amd/csrc"


def test_digest_covers_what_the_kernels_are_built_from():
    seen, todo = set(), ["rsg_kernels.hip"]
    while todo:
        name = todo.pop()
        seen.add(name)
        with open(os.path.join(bench.ROOT, CSRC, name)) as f:
            todo += [i for i in re.findall(r'#include "([^"]+)"', f.read()) if i not in seen]
    assert {"%s/%s" % (CSRC, n) for n in seen} == set(bench.KERNEL_SOURCES)


def test_a_changed_header_changes_the_digest(tmp_path, monkeypatch):
    for rel in bench.KERNEL_SOURCES:
        os.makedirs(tmp_path / os.path.dirname(rel), exist_ok=True)
        with open(os.path.join(bench.ROOT, rel), "rb") as f:
            (tmp_path / rel).write_bytes(f.read())
    before = bench.kernel_sources_digest()
    monkeypatch.setattr(bench, "ROOT", str(tmp_path))
    assert bench.kernel_sources_digest() == before
    header = tmp_path / CSRC / "rsg_device.h"
    header.write_bytes(header.read_bytes() + b"// changed\n")
    assert bench.kernel_sources_digest() != before
