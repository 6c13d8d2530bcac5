"""The committed HBM-traffic figure is of the decode sources as they are: bench.py's hash covers
every file the counted launch pair is compiled from, and the summary carries it."""
import os
import re
import shutil

import bench


def test_the_committed_figure_is_current():
    traffic, kernels = bench.measured_traffic()
    assert traffic is not None, kernels
    assert "paged_decode_kernel" in kernels and "merge_kernel" in kernels


def test_the_hash_covers_every_included_source(tmp_path):
    src = os.path.dirname(bench.DECODE_SOURCES[0])
    todo, seen = ["paged_decode.hip"], set()
    while todo:
        name = todo.pop()
        seen.add(name)
        with open(os.path.join(src, name)) as f:
            todo += [n for n in re.findall(r'#include "(\w+\.hpp)"', f.read()) if n not in seen]
    assert seen == {os.path.basename(p) for p in bench.DECODE_SOURCES}
    was = bench.source_sha16()
    for i, path in enumerate(bench.DECODE_SOURCES):
        copy = tmp_path / f"{i}"
        shutil.copy(path, copy)
        with open(copy, "a") as f:
            f.write("// changed\n")
        paths = list(bench.DECODE_SOURCES)
        paths[i] = str(copy)
        assert bench.source_sha16(paths) != was
