"""bench.py publishes a committed counter summary only while the hash of the
kernel sources is the one it was measured on, so that hash has to cover every
file the kernels are made of."""
import os
import re

import bench


def test_every_included_project_file_is_hashed():
    csrc = os.path.join(bench.ROOT, "dendro-gr_amd", "csrc")
    dirs = (csrc, os.path.join(bench.ROOT, "include"))
    todo, seen = [os.path.join(csrc, "dgr_bssn.hip")], set()
    while todo:
        f = todo.pop()
        if f in seen:
            continue
        seen.add(f)
        with open(f) as fh:
            for name in re.findall(r'^\s*#\s*include\s+"([^"]+)"', fh.read(), re.M):
                todo += [p for p in (os.path.join(d, name) for d in dirs) if os.path.exists(p)]
    rel = {os.path.relpath(f, bench.ROOT) for f in seen}
    assert "dendro-gr_amd/csrc/stream_tile.h" in rel  # included inside a kernel, not at the top
    assert rel <= set(bench.KERNEL_SOURCES), rel - set(bench.KERNEL_SOURCES)
