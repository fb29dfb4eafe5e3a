"""Results read through pinned staging when the device fails on the way.

The kernel that stores the last chunks never runs (the emulated device fails at
its launch, which only a query of the stream shows): the read has to raise, also
where another reader than the caller's thread waits for such a chunk.
"""
import os
import subprocess
import sys

import pytest

from emulated import emulated_path  # noqa: F401 (fixture)

CHILD = """
import ctypes, sys
sys.path[:0] = [{pkg!r}, {oracle!r}]
import numpy as np
import sgraph
sgraph.LIB_PATH = {path!r}
so = ctypes.CDLL({path!r})
nv = {chunks} * (1 << 17) - 5  # words in chunks of 512 KiB, eight to a launch
eng = sgraph.Engine("bfs", round_blocks=8)
eng.load_csr(np.zeros(nv + 1, np.uint64), np.zeros(0, np.uint32))
assert not eng.gather(sgraph.Q_DEGREE).any()
so.emulation_fail_launch(b"k_publish_chunks", {after})
try:
    eng.gather(sgraph.Q_DEGREE)
except sgraph.SgError as e:
    print("raised", e, flush=True)
    import os
    os._exit(0)
"""


@pytest.mark.parametrize("chunks,after", [(2, 0), (9, 0), (9, 1)])
def test_a_failed_read_raises(emulated_path, chunks, after):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = CHILD.format(pkg=os.path.join(root, "c-gpustreamgraph_amd"), oracle=os.path.join(root, "oracle"),
                        path=emulated_path, chunks=chunks, after=after)
    for _ in range(3):  # which reader waits for the chunk is up to the threads
        p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=60)
        assert p.returncode == 0 and "raised SG_EDEVICE" in p.stdout, p.stdout + p.stderr
