"""Results read through pinned staging by several threads.

* The device fails on the way: the kernel that stores the last chunks never runs
  (the emulated device fails at its launch, which only a query of the stream
  shows). The read has to raise, also where another reader than the caller's
  thread waits for such a chunk.
* A process with few cores starts no more readers than it has cores for.
"""
import os
import subprocess
import sys

import pytest


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


COUNT = """
import os, sys, threading
sys.path[:0] = [{pkg!r}, {oracle!r}]
os.sched_setaffinity(0, sorted(os.sched_getaffinity(0))[:{cores}])
import numpy as np
import sgraph
sgraph.LIB_PATH = {path!r}
nv = 26 * (1 << 17)
deg = np.arange(nv) % 3 == 0
row = np.zeros(nv + 1, np.uint64)
np.cumsum(deg, out=row[1:])
eng = sgraph.Engine("bfs", round_blocks=8)
eng.load_csr(row, np.zeros(int(row[-1]), np.uint32))
most, stop = 0, False
def watch():
    global most
    while not stop:
        most = max(most, len(os.listdir("/proc/self/task")))
w = threading.Thread(target=watch)
w.start()
before = len(os.listdir("/proc/self/task"))
assert np.array_equal(eng.gather(sgraph.Q_DEGREE), deg)
stop = True
w.join()
print("readers", most - before, flush=True)
os._exit(0)
"""


@pytest.mark.parametrize("cores,readers", [(1, 0), (2, 1)])
def test_no_more_readers_than_cores(emulated_path, cores, readers):
    if len(os.sched_getaffinity(0)) < 2:
        pytest.skip("one core")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = COUNT.format(pkg=os.path.join(root, "c-gpustreamgraph_amd"), oracle=os.path.join(root, "oracle"),
                        path=emulated_path, cores=cores)
    p = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert p.returncode == 0 and f"readers {readers}\n" in p.stdout, p.stdout + p.stderr
