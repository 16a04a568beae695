"""Host phases on several threads where no further thread can be started: the calling thread does their work.

A child process without room for another thread's stack classifies the 73,920 pairs of a
dense assembly, which takes place before the device is used; without a device the call then reports that."""
import os
import subprocess
import sys
import textwrap

CHILD = """
import resource
import threading
import numpy as np
import bembel_amd as B
op = B.LaplaceSingleLayerOperator()
ps = B.AnsatzSpace(B.Geometry(), 3, 1, op)
d = op.desc()
out = np.zeros(486 * 486)
lib = B.library()
with open("/proc/self/statm") as f:
    pages = int(f.read().split()[0])
resource.setrlimit(resource.RLIMIT_AS, (pages * resource.getpagesize() + (7 << 20),) * 2)
hold, none_left = threading.Event(), False
while not none_left:  # stacks of finished threads are used again: until there is none
    try:
        threading.Thread(target=hold.wait, daemon=True).start()
    except RuntimeError:
        none_left = True
st = lib.bmi_dense_assemble(ps._h, B.C.byref(d), 0, B._dp(out), B.MEM_HOST, None)
print("status", st, lib.bmi_last_error().decode(), flush=True)
hold.set()
"""


def test_dense_assembly_without_threads(tmp_path):
    r = subprocess.run([sys.executable, "-c", textwrap.dedent(CHILD)], capture_output=True, text=True, timeout=120,
                       env={**os.environ, "HIP_VISIBLE_DEVICES": "-1"})
    # past the pairs: the first that fails is the allocation on a device that is not there
    assert r.returncode == 0 and "status 3 hipMalloc" in r.stdout, (r.returncode, r.stdout, r.stderr[-2000:])
