"""Fields read back, used and dropped, step after step: the destinations'
memory stays with the process instead of being unmapped and faulted in again
(build.py, SOURCES).  In a process of its own, since what a process keeps
depends on what it has freed before."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SCRIPT = """
import resource
import lesgo_amd

def faults():
    return resource.getrusage(resource.RUSAGE_SELF).ru_minflt

cfg = lesgo_amd.Config(96, 48, 64, initu=False)
with lesgo_amd.Case(cfg) as c:
    c.seed_state(1)
    c.step(2)
    for n in range(8):
        before = faults()
        fields = [c.download(f) for f in ("u", "v", "w", "p")]
        del fields
        last = faults() - before
print("faults", last)
"""


def test_reads_fault_no_pages_in_again():
    """Four fields of 2.5 MB are 2430 pages; the first reads fault them in."""
    r = subprocess.run([sys.executable, "-c", SCRIPT], cwd=ROOT, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    n = int(r.stdout.split("faults")[1])
    print(f"  page faults of a round of reads: {n}", flush=True)
    assert n < 200
