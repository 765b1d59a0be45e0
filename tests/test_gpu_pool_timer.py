"""GPU check that freed memory goes back to the device without a further call: a program that has closed its systems
and makes none any more holds, some ten seconds later, none of the chunks they used. In a process of its own, whose
exit the timer must not delay, and again with a chunk that is young when the process ends.
"""
import os
import subprocess
import sys
import time

import pytest

from .conftest import ROOT

pytestmark = pytest.mark.gpu

PROGRAM = """
import sys, time
import torch
from cppe_amd import capi, synthetic
free = lambda: torch.cuda.mem_get_info()[0]
w = synthetic.water_box(8000, 3, anisotropic=True)
def use():
    S = capi.System(w.pos, w.pol, w.alpha_iso(), w.excl_csr(), summation="fmm", damping=2.1304)
    S.apply_b(w.pos.ravel())
    held = free()
    S.close()
    return held
use()
time.sleep(float(sys.argv[1]))
before = free()
held = use()
after = free()
time.sleep(float(sys.argv[1]))
print("held", before - held, "kept", before - after, "later", before - free(), flush=True)
"""


@pytest.mark.parametrize("wait", [13.0, 0.5])
def test_chunks_go_back_by_themselves(wait):
    print("pool timer, seconds", wait, flush=True)
    t = time.monotonic()
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(wait)], cwd=ROOT, capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, PYTHONPATH=ROOT))
    assert r.returncode == 0, r.stderr[-2000:]
    words = r.stdout.split()
    held, kept, later = (int(words[k]) for k in (1, 3, 5))
    if wait > 10.0:
        assert held > 4 << 20 and kept > 4 << 20  # a system's chunks, held back for a while
        assert later <= 2 << 20  # (what the runtime's own pool keeps)
    assert time.monotonic() - t < 2 * wait + 60.0
