"""A serving run whose stream slots are opened as launches need them: where memory runs out for a
further slot while requests are in flight, those already open serve the rest."""
from __future__ import annotations

import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# A dry run in a process of its own: a slot's descriptors for 200000 requests per launch take about
# 0.6 GiB of address space, and the limit leaves room for one slot only.  Requests arrive every
# 150 us and a launch stays in flight for 400000 polls, so that more than one slot is wanted.
CHILD = r"""
import resource, sys
sys.path[:0] = [%(root)r, %(tests)r]
import pfsolve_amd as pf
from test_serve_host import DryWorkload
import numpy as np
w = DryWorkload([(64, 3, i %% 4) for i in range(60)], seed=9)
for i, r in enumerate(w.reqs):
    r["arrival_s"] = 150e-6 * i
pf.serve(w.reqs[:1], hbm_budget=4 << 20, streams=1, dry_run=2)
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
if %(limit)d:
    resource.setrlimit(resource.RLIMIT_AS, (used + %(limit)d, used + %(limit)d))
st, out = pf.serve(w.reqs, hbm_budget=4 << 20, streams=4, max_batch=200000, max_inflight=64, dry_run=400000,
                   realtime=True)
assert st.requests == 60 and st.failed == 0 and st.rejected == 0, (st.requests, st.failed, st.rejected)
assert all(c == 0 for _, _, c in out)
for x, y in zip(w.ins, w.outs):
    np.testing.assert_array_equal(x, y)
print("launches", st.launches)
"""


def run(limit):
    code = CHILD % dict(root=ROOT, tests=os.path.join(ROOT, "tests"), limit=limit)
    p = subprocess.run([sys.executable, "-c", code], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                       timeout=120)
    assert p.returncode == 0, p.stdout
    return int(p.stdout.split()[-1])


def test_no_memory_for_a_further_slot():
    assert run(0) > 1                # without the limit: several launches in flight
    assert run(900 << 20) >= 1
