"""Steps in flight at the widths of the pipelined workloads (20 steps of 6 workgroups, 10 of 16): every step's sweep runs
beside the others' and equals the same steps one at a time, bit for bit.  In a process of its own, because the hardware
queues that let all steps run at once are fixed when HIP starts."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import sys
import numpy as np
import torch
import quarz_amd as qa
from quarz_amd import configs
work, case = sys.argv[1], sys.argv[2]
if case == "c2":   # the reference steps run on one workgroup
    deck, groups, ref, steps, depth, chunks = configs.deck("c2", workdir=work), 6, 1, 20, 20, 12
    ov = {"xi.min": -1.5, "time.steps": steps + 1, "driver.nparticles": 40000, "witness.nparticles": 20000,
          "driver.sigma_xi": 0.2, "driver.xi0": -0.6, "witness.sigma_xi": 0.05, "witness.xi0": -1.2}
else:
    deck, groups, ref, steps, depth, chunks = configs.c3_deck(workdir=work, xi_min=-1.5, steps=11, nd=100000, nw=20000,
                                                              driver_xi0=-0.6, witness_xi0=-1.2), 16, 16, 10, 10, 12
    ov = {"driver.sigma_xi": 0.2, "driver.x0": 0.05, "driver.n0": 2, "witness.sigma_xi": 0.05}
a = qa.Simulation(deck, {**ov, "sweep.groups": ref})
b = qa.Simulation(deck, {**ov, "sweep.groups": groups})
assert a.groups == ref and b.groups == groups
for n in range(steps + 1):
    a.step()
print("one at a time", flush=True)
b.step()
b.run_pipelined(steps, chunks=chunks, depth=depth)
print("in flight", flush=True)
for w in ("fld", "diag", "bsrc"):
    x, y = np.array(getattr(a, w)), np.array(getattr(b, w))
    assert x.shape == y.shape and np.array_equal(x, y), (w, int((x != y).sum()), np.argwhere(x != y)[:3])
for i in range(a.nbeams):
    for k in qa.BEAM_ARRAYS:
        assert np.array_equal(a.get(f"beam{i}.{k}"), b.get(f"beam{i}.{k}")), (i, k)
assert a.lost() == b.lost()
print("same", flush=True)
"""


@pytest.mark.parametrize("case,queues", [("c2", 24), ("c3", 14)])
def test_steps_in_flight_at_full_width(tmp_path, case, queues):
    env = dict(os.environ, PYTHONPATH=ROOT, GPU_MAX_HW_QUEUES=str(queues))
    r = subprocess.run([sys.executable, "-u", "-c", CHILD, str(tmp_path), case], env=env, cwd=ROOT, capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("same\n"), (r.returncode, r.stdout[-500:], r.stderr[-2000:])
