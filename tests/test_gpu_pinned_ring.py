"""The pinned ring of the field transfers does not depend on the runtime's default for host memory."""
import os
import re
import subprocess
import sys

import pytest

from conftest import ROOT

CHILD = """
import sys
for p in {paths!r}:
    sys.path.insert(0, p)
import numpy as np
import peridynamics as pd
pos, vol = pd.lattice_block(200, 200, 37, 1e-3)  # 35.5 MB per vector field: the ring comes round twice
b = pd.Body(pd.BBMaterial(), pos, vol)
pd.material(b, horizon=1.2e-3, rho=2700.0, E=70e9)
dh = pd.MI355XBodyDataHandler(b)
for k in range(6):  # another field each time: a slot that was read before would show its old values
    v = np.random.default_rng(k).standard_normal((b.n_points, 3))
    dh.set("velocity", v)
    assert np.array_equal(dh.get("velocity"), v), k
    print("transfer", k, flush=True)
dh.close()
print("WHOLE", flush=True)
"""


def test_ring_and_events_name_their_coherence():
    """A kernel stores into the ring and host threads read it behind an event: neither may be left to
    HIP_HOST_COHERENT."""
    with open(os.path.join(ROOT, "peridynamics.jl_amd", "csrc", "pdx_export.hip")) as f:
        src = f.read()
    ring = re.search(r"hipHostMalloc\([^;{]*PDX_PIN_SLOTS[^;{]*\)", src).group(0)
    assert "hipHostMallocCoherent" in ring
    event = re.search(r"hipEventCreateWithFlags\(&c->pin_ev[^;{]*\)", src).group(0)
    assert "hipEventReleaseToSystem" in event


@pytest.mark.gpu
def test_fields_arrive_whole_with_another_default(need_gpu):
    """HIP_HOST_COHERENT=0 makes host memory non-coherent where an allocation does not say."""
    code = CHILD.format(paths=[ROOT, os.path.join(ROOT, "peridynamics.jl_amd")])
    r = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, HIP_HOST_COHERENT="0"),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "WHOLE" in r.stdout
