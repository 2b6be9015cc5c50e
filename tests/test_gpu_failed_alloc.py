"""Allocations that fail, refused on the host (tests/cpp/hip_faults.c) in a
process of their own: what the call returns, and the calls after it."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

pytestmark = pytest.mark.gpu

SETUP = """
import ctypes as C
import sys
faults = C.CDLL({faults!r}, mode=C.RTLD_GLOBAL)   # ahead of libvfps.so
faults.hip_faults_pinned.argtypes = [C.c_size_t]
import numpy as np
import inovesa_amd as V
from inovesa_amd.workloads import impedances, initial_mesh, kick_drift_config


def make_batch(k=3):
    descs, inits, zs = [], [], []
    for i, (n, wake) in enumerate(((64, 2), (36, 1), (100, 2))[:k]):
        desc, d = kick_drift_config(n=n, steps_per_ts=500)
        descs.append(dict(desc, wake_method=wake))
        inits.append(initial_mesh(n, seed=i))
        zs.append(impedances(d))
    b = V.Batch(descs, inits, [z[0] for z in zs], [z[1] for z in zs])
    b.record(8)
    return b
"""


def run_alone(body):
    code = SETUP.format(faults=os.path.join(HERE, "cpp", "libhip_faults.so"))
    r = subprocess.run([sys.executable, "-c", code + textwrap.dedent(body)],
                       cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr


def test_batch_descriptors():
    """A batch's descriptors are built by the first run: if one of their two
    allocations or uploads fails, so does the run, nothing of them is kept or
    lost, and the next run builds them."""
    run_alone("""
    ref = make_batch()
    ref.run(5)
    expect = ref.csr_histories(0, 5), ref.projections()
    for call in (1, 2, 3, 4):
        b = make_batch()
        live = faults.hip_faults_live()
        seen = faults.hip_faults_refused()
        faults.hip_faults_at(call)
        try:
            b.run(5)
            sys.exit("run() with a failed allocation succeeded")
        except V.VfpsError:
            pass
        assert faults.hip_faults_refused() == seen + 1
        assert faults.hip_faults_live() == live
        b.run(5)
        assert faults.hip_faults_live() == live + 2
        np.testing.assert_array_equal(b.csr_histories(0, 5), expect[0])
        for a, e in zip(b.projections(), expect[1]):
            np.testing.assert_array_equal(a, e)
    """)
