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


def test_results_without_the_pinned_buffer():
    """Where the 4 MB read-back buffer cannot be pinned, every call copies its
    results instead and returns the same."""
    run_alone("""
    rng = np.random.default_rng(1)
    x = rng.random((20, 3)).astype(np.float32)

    def everything():
        out = {}
        b = make_batch()
        b.run(7)
        out["batch csr"] = b.csr_histories(0, 7)
        out["batch profiles"] = np.concatenate(b.projections())
        desc, d = kick_drift_config(n=60, steps_per_ts=500)
        zw, zc = impedances(d)
        st = V.Step(desc, initial_mesh(60, seed=4), zw, zc)
        st.record(5)
        st.run(5)
        for k, v in st.moments().items():
            out["moments " + k] = v
        out["mesh"], out["profile"], out["wake"] = st.mesh()
        out["history"] = st.history()[0]
        ps = V.PhaseSpace(40, -6.0, 6.0, 1e-3, -6.0, 6.0, 1e5,
                          filling=[0.25, 0.75])
        out["variance"] = np.concatenate(
            [np.ravel(v) for axis in (0, 1) for v in ps.variance(axis)])
        out["integral"] = np.append(*ps.integrate())
        f = V.ElectricField(ps, V.Impedance(256, 1e12,
                                            table=np.ones(256, np.complex64)),
                            [0, 1], 50)
        out["potential"] = f.wakePotential()
        out["csr"] = f.updateCSR(0.0)[0]
        net = V.MLP((3, 40, 9), max_batch=20, seed=2)
        out["net"] = net.forward(x)
        return out

    faults.hip_faults_pinned(1 << 20)
    without = everything()
    seen = faults.hip_faults_refused()
    assert seen >= 10
    faults.hip_faults_pinned(0)
    with_it = everything()
    assert faults.hip_faults_refused() == seen
    assert without.keys() == with_it.keys()
    for k in without:
        for a, e in zip(np.atleast_1d(without[k]), np.atleast_1d(with_it[k])):
            np.testing.assert_array_equal(a, e, err_msg=k)
    """)


def test_refused_meshes_are_freed():
    """A mesh whose row exceeds the LDS of a CU is refused after its 6.7 GB
    are allocated; nothing of it stays."""
    run_alone("""
    keep = V.PhaseSpace(32, -6.0, 6.0, 1e-3, -6.0, 6.0, 1e6)
    live = faults.hip_faults_live()
    try:
        V.PhaseSpace(40961, -6.0, 6.0, 1e-3, -6.0, 6.0, 1e6)
        sys.exit("a row beyond the LDS was accepted")
    except V.VfpsInvalid:
        pass
    assert faults.hip_faults_live() == live
    """)
