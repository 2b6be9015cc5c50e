"""Fused steps of meshes whose rows are no whole groups of four: the same
maps one by one, bit for bit (the kicks make four outputs a thread), and the
oracle's step."""
import numpy as np
import pytest

from _helpers import oracle_cfg, rel_linf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 6, 7, 17, 18, 33, 65, 66, 130, 259])
@pytest.mark.parametrize("scheme", [0, 1])
@pytest.mark.parametrize("use_wake", [0, 1])
def test_fused_equals_the_maps(n, scheme, use_wake):
    import inovesa_amd as V
    from inovesa_amd.workloads import (impedances, initial_mesh,
                                       kick_drift_config, rotation_config)
    conf = rotation_config if scheme else kick_drift_config
    desc, d = conf(n=n, steps_per_ts=4000)
    zw, zc = impedances(d)
    desc = dict(desc, use_wake=use_wake, use_csr=0, wake_method=1)
    init = initial_mesh(n, seed=2)
    got = {}
    for fused in (0, 1):
        st = V.Step(dict(desc, fused=fused), init, zw if use_wake else None)
        st.run(3)
        got[fused] = st.mesh()
    for a, b in zip(got[0], got[1]):
        assert np.all(np.isfinite(b))
        np.testing.assert_array_equal(a, b)
    b = V.Batch([desc] * 2, [init] * 2, [zw if use_wake else None] * 2,
                [None] * 2)
    b.run(3)
    for x, y in zip(b.mesh(1), got[1]):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("n", [33, 130])
def test_direct_wake_matches_oracle(n, orc):
    import inovesa_amd as V
    from inovesa_amd.workloads import (impedances, initial_mesh,
                                       kick_drift_config)
    desc, d = kick_drift_config(n=n, steps_per_ts=4000)
    zw, zc = impedances(d)
    init = initial_mesh(n, seed=2)
    st = V.Step(desc, init, zw, zc)
    st.run(1)
    mesh, proj, wake = st.mesh()
    sim = orc.sim(oracle_cfg(desc, zw.n), init, zw.data(), zc.data())
    sim.run(1, want_csr=True)
    omesh, oproj, owake = sim.get()
    # bounds of test_gpu_step.py
    assert rel_linf(wake, owake) <= 1e-5
    assert rel_linf(mesh, omesh) <= 1e-5
    assert rel_linf(proj, oproj) <= 1e-5
