"""Results that come back through the device handle's pinned buffer, and
small arrays that go up as kernel arguments, at the sizes where the route
changes; the y projection and the moments at every kind of remainder."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(V, n, nb, seed):
    rng = np.random.default_rng(seed)
    m = rng.random((nb, n, n)).astype(np.float32)
    return m, V.PhaseSpace(n, -6.0, 5.0, 1e-3, -6.0, 6.5, 1e6,
                           filling=[1.0 / nb] * nb, data=m)


@pytest.mark.parametrize("n", [3, 4, 15, 16, 20, 61, 250, 512, 516, 1028])
@pytest.mark.parametrize("nb", [1, 2])
def test_projections_and_moments(n, nb):
    import inovesa_amd as V
    m, ps = _mesh(V, n, nb, n)
    ws = ps.simpsonWeights()
    acc = np.zeros((nb, n), np.float32)
    for x in range(n):                       # the reference's order
        acc = acc + m[:, x, :] * ws[x]
    ps.updateXProjection()
    ps.updateYProjection()
    np.testing.assert_array_equal(ps.getProjection(1), acc)
    fill, tot = ps.integrate()
    px = ps.getProjection(0).astype(np.float64)
    np.testing.assert_allclose(fill, px @ ws.astype(np.float64), rtol=1e-12)
    assert tot == pytest.approx(fill.sum(), rel=1e-12)
    for axis, p in ((0, px), (1, acc.astype(np.float64))):
        a = ps.getAxis(axis).astype(np.float64)
        d = float(ps.getDelta(axis))
        mean, var, rms = ps.variance(axis)
        rm = p @ a * d / fill
        rv = ((a - rm[:, None]) ** 2 * p).sum(1) * d / fill
        # the mean is rounded to float before it enters the variance
        np.testing.assert_allclose(mean, rm, rtol=1e-6, atol=1e-6)
        np.testing.assert_allclose(var, rv, rtol=1e-5)
        np.testing.assert_allclose(rms, np.sqrt(rv), rtol=1e-5)


@pytest.mark.parametrize("n,nb", [(480, 2), (481, 2), (1000, 1), (320, 12),
                                  (321, 12), (700, 30)])
def test_small_uploads_and_readbacks(n, nb):
    """960 floats a launch, 3840 in all, 64 KiB back."""
    import inovesa_amd as V
    ps = V.PhaseSpace(n, -6.0, 6.0, 1e-3, -6.0, 6.0, 1e6,
                      filling=[1.0 / nb] * nb)
    rng = np.random.default_rng(n)
    p = rng.random((nb, n)).astype(np.float32)
    ps.setProjection(0, p)
    q = p.copy()
    p[:] = 0                                 # borrowed for the call only
    np.testing.assert_array_equal(ps.getProjection(0), q)
    k = V.KickMap(ps, ps.clone(), 4, False, V.Axis.y)
    k.swapOffset(q.ravel())
    np.testing.assert_array_equal(k.getForce(), q.ravel())


@pytest.mark.parametrize("fused,scheme,steps", [(1, 0, 3), (1, 1, 4), (0, 0, 3)])
def test_step_moments_are_the_mesh_s(fused, scheme, steps):
    import inovesa_amd as V
    from inovesa_amd.workloads import (impedances, initial_mesh,
                                       kick_drift_config, rotation_config)
    desc, d = (rotation_config if scheme else kick_drift_config)(n=100)
    desc = dict(desc, fused=fused)
    st = V.Step(desc, initial_mesh(100, seed=2), *impedances(d))
    st.record(20000)
    st.run(steps)
    m = st.moments()
    mesh, proj, _ = st.mesh()
    ps = V.PhaseSpace(100, desc["qmin"], desc["qmax"], desc["qscale"],
                      desc["pmin"], desc["pmax"], desc["pscale"], data=mesh)
    ps.updateXProjection()
    ps.updateYProjection()
    fill, _ = ps.integrate()
    mx, _, rx = ps.variance(0)
    my, _, ry = ps.variance(1)
    np.testing.assert_array_equal(m["xproj"], proj)
    np.testing.assert_array_equal(m["yproj"], ps.getProjection(1)[0])
    assert (m["population"], m["position"], m["length"], m["average"],
            m["spread"]) == (np.float32(fill[0]), mx[0], rx[0], my[0], ry[0])
    assert len(st.history()[0]) == steps     # a history past 64 KiB
