"""The x projection's sequential sums at row lengths with every kind of
remainder (16s, 4s, odd), in the per-map kernel, the one-mesh step and the
batch, bit for bit against a sequential float sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sequential(mesh, ws):
    acc = np.zeros(mesh.shape[:-1], np.float32)
    for y in range(mesh.shape[-1]):
        acc = acc + mesh[..., y] * ws[y]
    return acc


@pytest.mark.parametrize("n", [3, 5, 15, 16, 17, 63, 64, 68, 250, 252, 257,
                               300, 516])
@pytest.mark.parametrize("nb", [1, 3])
def test_phase_space_projection(n, nb):
    import inovesa_amd as V
    rng = np.random.default_rng(n)
    m = rng.standard_normal((nb, n, n)).astype(np.float32)
    ps = V.PhaseSpace(n, -6.0, 6.0, 1e-3, -6.0, 6.0, 1e6,
                      filling=[1.0 / nb] * nb, data=m)
    ps.updateXProjection()
    np.testing.assert_array_equal(ps.getProjection(0),
                                  _sequential(m, ps.simpsonWeights()))


@pytest.mark.parametrize("n", [4, 16, 36, 60, 64, 68, 100, 124, 128, 188, 260,
                               388])
def test_step_and_batch_projection(n):
    import inovesa_amd as V
    from inovesa_amd.workloads import (impedances, initial_mesh,
                                       kick_drift_config, simpson_weights)
    desc, d = kick_drift_config(n=n, steps_per_ts=500)
    zw, zc = impedances(d)
    init = initial_mesh(n, seed=n)
    ws = simpson_weights(n, np.float32(12.0) / np.float32(n - 1))
    st = V.Step(desc, init, zw, zc)
    st.run(2)
    mesh, proj, _ = st.mesh()
    np.testing.assert_array_equal(proj, _sequential(mesh, ws))
    b = V.Batch([desc], [init], [zw], [zc])
    b.run(2)
    bm, bp, _ = b.mesh(0)
    np.testing.assert_array_equal(bm, mesh)
    np.testing.assert_array_equal(bp, proj)


@pytest.mark.parametrize("n", [8180, 13641, 40956])
def test_longest_rows(n):
    """Rows that fill a workgroup's LDS: several to one, and the longest row
    that leaves no room beside it (6.7 GB of mesh)."""
    import inovesa_amd as V
    ps = V.PhaseSpace(n, -6.0, 6.0, 1e-3, -6.0, 6.0, 1e6)
    ps.updateXProjection()
    proj, ws, mesh = ps.getProjection(0)[0], ps.simpsonWeights(), ps.getData()[0]
    for r in (0, 1, n // 2 - 1, n // 2, n - 2, n - 1):
        seq = np.add.accumulate(np.append(np.float32(0), mesh[r] * ws),
                                dtype=np.float32)
        assert proj[r] == seq[-1], r
    assert proj[n // 2] > 0


def test_a_row_beyond_the_lds_is_refused():
    import inovesa_amd as V
    with pytest.raises(V.VfpsInvalid):
        V.PhaseSpace(40961, -6.0, 6.0, 1e-3, -6.0, 6.0, 1e6)


@pytest.mark.parametrize("n", [5, 7, 8, 9, 15, 17, 23, 24, 66, 129, 250, 268])
@pytest.mark.parametrize("wake", [1, 2])
def test_step_and_batch_projection_in_words(n, wake):
    """Lengths with every remainder of the eight words a turn, and of the 16
    and 64 values a turn, in each wake form and with one, two and four columns
    a thread."""
    import inovesa_amd as V
    from inovesa_amd.workloads import (impedances, initial_mesh,
                                       kick_drift_config, simpson_weights)
    desc, d = kick_drift_config(n=n, steps_per_ts=2000)
    desc = dict(desc, wake_method=wake)
    zw, zc = impedances(d)
    init = initial_mesh(n, seed=n)
    ws = simpson_weights(n, np.float32(12.0) / np.float32(n - 1))
    st = V.Step(desc, init, zw, zc)
    st.run(2)
    mesh, proj, _ = st.mesh()
    np.testing.assert_array_equal(proj, _sequential(mesh, ws))
    for threads in (64, 128, 512):
        if threads * 4 < n:
            continue
        b = V.Batch([dict(desc, tile_rows=2, threads=threads)], [init], [zw], [zc])
        b.run(2)
        bm, bp, _ = b.mesh(0)
        np.testing.assert_array_equal(bm, mesh)
        np.testing.assert_array_equal(bp, proj)
