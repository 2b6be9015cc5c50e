"""Results of all instances of a batch in one transfer: in one part, in
several, and histories longer than the staging buffer, with direct- and
FFT-wake instances of uneven sizes side by side."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def batch():
    import inovesa_amd as V
    from inovesa_amd.workloads import impedances, initial_mesh, kick_drift_config
    descs, inits, zs = [], [], []
    for k, (n, wake) in enumerate(((64, 2), (36, 1), (100, 2))):
        desc, d = kick_drift_config(n=n, steps_per_ts=500)
        descs.append(dict(desc, wake_method=wake))
        inits.append(initial_mesh(n, seed=k))
        zs.append(impedances(d))
    return V.Batch(descs, inits, [z[0] for z in zs], [z[1] for z in zs])


@pytest.mark.parametrize("cap,first,count", [
    (70, 0, 70), (70, 13, 57), (70, 69, 1),
    (600000, 0, 600000),      # 7.2 MB: an instance at a time
    (1100000, 5, 1099995)])   # 4.4 MB each: past the buffer
def test_histories_and_profiles(batch, cap, first, count):
    batch.record(cap)
    batch.run(67)
    got = batch.csr_histories(first, count)
    profs = batch.projections()
    for i in range(3):
        csr, _ = batch.history(i)
        full = np.zeros(cap, np.float32)
        full[:len(csr)] = csr
        assert len(csr) == 67 and np.all(csr > 0)
        np.testing.assert_array_equal(got[i], full[first:first + count])
        np.testing.assert_array_equal(profs[i], batch.mesh(i)[1])


def test_out_of_the_recorded_range_is_refused(batch):
    import inovesa_amd as V
    batch.record(8)
    for first, count in ((0, 9), (8, 1), (0xFFFFFFFF, 2)):
        with pytest.raises(V.VfpsInvalid):
            batch.csr_histories(first, count)
    assert batch.csr_histories(8, 0).shape == (3, 0)
