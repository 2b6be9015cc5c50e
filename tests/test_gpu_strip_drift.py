"""The strip form's drift: tiles of four rows read windows of their own size,
from one row for the whole wavefront where its columns agree.  Pinned by the
single-mesh step bit for bit, with full tiles of four rows, other heights, and
a height whose last tile has four rows (64 = 12 x 5 + 4)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile,strip,threads", [(4, 8, 256), (5, 4, 64),
                                                (3, 8, 128)])
def test_strip_drift_equals_single_steps(tile, strip, threads):
    import inovesa_amd as V
    from inovesa_amd.workloads import batched_scan_config, impedances
    inst = [(desc, init, *impedances(d)) for desc, d, init in
            batched_scan_config(sizes=(64, 100, 260), per_size=1, seed=7)
            if desc["n"] <= 4 * threads]
    b = V.Batch(*[[i[k] for i in inst] for k in range(4)])
    for k in range(len(inst)):
        b.retile(k, tile, threads, strip=strip)
    b.record(10)
    b.run(7)
    for k, (desc, init, zw, zc) in enumerate(inst):
        s = V.Step(dict(desc, wake_method=2), init, zw, zc)
        s.record(10)
        s.run(7)
        for x, y in zip(b.mesh(k), s.mesh()):
            assert np.array_equal(x, y), k
        assert np.array_equal(b.history(k)[0], s.history()[0]), k
