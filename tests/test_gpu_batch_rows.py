"""The wake and CSR dot products of a batch's tiles, whose rows are dealt out
over the wavefronts.  Pinned by the single-mesh step: a row's sum has the same
order there, so the meshes and the CSR powers are equal bit for bit, wherever
the rows of a tile end and however many wavefronts share them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme", ["kick_drift", "rotation"])
@pytest.mark.parametrize("tile,threads", [(1, 512), (1, 128), (3, 256), (5, 128),
                                          (7, 256)])
def test_rows_per_wavefront_equal_single_steps(scheme, tile, threads):
    import inovesa_amd as V
    from inovesa_amd.workloads import batched_scan_config, impedances
    inst = [(desc, init, *impedances(d)) for desc, d, init in
            batched_scan_config(sizes=(64, 128), per_size=1, seed=5,
                                scheme=scheme)]
    b = V.Batch(*[[i[k] for i in inst] for k in range(4)])
    for k in range(len(inst)):
        b.retile(k, tile, threads)
    b.record(8)
    b.run(5)
    for k, (desc, init, zw, zc) in enumerate(inst):
        s = V.Step(dict(desc, wake_method=2), init, zw, zc)
        s.record(8)
        s.run(5)
        for x, y in zip(b.mesh(k), s.mesh()):
            assert np.array_equal(x, y), k
        assert np.array_equal(b.history(k)[0], s.history()[0]), k
