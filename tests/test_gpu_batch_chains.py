"""Captured batch runs: every launch group advances as a chain of its own,
FFT-wake members keep the groups together.  Pinned by the single-mesh step,
bit for bit, over runs that end on either parity, follow one another and
reuse a captured run."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,fft_every,runs", [
    ((64,), 0, (1, 64, 3)),
    ((64, 128, 256, 512), 0, (65, 1, 63, 65)),
    ((128, 256, 384), 2, (33, 64, 33)),
])
def test_chains_equal_single_steps(sizes, fft_every, runs):
    import inovesa_amd as V
    from inovesa_amd.workloads import batched_scan_config, impedances
    inst = [(dict(desc, wake_method=1 if fft_every and k % fft_every == 0 else 2),
             init, *impedances(d)) for k, (desc, d, init) in
            enumerate(batched_scan_config(sizes=sizes, per_size=2, seed=9))]
    b = V.Batch(*[[i[k] for i in inst] for k in range(4)])
    assert (b.info()["launch_groups"] > 1) == (len(sizes) > 1)
    total = sum(runs)
    b.record(total)
    for r in runs:
        b.run(r)
    for k, (desc, init, zw, zc) in enumerate(inst):
        s = V.Step(desc, init, zw, zc)
        s.record(total)
        s.run(total)
        for x, y in zip(b.mesh(k), s.mesh()):
            assert np.array_equal(x, y), k
        assert np.array_equal(b.history(k)[0], s.history()[0]), k


def test_timing_is_the_time_of_a_run():
    """Batch.timing gives the step time that a run has (launch groups as
    chains), not that of steps joined one by one: over many groups these lie
    far apart, so the bound on wall-clock times can be wide.  It advances the
    state by as many steps."""
    import time

    import inovesa_amd as V
    from inovesa_amd.workloads import batched_scan_config, impedances
    sizes = (64, 96, 128, 160, 192, 256, 320, 384, 448, 512)
    inst = [(desc, init, *impedances(d)) for desc, d, init in
            batched_scan_config(sizes=sizes, per_size=1, seed=4)]
    a, b = (V.Batch(*[[i[k] for i in inst] for k in range(4)])
            for _ in range(2))
    groups = a.info()["launch_groups"]
    steps = 192
    a.run(steps)
    b.timing(steps)
    for k in range(len(inst)):
        assert np.array_equal(a.mesh(k)[0], b.mesh(k)[0]), k
    run, timing = [], []
    for _ in range(3):
        t0 = time.perf_counter()
        a.run(steps)
        run.append((time.perf_counter() - t0) / steps * 1e6)
        timing.append(b.timing(steps) * 1e3)
    print(f"{groups} groups: run {min(run):.1f}, timing {min(timing):.1f} us")
    assert min(timing) <= 1.5 * min(run)


@pytest.mark.parametrize("count,n,T", [(1, 32, 1), (1, 40, 8), (3, 24, 2),
                                       (7, 17, 4), (8, 8, 8), (9, 20, 16),
                                       (13, 36, 5)])
@pytest.mark.parametrize("persistent", [False, True])
def test_shares_of_the_block_map(count, n, T, persistent):
    """Tiles and closing workgroups dealt out over eight shares: fewer tiles
    than shares, equal and uneven shares, more closing workgroups than
    shares, padding; every instance as on its own."""
    import inovesa_amd as V
    from inovesa_amd.workloads import (impedances, initial_mesh,
                                       kick_drift_config)
    desc, d = kick_drift_config(n=n, steps_per_ts=4000)
    zw, zc = impedances(d)
    inits = [initial_mesh(n, seed=k) for k in range(count)]
    b = V.Batch([desc] * count, inits, [zw] * count, [zc] * count)
    b.retile_size(n, T, 128, persistent=persistent)
    b.record(5)
    b.run(5)
    for k in range(count):
        s = V.Step(desc, inits[k], zw, zc)
        s.record(5)
        s.run(5)
        for x, y in zip(b.mesh(k), s.mesh()):
            np.testing.assert_array_equal(x, y)
        np.testing.assert_array_equal(b.history(k)[0], s.history()[0])
