"""The field's transforms whose length is no power of two (direct sums, from
178 on a chirp DFT): primes, the smallest and largest lengths, either side of
a doubling of the inner transform and of the direct sums' longest, several
bunches, and mixed with power-of-two lengths in one batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def V():
    import inovesa_amd as V
    return V


def _field(V, n, nb, nmax, seed):
    rng = np.random.default_rng(seed)
    ps = V.PhaseSpace(n, -6.0, 6.0, 1e-3, -6.0, 6.0, 1e6,
                      filling=[1.0 / nb] * nb)
    z = (rng.standard_normal(nmax) + 1j * rng.standard_normal(nmax)).astype(
        np.complex64)
    spacing = n if nb == 1 else (nmax - n) // (nb - 1)
    f = V.ElectricField(ps, V.Impedance(nmax, 1e12, table=z), range(nb),
                        spacing, 1.0, 1.0, 1.0)
    prof = rng.random((nb, n)).astype(np.float32)
    ps.setProjection(0, prof)
    return ps, f, z, prof, spacing


@pytest.mark.parametrize("nmax,n,nb", [
    (6, 3, 1), (10, 4, 2), (14, 7, 1), (62, 5, 3), (66, 33, 1), (254, 100, 2),
    (258, 60, 4), (1022, 200, 3), (1026, 512, 1), (3000, 250, 3),
    (4094, 300, 4), (4098, 512, 5), (4802, 333, 2), (8186, 512, 6),
    (8190, 128, 9)])
def test_chirp_lengths_match_numpy(V, nmax, n, nb):
    """Against numpy's FP64 transforms of the reference's recipe.  The
    result is a float (2^-24 of each bin, which the random impedance spreads
    evenly), as are the spectrum and its product with Z: 1e-6 of the rms."""
    ps, f, z, prof, spacing = _field(V, n, nb, nmax, nmax)
    M = nmax // 2
    pad = np.zeros(nmax)
    for b in range(nb):
        pad[b * spacing:b * spacing + n] = prof[b]
    W = np.fft.rfft(pad) * z[:M + 1]
    W[M] = 0
    w = np.fft.irfft(W, nmax)
    got = f.wakePotential()
    ref = np.stack([w[b * spacing:b * spacing + n] for b in range(nb)])
    rms = np.sqrt((w ** 2).mean())
    assert np.abs(got - ref).max() <= 3e-6 * rms
    power, spec = f.updateCSR(np.float32(0))
    F = np.abs(np.fft.rfft(prof, nmax)) ** 2
    d = float(ps.getDelta(0))
    s = d * d * z[:M + 1].real.astype(np.float64) * F
    assert np.abs(spec[:, :M + 1] - s).max() <= 2e-6 * np.abs(s).max()
    assert not spec[:, M + 1:].any()


def test_batch_of_mixed_lengths(V):
    """FFT-wake instances of a power-of-two and a longer-in-LDS odd length in
    one field launch, each equal to its single-mesh run bit for bit."""
    from inovesa_amd.workloads import impedances, initial_mesh, kick_drift_config
    descs, inits, zs = [], [], []
    for n, pad in ((64, 16.0), (64, 11.7), (68, 21.3)):
        desc, d = kick_drift_config(n=n, steps_per_ts=500, padding=pad)
        nmax = int(n * pad) // 2 * 2
        d = dict(d, padded_bins=nmax)
        descs.append(dict(desc, wake_method=1))
        inits.append(initial_mesh(n, seed=n))
        zs.append(impedances(d))
    b = V.Batch(descs, inits, [z[0] for z in zs], [z[1] for z in zs])
    b.run(9)
    for i in range(3):
        st = V.Step(descs[i], inits[i], *zs[i])
        st.run(9)
        for x, y in zip(b.mesh(i), st.mesh()):
            np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("nmax,n,nb", [(202, 90, 2), (346, 100, 3),
                                       (352, 176, 2), (354, 120, 2),
                                       (356, 100, 3), (358, 333, 1)])
def test_either_side_of_the_direct_sums(V, nmax, n, nb):
    test_chirp_lengths_match_numpy(V, nmax, n, nb)


@pytest.mark.parametrize("nmax", [250, 352, 354, 1000])
def test_fft_step_beside_a_batch(V, nmax):
    """A step with its own transform kernel and the batch's shared one."""
    from inovesa_amd.workloads import initial_mesh, kick_drift_config
    rng = np.random.default_rng(nmax)
    z = V.Impedance(nmax, 1e12, table=(1e-3 * rng.random(nmax)).astype(
        np.complex64))
    desc, _ = kick_drift_config(n=64, steps_per_ts=4000)
    desc = dict(desc, wake_method=1)
    init = initial_mesh(64, seed=1)
    st = V.Step(desc, init, z, z)
    st.record(3)
    st.run(3)
    b = V.Batch([desc] * 2, [init] * 2, [z] * 2, [z] * 2)
    b.record(3)
    b.run(3)
    for x, y in zip(b.mesh(1), st.mesh()):
        np.testing.assert_array_equal(x, y)
    np.testing.assert_array_equal(b.history(1)[0], st.history()[0])
