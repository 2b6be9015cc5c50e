"""The direct wake's tables as the device makes them: the wake offsets and
CSR power of one step against numpy's FP64 transforms of the reference's
recipe, over short, long and odd transform lengths."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nmax", [(4, 8), (8, 510), (64, 128), (64, 130),
                                    (100, 768), (128, 8192), (260, 4098),
                                    (512, 1024)])
@pytest.mark.parametrize("use", ["wake", "csr", "both"])
def test_tables_match_numpy(n, nmax, use):
    import inovesa_amd as V
    from inovesa_amd.workloads import initial_mesh, kick_drift_config
    desc, d = kick_drift_config(n=n, steps_per_ts=500)
    rng = np.random.default_rng(n * nmax)
    z = (rng.random(nmax) + 1j * rng.standard_normal(nmax)).astype(np.complex64)
    imp = V.Impedance(nmax, 1e12, table=z)
    desc = dict(desc, use_wake=int(use != "csr"), use_csr=int(use != "wake"),
                fc=0.0)
    st = V.Step(desc, initial_mesh(n, seed=3), imp if use != "csr" else None,
                imp if use != "wake" else None)
    p = st.mesh()[1].astype(np.float64)
    st.record(1)
    st.run(1)
    M = nmax // 2
    F = np.fft.rfft(p, nmax)
    if use != "csr":
        W = F * z[:M + 1]
        W[M] = 0
        w = np.fft.irfft(W, nmax) * np.float32(desc["wakescaling"])
        # a float each (2^-24), and the scaling's own rounding
        assert np.abs(st.mesh()[2] - w[:n]).max() <= 2e-7 * np.abs(w).max()
    if use != "wake":
        q = np.float64(desc["qmax"] - desc["qmin"]) / (n - 1)
        df = 1.0 / q / (nmax - 1)
        ref = q * q * df * (z[:M + 1].real.astype(np.float64)
                            * np.abs(F) ** 2).sum()
        # the renormalisation and the frequency step are floats
        assert st.history()[0][0] == pytest.approx(ref, rel=1e-6)


@pytest.mark.parametrize("n,nmax", [(4, 8), (8, 510), (20, 42), (64, 128),
                                    (64, 130), (100, 768), (128, 8190),
                                    (128, 8192), (260, 4098), (512, 1024),
                                    (512, 514), (1024, 8192)])
@pytest.mark.parametrize("use", ["wake", "csr", "both"])
def test_device_tables_in_fp64(n, nmax, use):
    """The tables read back, against numpy's FP64 transforms and the host's
    sums (pinned at the same bound in test_toeplitz.py): an entry is a sum of
    up to M + 1 terms, each with its twiddle rounded once, whose errors stay
    below 1e-13 of the largest entry."""
    import inovesa_amd as V
    from inovesa_amd.workloads import initial_mesh, kick_drift_config
    desc, _ = kick_drift_config(n=n, steps_per_ts=4000)
    rng = np.random.default_rng(n + nmax)
    z = (rng.random(nmax) + 1j * rng.standard_normal(nmax)).astype(np.complex64)
    imp = V.Impedance(nmax, 1e12, table=z)
    wake, csr = use != "csr", use != "wake"
    desc = dict(desc, use_wake=int(wake), use_csr=int(csr), fc=0.0)
    st = V.Step(desc, initial_mesh(n, seed=3), imp if wake else None,
                imp if csr else None)
    g, h = st.toeplitz(wake, csr)
    M, d = nmax // 2, np.arange(-(n - 1), n)
    delta = (np.float32(desc["qmax"]) - np.float32(desc["qmin"])) / np.float32(n - 1)
    renorm = np.full(nmax, delta * delta, np.float32)
    fdelta = np.float32(1) / delta / np.float32(nmax - 1)
    if wake:
        w = z[:M + 1].astype(np.complex128)
        w[0], w[M] = w[0].real, 0
        ref = np.fft.irfft(w, nmax)[d % nmax] * nmax
        assert np.abs(g - ref).max() <= 1e-13 * np.abs(ref).max()
    if csr:
        c = np.float64(fdelta) * renorm[:M + 1] * z[:M + 1].real.astype(np.float64)
        c[1:M] /= 2
        ref = np.fft.irfft(c, nmax)[d % nmax] * nmax
        assert np.abs(h - ref).max() <= 1e-13 * np.abs(ref).max()
    if n <= nmax // 2:
        hg, hh = V.toeplitz_kernels(nmax, n, z if wake else None,
                                    z if csr else None, renorm, fdelta)
        for a, b in ((g, hg), (h, hh)):
            assert a is None or np.abs(a - b).max() <= 1e-13 * np.abs(b).max()


def test_missing_tables_are_refused():
    import inovesa_amd as V
    from inovesa_amd.workloads import (impedances, initial_mesh,
                                       kick_drift_config)
    desc, d = kick_drift_config(n=64, steps_per_ts=500)
    zw, zc = impedances(d)
    fft = V.Step(dict(desc, wake_method=1), initial_mesh(64, seed=1), zw, zc)
    with pytest.raises(V.VfpsInvalid):
        fft.toeplitz(True, False)
    with pytest.raises(V.VfpsInvalid):
        fft.toeplitz(False, True)
    only = V.Step(dict(desc, use_csr=0), initial_mesh(64, seed=1), zw)
    assert np.all(np.isfinite(only.toeplitz(True, False)[0]))
    with pytest.raises(V.VfpsInvalid):
        only.toeplitz()
