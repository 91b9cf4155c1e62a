"""The device's hit sigmas (k_hit_sigmas): every candidate carries the sigma
that the host formula gives for its power, rounded to FP32 (the FP64 values
may differ in their last bits, so a neighbouring FP32 value is allowed), in
every branch of the formula -- up to 100 and 1200 in chi-squared, the
asymptotic forms above, log-probabilities below -600 -- and with fewer and
more hits than come back with the count (1023)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
A = pytest.importorskip("presto_amd.accel")


@pytest.mark.parametrize("numharm,amps", [
    (1, (5.0, 6.5, 20.0, 35.0, 80.0)),
    (16, (3.0, 6.0, 9.0, 30.0, 60.0)),
    (32, (3.0, 6.0, 9.0, 30.0, 60.0)),
])
def test_candidate_sigmas_equal_the_host_formula(numharm, amps):
    nbins = 1 << 16
    rng = np.random.Generator(np.random.PCG64(5))
    X = (rng.standard_normal(nbins) + 1j * rng.standard_normal(nbins)) / np.sqrt(2.0)
    for i, amp in enumerate(amps):
        r = 300 + 211 * i
        for h in range(1, numharm + 1):
            X[h * r] += amp
    p = A.make_params(nbins, 2 * nbins, 1e-3, zmax=20, numharm=numharm, sigma=1.0, rlo=100,
                      rhi=nbins - 1, dat_input=False)
    with A.Search(p) as s:
        s.set_spectrum(X.astype(np.complex64))
        s.run()
        cands, nhits, g = s.candidates(), len(s.hits()), s.geom
        assert len(cands) >= len(amps) and (numharm == 1 or nhits > 1023)
        for c in cands:
            st = int(c["numharm"]).bit_length() - 1
            want = np.float32(A.lib.accel_candidate_sigma(float(c["power"]), int(c["numharm"]),
                                                          float(g.numindep[st])))
            assert abs(c["sigma"] - want) <= np.spacing(want)
