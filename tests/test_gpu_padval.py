"""The padding value of a de-dispersion: the running mean of the first DM
trial, every step rounded (update_stats), must come out to the last bit of
the plain recurrence also where its steps are run ahead and verified -- past
65536 samples, in several copies, for noise, a large offset, a constant and
a series that turns NaN."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
A = pytest.importorskip("presto_amd.accel")


@pytest.mark.parametrize("kind", ["noise", "offset", "constant", "nan"])
def test_padval_is_the_plain_recurrence(kind):
    B, numout = 4096, 300001
    nspec = (numout // B + 4) * B
    rng = np.random.Generator(np.random.PCG64(3))
    raw = rng.standard_normal((nspec, 4), dtype=np.float32)
    if kind == "offset":
        raw += 1000.0
    if kind == "constant":
        raw[:] = 0.1
    if kind == "nan":
        raw[200000] = np.nan
    p = A.dedisp_params(4, 64e-6, 1400.0, 1.0, B, 2, 1, 2, 0.0, 1.0, numout)
    out, n, pad = A.dedisperse(p, raw)
    assert n == numout
    avg = 0.0
    for i, x in enumerate(out[0].tolist()):
        avg += (x - avg) / (i + 1.0)
    assert pad == avg or (np.isnan(pad) and np.isnan(avg))
