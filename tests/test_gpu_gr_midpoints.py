"""The FP64 GR push where its midpoints' exp, sin and cos do not follow from the
particle's: on a coarse grid with a long step the midpoint of the coordinate
push lies up to a cell (0.3 rad) from the particle, on a fine one within the
series' range.  Tolerances are those of test_gpu_gr.py: the outputs are FP32
roundings of FP64 results that agree to a few units of 2^-53 times the
conditioning of ten fixed-point iterations."""
import numpy as np
import pytest

import test_gpu_gr as base

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric", ["ks", "qks", "qks_h"])
@pytest.mark.parametrize("massless", [False, True])
@pytest.mark.parametrize("n,dt", [((12, 10), 0.4), ((12, 10), 0.05), ((400, 300), 0.01)])
def test_midpoints_near_and_far(hip, oracle, monkeypatch, metric, massless, n, dt):
    monkeypatch.setattr(base, "N", n)
    em, em0 = base._fields(5, 0.01)
    p = base._particles(11, npart=1500, umax=0.3, near_axis=False)
    got = base._run_gpu(hip, metric, p, None if massless else em, None if massless else em0,
                        massless=massless, order=1, precision=64, dt=dt)
    ref = base._run_oracle(oracle, metric, p, None if massless else em,
                           None if massless else em0, massless=massless, order=1, prec="f64",
                           dt=dt)
    assert np.isfinite(ref["ux1"]).all()
    # positions: two float ulps of the largest code coordinate
    base._compare(got, ref, rtol=2e-6, xtol=2 * float(np.spacing(np.float32(max(n)))), inp=p)
