"""The FP64 GR push and the GR deposit where their shortcuts change over.

Push: the midpoints' exp, sin and cos follow from the particle's when they are
near; on a coarse grid with a long step the midpoint lies up to a cell (0.3
rad) away, on a fine one within the series' range.  Tolerances are those of
test_gpu_gr.py: the outputs are FP32 roundings of FP64 results that agree to a
few units of 2^-53 times the conditioning of ten fixed-point iterations."""
import numpy as np
import pytest

import test_gpu_gr as base
from _helpers import G

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


@pytest.mark.parametrize("metric", ["ks", "qks", "qks_h"])
@pytest.mark.parametrize("massless", [False, True])
@pytest.mark.parametrize("dt", [0.001, 0.02])
def test_midpoints_next_to_the_axis(hip, oracle, monkeypatch, metric, massless, dt):
    """A fine grid with an eighth of the particles in the cells next to the axis,
    whose midpoints lie closer to it than a quarter of their own distance or
    further: on both sides of that line (fields off, as in
    test_gr_axis_massive_zero_fields)."""
    n = (400, 300)
    monkeypatch.setattr(base, "N", n)
    em = np.zeros((6, n[1] + 2 * G, n[0] + 2 * G), np.float32)
    p = base._particles(12, npart=1500, umax=0.3, near_axis=True)
    got = base._run_gpu(hip, metric, p, em, em, massless=massless, order=1, precision=64, dt=dt)
    ref = base._run_oracle(oracle, metric, p, em, em, massless=massless, order=1, prec="f64",
                           dt=dt)
    base._compare(got, ref, rtol=2e-6, xtol=2 * float(np.spacing(np.float32(max(n)))), inp=p)


@pytest.mark.parametrize("kind", ["kerr_schild", "qkerr_schild", "kerr_schild_0"])
@pytest.mark.parametrize("n,npart", [((150, 24), 9001), ((70, 30), 5000), ((131, 9), 1)])
def test_gr_deposit_rows(hip, oracle, kind, n, npart):
    """Cell order on grids wider than the deposit's window: workgroups inside a
    row, at its end (the next row's particles are taken one array row further)
    and, with few particles per row, over several rows (direct adds).
    Tolerance as in test_gpu_gr_step.test_gr_deposit."""
    import torch

    import test_gpu_gr_step as step
    from entity_amd.containers import Particles
    from entity_amd.kernels import device_errors, gr
    prm, met, shape = step._setup(oracle, kind, n, a=0.9 if kind != "kerr_schild_0" else 0.0)
    h = step._gr_particles(np.random.default_rng(npart), n, npart)
    order = np.lexsort((h["i1"], h["i2"]))
    h = {k: v[order] for k, v in h.items()}
    h["tag"][:1] = 1
    sp = Particles(2, npart, device="cuda", with_phi=True)
    step._load(sp, h)
    J = torch.zeros(shape.tensor_shape(3), device="cuda")
    gr.DepositCurrents_kernel(J, shape, sp, met, -1.0, 0.37, 64)()
    torch.cuda.synchronize()
    assert device_errors() == 0
    ref = np.zeros((3, n[1] + 2 * G, n[0] + 2 * G))
    assert oracle.gr_deposit(prm, h, ref, charge=-1.0, dt=float(np.float32(0.37))) == 0
    step._close(J.cpu().numpy(), ref, "J", rtol=4e-6)


@pytest.mark.parametrize("kind", ["kerr_schild", "qkerr_schild", "kerr_schild_0"])
@pytest.mark.parametrize("precision", [32, 64])
def test_gr_deposit_infinite_momentum(hip, oracle, kind, precision):
    """An infinite u_theta makes no out-of-plane current (the energy is infinite
    and v^phi finite): J stays finite.  A NaN shows where its particle is."""
    import torch

    import test_gpu_gr_step as step
    from entity_amd.containers import Particles
    from entity_amd.kernels import device_errors, gr
    n = (70, 30)
    prm, met, shape = step._setup(oracle, kind, n, a=0.9 if kind != "kerr_schild_0" else 0.0)
    h = step._gr_particles(np.random.default_rng(5), n, 600)
    h["tag"][:] = 1
    h["ux2"][3], h["ux2"][77], h["ux1"][300] = np.inf, -np.inf, np.nan
    sp = Particles(2, 600, device="cuda", with_phi=True)
    step._load(sp, h)
    J = torch.zeros(shape.tensor_shape(3), device="cuda")
    gr.DepositCurrents_kernel(J, shape, sp, met, -1.0, 0.37, precision)()
    torch.cuda.synchronize()
    assert device_errors() == 0
    ref = np.zeros((3, n[1] + 2 * G, n[0] + 2 * G))
    assert oracle.gr_deposit(prm, h, ref, charge=-1.0, dt=float(np.float32(0.37))) == 0
    nan = np.isnan(ref)
    assert 0 < nan.sum() <= 9
    got = J.cpu().numpy()
    np.testing.assert_array_equal(np.isnan(got), nan)
    ok = ~nan
    # tolerances of test_gpu_gr_step.test_gr_deposit
    step._close(got[ok], ref[ok], "J", rtol=4e-6 if precision == 64 else 2e-5)
