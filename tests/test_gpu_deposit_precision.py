"""What ntt_deposit_currents keeps of each contribution: particles much lighter
than their neighbours, a cold plasma's out-of-plane current, particles next to
a node that are added to J directly, and momenta that are not finite."""
import numpy as np
import pytest
import torch

from _helpers import G, field_array

pytestmark = pytest.mark.gpu

DT = float(np.float32(0.35))


def _deposit(p, dim, n, order):
    from entity_amd.containers import GridShape, Particles
    from entity_amd.kernels import DepositCurrents_kernel, Minkowski, device_errors
    shape = GridShape(dim, n)
    J = torch.zeros(shape.tensor_shape(3), device="cuda")
    prt = Particles(dim, len(p["tag"])).load(**p)
    DepositCurrents_kernel(J, shape, prt, Minkowski(dim), -1.0, DT, order)()
    torch.cuda.synchronize()
    assert device_errors() == 0
    return J.cpu().numpy().astype(np.float64)


def _oracle(oracle, p, dim, n, order, prec):
    """The oracle's J, in FP64 with the single-precision builds' constant
    0.333333 for a third where the scheme uses it."""
    J = field_array(dim, n, 3, dtype=np.float32 if prec == "f32" else np.float64)
    assert oracle.deposit(p, J, dim=dim, charge=-1.0, dt=DT, order=order, prec=prec) == 0
    J = J.astype(np.float64)
    if prec == "f64" and order > 0:
        J[0 if dim == 3 else 2:] *= 3 * float(np.float32(0.333333))
    return J


def _tile_particles(dim, npart, seed, umax):
    """Particles of one 8 x 4 x 4 tile, moved by less than half a cell."""
    rng = np.random.default_rng(seed)
    p = {}
    for d in range(dim):
        c = 8 + rng.integers(0, (8, 4, 4)[d], npart)
        x = rng.random(npart).astype(np.float32) * np.float32(0.999)
        y = x + rng.uniform(-0.45, 0.45, npart).astype(np.float32)
        step = (y >= 1).astype(np.int32) - (y < 0).astype(np.int32)
        p[f"i{d+1}"] = (c + step).astype(np.int32)
        p[f"dx{d+1}"] = np.clip(y - step, 0, 1).astype(np.float32)
        p[f"i{d+1}_prev"], p[f"dx{d+1}_prev"] = c.astype(np.int32), x
    for d in range(3):
        p[f"ux{d+1}"] = (umax * rng.standard_normal(npart)).astype(np.float32)
    p["weight"] = np.ones(npart, np.float32)
    p["tag"] = np.ones(npart, np.int16)
    return p


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("order", [0, 1, 2])
@pytest.mark.parametrize("light", [1.0 / 15, 1e-4])
def test_light_and_cold(hip, oracle, dim, order, light):
    """Light particles share their workgroups with heavy ones, and the plasma is
    cold (|u| of 1e-4).  Per component, over the cells that only light particles
    reach and over the others, the error against 64 bits is at most twice that
    of the same sums in FP32 throughout: a contribution takes the same few
    roundings in both, and the window's sum fewer than the FP32 oracle's."""
    n = (26, 18) if dim == 2 else (26, 18, 17)
    p = _tile_particles(dim, 1500, 3 * order + dim, 1e-4)
    p["weight"][p["i1_prev"] >= 11] = light
    ref = _oracle(oracle, p, dim, n, order, "f64")
    f32 = np.abs(_oracle(oracle, p, dim, n, order, "f32") - ref)
    err = np.abs(_deposit(p, dim, n, order) - ref)
    # magnitudes that meet in each entry
    A = {True: np.zeros_like(ref), False: np.zeros_like(ref)}
    for k in range(len(p["tag"])):
        q = {name: v[k:k + 1] for name, v in p.items()}
        A[bool(p["weight"][k] < 1)] += np.abs(_oracle(oracle, q, dim, n, order, "f64"))
    for mask in ((A[False] == 0) & (A[True] > 0), A[False] > 0):
        for c in range(3):
            m = mask[c]
            S = (A[True] + A[False])[c][m].sum()
            assert m.sum() > 20
            assert err[c][m].sum() <= 2 * f32[c][m].sum(), (c, err[c][m].sum() / S,
                                                            f32[c][m].sum() / S)


@pytest.mark.parametrize("order", [0, 1, 2])
def test_nonfinite_momenta_2d(hip, oracle, order):
    """A momentum that is not a number shows in the out-of-plane current of
    exactly the cells its particle touches; an infinite one along the plane
    makes none."""
    n = (26, 18)
    p = _tile_particles(2, 400, 11 + order, 0.5)
    p["ux1"][17], p["ux2"][200], p["ux3"][399] = np.nan, np.inf, np.nan
    got = _deposit(p, 2, n, order)
    ref = _oracle(oracle, p, 2, n, order, "f64")
    nan = np.isnan(ref)
    assert nan[2].any() and not nan[:2].any()
    np.testing.assert_array_equal(np.isnan(got), nan)
    # 400 contributions of at most 1/dt, a few roundings each
    tol = 16 * 2.0 ** -24 / DT * 400
    assert np.abs(got - ref)[~nan].max() <= tol


@pytest.mark.parametrize("order", [1, 2])
def test_direct_near_nodes_3d(hip, oracle, order):
    """Particles too far apart for a window, moving along x, next to a node (order
    1) or to the middle of their cell (order 2) along y and z, where one weight
    is tiny: it keeps its relative accuracy, so every slot of J1 does.  The
    longitudinal factor (a difference of shapes that move by 0.4 of a cell)
    takes under 8 roundings of its value, each transverse product 3 (all of one
    sign)."""
    n = (60, 55, 50)
    k = np.arange(30)
    p = {}
    for d in range(3):
        c = ((7 * k, 11 * k, 13 * k)[d] % (n[d] - 8) + 4).astype(np.int32)
        p[f"i{d+1}"], p[f"i{d+1}_prev"] = c, c.copy()
    tiny = np.float32(10.0) ** np.linspace(-6.5, -3, 30).astype(np.float32)
    at = np.float32(0.5 if order == 2 else 0.0)
    p["dx1_prev"] = np.full(30, 0.55, np.float32)
    p["dx1"] = np.full(30, 0.95, np.float32)
    for d in (2, 3):
        sign = -1 if order == 2 else 1
        p[f"dx{d}_prev"] = (at + sign * tiny).astype(np.float32)
        p[f"dx{d}"] = (at + sign * 3 * tiny).astype(np.float32)
    for d in range(3):
        p[f"ux{d+1}"] = np.zeros(30, np.float32)
    p["weight"] = np.ones(30, np.float32)
    p["tag"] = np.ones(30, np.int16)
    got, ref = _deposit(p, 3, n, order)[0], _oracle(oracle, p, 3, n, order, "f64")[0]
    m = np.abs(ref) > 1e-30
    assert m.sum() >= 30 * 4
    assert (np.abs(got - ref)[m] <= 16 * 2.0 ** -24 * np.abs(ref)[m]).all(), \
        (np.abs(got - ref)[m] / np.abs(ref)[m]).max()
