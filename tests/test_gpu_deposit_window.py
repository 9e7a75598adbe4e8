"""ntt_deposit_currents against the FP64 oracle where its LDS window can go
wrong: particle counts around a workgroup's, particles in tile order, across
the periodic boundary, across rows of tiles, in no order, and weights over many
decades."""
import numpy as np
import pytest
import torch

from _helpers import G, field_array

pytestmark = pytest.mark.gpu

TILE = (8, 4, 4)


def _particles(dim, npart, layout, weights, seed):
    rng = np.random.default_rng(seed)
    n = (43, 30) if dim == 2 else (29, 18, 13)
    box = n if layout != "corner" else (8, 4, 4)[:dim]
    c = [rng.integers(0, box[d], npart) for d in range(dim)]
    if layout != "random":
        # tile order; "corner": every particle next to the box's lower corner,
        # so that the moves below it wrap to the other side
        key, mul = np.zeros(npart, np.int64), 1
        for d in range(dim):
            key += mul * (c[d] // TILE[d])
            mul *= -(-n[d] // TILE[d])
        order = np.argsort(key, kind="stable")
        c = [x[order] for x in c]
    p = {}
    for d in range(dim):
        x = rng.random(npart).astype(np.float32)
        x = np.minimum(x, np.float32(0.9999999))
        move = rng.uniform(-0.45, 0.45, npart).astype(np.float32)
        y = x + move
        step = (y >= 1).astype(np.int32) - (y < 0).astype(np.int32)
        y = np.clip(y - step, 0, 1).astype(np.float32)
        i = c[d].astype(np.int32) + step
        wrap = np.where(i < 0, n[d], np.where(i >= n[d], -n[d], 0)).astype(np.int32)
        p[f"i{d+1}"], p[f"dx{d+1}"] = i + wrap, y
        p[f"i{d+1}_prev"], p[f"dx{d+1}_prev"] = c[d].astype(np.int32) + wrap, x
    for d in range(3):
        p[f"ux{d+1}"] = rng.standard_normal(npart).astype(np.float32)
    w = np.ones(npart)
    if weights == "mixed":
        w = 10.0 ** rng.uniform(-6, 3, npart)
    elif weights == "zeros":
        w = (rng.random(npart) < 0.3).astype(float)
    elif weights == "tiny":
        w = np.where(rng.random(npart) < 0.5, 1e-33, 2e-33)
    p["weight"] = w.astype(np.float32)
    p["tag"] = np.where(rng.random(npart) < 0.05, 0, 1).astype(np.int16)
    return n, p


def _touched(p, dim, n):
    """Per cell, the weights of the live particles whose stencil may reach it."""
    S = np.zeros(field_array(dim, n, 1).shape[1:])
    live = p["tag"] == 1
    for off in np.ndindex(*(7,) * dim):
        at = [np.clip(p[f"i{d+1}"][live] + off[d] - 3 + G, 0, n[d] + 2 * G - 1)
              for d in range(dim)]
        np.add.at(S, tuple(reversed(at)), p["weight"][live].astype(float))
    return S


CASES = [(1, "tiles", "one"), (63, "tiles", "one"), (512, "tiles", "one"), (513, "tiles", "mixed"),
         (9000, "tiles", "one"), (9000, "tiles", "mixed"), (9000, "tiles", "zeros"),
         (9000, "tiles", "tiny"), (3000, "corner", "one"), (3000, "corner", "mixed"),
         (9000, "random", "one"), (2000, "random", "mixed")]


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("order", [0, 1, 2])
@pytest.mark.parametrize("npart,layout,weights", CASES)
def test_deposit_window(hip, oracle, dim, order, npart, layout, weights):
    """A slot's value is a product of single-precision shapes of at most 1, a
    few roundings of |q w| / dt each; the sums round once per workgroup that
    touches the cell.  16 units of 2^-24 of the weight in reach cover both."""
    from entity_amd.containers import GridShape, Particles
    from entity_amd.kernels import DepositCurrents_kernel, Minkowski, device_errors
    n, p = _particles(dim, npart, layout, weights, 7 * order + dim)
    dt = float(np.float32(0.35))
    shape = GridShape(dim, n)
    J = torch.zeros(shape.tensor_shape(3), device="cuda")
    prt = Particles(dim, npart).load(**p)
    DepositCurrents_kernel(J, shape, prt, Minkowski(dim), -1.0, dt, order)()
    torch.cuda.synchronize()
    assert device_errors() == 0
    ref = field_array(dim, n, 3, dtype=np.float64)
    assert oracle.deposit(p, ref, dim=dim, charge=-1.0, dt=dt, order=order, prec="f64") == 0
    tol = 16 * 2.0 ** -24 / dt * _touched(p, dim, n) + 1e-37
    err = np.abs(J.cpu().numpy().astype(np.float64) - ref)
    assert (err <= tol).all(), (err / tol).max()
    assert npart == 1 or np.abs(ref).max() > 0
