"""The current after 0 to 3 filter passes: the passes alternate between cur and
buff and end in cur, the first one of a 2D step reads the fixed-point
accumulator, and several species share a launch."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(37, 26), (19, 11, 14)])
@pytest.mark.parametrize("nfilters", [0, 1, 2, 3])
@pytest.mark.parametrize("nspecies", [1, 3, 9])
def test_step_current(hip, oracle, n, nfilters, nspecies):
    """One step against the oracle's (strict build), J and E within 4e-6 of
    their largest value as in test_gpu_engine.py; and the batched step's
    fields bit for bit."""
    from entity_amd import _abi
    from entity_amd.engine import SRParams, SpeciesSpec, SRPICEngine
    from entity_amd.ensemble import SREnsemble
    from entity_amd.kernels import device_errors
    dim = len(n)
    rng = np.random.default_rng(nfilters)

    def box(strict):
        prm = SRParams(dim=dim, n=n, shape_order=1, n_filters=nfilters, ppc0=4.0, larmor0=0.5,
                       skindepth0=2.0)
        sp = [SpeciesSpec(f"s{k}", 1.0 + k, (-1.0) ** k,
                          _abi.PUSHER_VAY if k == 2 else _abi.PUSHER_BORIS)
              for k in range(nspecies)]
        return SRPICEngine(prm, sp, 700, strict=strict)

    parts = []
    for _ in range(nspecies):
        p = {"tag": np.ones(700, np.int16)}
        for d in range(dim):
            p[f"i{d+1}"] = rng.integers(0, n[d], 700).astype(np.int32)
            p[f"dx{d+1}"] = rng.random(700, dtype=np.float32)
        for d in range(3):
            p[f"ux{d+1}"] = rng.standard_normal(700).astype(np.float32)
        parts.append(p)
    em = (0.1 * rng.standard_normal((6,) + tuple(m + 4 for m in reversed(n)))).astype(np.float32)
    oracle.communicate(em, 0, 6, dim=dim)
    eng = {}
    for strict in (True, False):
        eng[strict] = box(strict)
        for s, p in zip(eng[strict].species, parts):
            s.load(**p)
        eng[strict].fields.em.copy_(torch.from_numpy(em))
    e = eng[True]
    sp = [{"p": oracle.normalize_particles(s.to_host(), "f32"), "mass": s.mass,
           "charge": s.charge, "pusher": s.pusher} for s in e.species]
    p = e.params
    prm = dict(dt=p.dt, correction=p.correction, omegaB0=p.omegaB0, q0=p.q0, B0=p.B0, V0=p.V0,
               ppc0=p.ppc0, dx=p.dx, shape_order=1, n_filters=nfilters, fieldsolver_enable=1,
               deposit_enable=1, step=0)
    ref_em, ref_cur = em.copy(), np.zeros((3,) + em.shape[1:], np.float32)
    assert oracle.sr_step(ref_em, ref_cur, np.zeros_like(ref_cur), sp, dim=dim, prm=prm,
                          bc=((1, 1),) * 3) == 0
    e.step_forward()
    for got, ref in ((e.fields.cur, ref_cur), (e.fields.em, ref_em)):
        np.testing.assert_allclose(got.cpu().numpy(), ref, rtol=0, atol=4e-6 * np.abs(ref).max())
    # the product build: alone and batched
    a, b = eng[False], box(False)
    for s, q in zip(b.species, parts):
        s.load(**q)
    b.fields.em.copy_(torch.from_numpy(em))
    a.step_forward()
    SREnsemble([b]).step_forward()
    torch.cuda.synchronize()
    assert torch.equal(a.fields.em, b.fields.em) and torch.equal(a.fields.cur, b.fields.cur)
    assert device_errors() == 0 and device_errors(True) == 0
