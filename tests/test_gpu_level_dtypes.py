"""Bookkeeping arrays of other element types: a particle system made from
float step counters keeps them as floats (and integer times as integers), and
the native level operations, which write float64 and int64 words, leave such
arrays to the array operations: counters count, integer times are refused."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def system(n, **extra):
    from tupan_amd.particles import ParticleSystem
    rng = np.random.default_rng(5)
    d = {k: rng.standard_normal(n) for k in ("rx", "ry", "rz", "vx", "vy",
                                             "vz")}
    d["mass"] = rng.uniform(0.1, 2.0, n)**2 / n
    d["eps2"] = np.full(n, 1e-4)
    d.update(extra)
    ps = ParticleSystem.from_numpy(d, device="cuda:0")
    type(ps).t_curr = 0.0
    return ps


def step(ps, **kw):
    from tupan_amd.integrator import Integrator
    Integrator(2.0**-9, 0.0, ps, method="sia21h.dkd", **kw).evolve_step(1.0)
    order = torch.argsort(ps.id)
    return {k: getattr(ps, k)[order].cpu().numpy()
            for k in ("rx", "vz", "time", "nstep")}


@pytest.mark.parametrize("kw", [{}, {"device_subtree": False}])
def test_float_step_counters_count(kw):
    n = 300
    a = step(system(n), **kw)
    ps = system(n, nstep=np.zeros(n))
    assert ps.nstep.dtype == torch.float64
    b = step(ps, **kw)
    assert a["nstep"].min() >= 1
    np.testing.assert_array_equal(a["nstep"], b["nstep"])
    for k in ("rx", "vz", "time"):
        np.testing.assert_array_equal(a[k], b[k])


def test_integer_times_are_refused():
    n = 300
    ps = system(n, time=np.zeros(n, dtype=np.int64))
    assert ps.time.dtype == torch.int64
    with pytest.raises(RuntimeError):
        step(ps, device_subtree=False)


def test_update_takes_its_own_types_only():
    from tupan_amd.integrator.device_update import BOOK, device_update
    f = [torch.zeros(8, dtype=torch.float64, device="cuda:0")
         for _ in range(3)]
    i = torch.zeros(8, dtype=torch.int64, device="cuda:0")
    assert not device_update(BOOK, f, 0.5)
    assert not device_update(BOOK, (f[0], i, i), 0.5)
    assert device_update(BOOK, (f[0], f[1], i), 0.5)
    assert i.tolist() == [1] * 8 and f[1].tolist() == [0.5] * 8
