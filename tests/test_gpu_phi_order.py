"""Initial conditions are scaled with the FP64 potential of a set against
itself, so its sums keep one order up to 32768 particles: shape 5 (one-wave
workgroups) with j-splits for four workgroups per CU below 2^22 pairs and for
sixteen below 2^30, then shape 1."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("n,shape,wg", [
    (1449, 5, 4), (1500, 5, 4), (2047, 5, 4), (2048, 5, 16), (2500, 5, 16),
    (6000, 5, 16), (32767, 5, 16), (32768, 1, 16)])
def test_self_potential_keeps_its_order(n, shape, wg):
    from tupan_amd import _native, tune
    from tupan_amd.lib import extensions
    from tupan_amd.particles import ParticleSystem
    rng = np.random.default_rng(n)
    d = {k: rng.standard_normal(n) for k in ("rx", "ry", "rz")}
    d["mass"] = rng.uniform(0.5, 1.5, n) / n
    d["eps2"] = np.zeros(n)
    ps = ParticleSystem.from_numpy(d, device="cuda:0")
    ext = extensions.Phi("HIP", "float64", mode="fp64")
    got = ext.calc(ps, ps)[0].clone()
    lib = _native.lib()
    kid, slot = tune.KERNEL_IDS["phi"], tune.SLOTS["fp64"]
    saved = []
    for b in range(3):
        s, w = ctypes.c_int(), ctypes.c_int()
        lib.tupan_tune_get(kid, slot, b, ctypes.byref(s), ctypes.byref(w))
        saved.append((s.value, w.value))
    try:
        for b in range(3):
            _native.check(lib.tupan_tune_set(kid, slot, b, shape, wg),
                          "tupan_tune_set")
        ref = ext.calc(ps, ps)[0].clone()
    finally:
        for b, e in enumerate(saved):
            lib.tupan_tune_set(kid, slot, b, *e)
    assert torch.equal(got.view(torch.int64), ref.view(torch.int64))
