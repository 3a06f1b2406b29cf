"""Pairs that overflow next to the padding of a ragged last block: the
symmetric engine's padding particles sit at the set's last particle without
mass, and a real particle whose distance to it overflows 1/R^3 gets the
infinities of the tile engine (the same set against a copy of itself), not
NaN, in both particles' sums, with the other particle in another block or in
the last one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from test_gpu_symmetric import state, system  # noqa: E402


@pytest.mark.parametrize("soft", [0.0, 1e-6])
@pytest.mark.parametrize("kernel,mode,n", [
    ("Acc", "fp64", 2051), ("AccJerk", "fp64", 2051),
    ("AccJerk", "fp64", 9300), ("SnapCrackle", "fp64", 2051),
    ("Acc", "float", 4099), ("AccJerk", "float", 4099),
    ("AccJerk", "float", 9300), ("SnapCrackle", "float", 4099)])
@pytest.mark.parametrize("where", [5, -3])
def test_overflowing_pair_with_the_last_particle(kernel, mode, n, soft, where):
    from tupan_amd.lib import extensions
    print(kernel, mode, n, soft, where, flush=True)
    d = state(n, n, "uniform")
    flt = mode == "float"
    if flt:
        d = {k: v.astype(np.float32).astype(np.float64)
             for k, v in d.items()}
    d["eps2"][:] = soft
    last, i = n - 1, where % n
    for k in ("rx", "ry", "rz"):
        d[k][3] += 0.5  # away from the last particle
        d[k][last] = 0.0
        d[k][i] = 1e-14 if flt else 1e-110
    dtype = torch.float32 if flt else torch.float64
    ps, copy = system(d, dtype), system(d, dtype)
    ext = getattr(extensions, kernel)("HIP", "float32" if flt else "float64")
    got = [o.cpu().numpy().copy() for o in ext.calc(ps, ps)]
    ref = [o.cpu().numpy().copy() for o in ext.calc(ps, copy)]
    pair = np.array([i, last])
    rest = np.setdiff1d(np.arange(n), pair)
    for g, r in zip(got, ref):
        np.testing.assert_array_equal(np.isnan(g[pair]), np.isnan(r[pair]))
        if soft == 0.0:
            np.testing.assert_array_equal(g[pair], r[pair])
        assert np.isfinite(g[rest]).all() and np.isfinite(r[rest]).all()
    if soft == 0.0 and kernel != "SnapCrackle":
        assert all(np.isinf(g[pair]).all() for g in got[:3])
