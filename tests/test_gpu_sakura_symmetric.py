"""The symmetric far pass of the two-pass Sakura form (sakura.hip) against the
one-pass form: the first size it takes (5121), a ragged and a whole last
block, both particle-per-lane counts (20480 | 20481), odd and even block
counts; states whose slow core makes entries outgrow their near-pair lists.
The pairs' drifts are the one-pass arithmetic and the counters the same; dr
and dv of a particle differ by the order of its sum: 1e-12 of its vector."""
import numpy as np
import pytest

from conftest import vec_rel_err

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def system(n, seed, slow):
    from tupan_amd.particles import ParticleSystem
    rng = np.random.default_rng(seed)
    d = {k: rng.standard_normal(n) for k in ("rx", "ry", "rz", "vx", "vy",
                                             "vz")}
    # the first `slow` particles move slowly: all their mutual pairs are near
    for k in ("vx", "vy", "vz"):
        d[k][:slow] *= 1e-3
    d["mass"] = rng.uniform(0.5, 1.5, n) / n
    d["eps2"] = np.zeros(n)
    return ParticleSystem.from_numpy(d, device="cuda:0")


def run(ps, flag, path):
    from tupan_amd.lib import extensions
    ext = extensions.Sakura("HIP", "float64", path=path)
    ext.kernel.counters = torch.zeros(5, dtype=torch.int64, device="cuda:0")
    out = ext.calc(ps, ps, 1.0 / 64, flag)
    torch.cuda.synchronize()
    return ([o.cpu().numpy().copy() for o in out],
            ext.kernel.counters.cpu().tolist()[:4])


@pytest.mark.parametrize("n,slow,flag", [
    (n, slow, flag) for n, slow in ((5121, 0), (5121, 700), (5376, 100),
                                    (20480, 300), (20481, 300))
    for flag in (-1, 1, 2, -2)] + [(5503, 5503, -1)])  # the last: all near
def test_equals_one_pass(n, slow, flag):
    print(n, slow, flag, flush=True)
    ps = system(n, n + slow, slow)
    a, ca = run(ps, flag, "one-pass")
    b, cb = run(ps, flag, "two-pass")
    assert vec_rel_err(b[:3], a[:3]) <= 1e-12
    assert vec_rel_err(b[3:], a[3:]) <= 1e-12
    if flag in (-1, 1):
        assert ca == cb
    again, _ = run(ps, flag, "two-pass")
    assert all(np.array_equal(x, y) for x, y in zip(b, again))
