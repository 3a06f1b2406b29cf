"""Near-pair lists of the symmetric far pass (a set against itself above 5120
particles) against the tile form (the same set against a copy of itself),
with slow cores whose entries hold more near pairs than a few: the same
pairs are listed, logged and solved from the learned guess; the list is
solved in windows when it is longer than one; and the graph-safe form takes
the tile form beyond the capacity where the symmetric lists would grow past
their bound."""
import os

import numpy as np
import pytest

from conftest import vec_rel_err

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

FIELDS = ("mass", "rx", "ry", "rz", "eps2", "vx", "vy", "vz")


def system(n, slow, seed=3):
    from tupan_amd.particles import ParticleSystem
    rng = np.random.default_rng(seed)
    d = {k: rng.standard_normal(n) for k in ("rx", "ry", "rz", "vx", "vy",
                                             "vz")}
    for k in ("vx", "vy", "vz"):
        d[k][slow] *= 1e-3
    d["mass"] = rng.uniform(0.5, 1.5, n) / n
    d["eps2"] = np.zeros(n)
    return ParticleSystem.from_numpy(d, device="cuda:0")


def call(ips, jps, flag=-1, path="two-pass", guess=None, log=None):
    from tupan_amd.learned import sakura_kernel
    ext = sakura_kernel(path=path, guess=guess)
    ext.kernel.counters = torch.zeros(5, dtype=torch.int64, device="cuda:0")
    if log is not None:
        ext.kernel.solve_log = log
    out = [o.cpu().numpy().copy() for o in ext.calc(ips, jps, 1.0 / 64, flag)]
    return out, ext.kernel.counters.cpu().tolist(), ext.kernel.near_pairs


def logged(log):
    f, t, it = log.valid()
    key = torch.cat([f, t[None, :]]).cpu().numpy()
    order = np.lexsort(key)
    return log.count, key[:, order], int(it.sum())


# 24 slow particles side by side: 24 near pairs in each one's own entry
@pytest.mark.parametrize("n,slow", [(5200, range(24)),
                                    (20600, range(4096, 4120)),
                                    (5200, range(0, 5200, 26))])
def test_guess_and_log_cover_the_tile_forms_pairs(n, slow):
    from tupan_amd.learned import KeplerNet, SolveLogBuffer
    import tupan_amd.learned as learned
    net = KeplerNet.load(os.path.join(os.path.dirname(learned.__file__),
                                      "kepler_net.npz"))
    ps = system(n, list(slow))
    got = []
    for jps in (ps, ps.copy()):
        log = SolveLogBuffer(1 << 20)
        out, cnt, near = call(ps, jps, guess=net, log=log)
        assert log.count == near
        got.append((out, cnt, near, logged(log)))
    (a, ca, na, la), (b, cb, nb, lb) = got
    assert na == nb > len(slow)**2
    assert ca == cb  # solves, Laguerre steps, subdivisions, far pairs, misses
    assert la[0] == lb[0] and la[2] == lb[2]
    np.testing.assert_array_equal(la[1], lb[1])
    assert vec_rel_err(a[:3], b[:3]) <= 1e-12
    assert vec_rel_err(a[3:], b[3:]) <= 1e-12


@pytest.mark.parametrize("n,slow,flag", [
    (5200, range(100), -1),       # more than 32 in an entry
    (5300, range(5200, 5300), 2),   # in the ragged last block
    (21000, range(500, 800), 1),
    (9001, range(9001), -1)])     # every pair near
@pytest.mark.parametrize("logging", [False, True])
def test_overfull_entries_equal_one_pass(n, slow, flag, logging):
    """Over-full entries solved whole (plain calls) or beyond their first 32
    (calls with a log, here longer than one window at n = 9001)."""
    from tupan_amd.learned import SolveLogBuffer
    print(n, flag, logging, flush=True)
    ps = system(n, list(slow))
    log = SolveLogBuffer(1 << (25 if n == 9001 else 20)) if logging else None
    a, ca, _ = call(ps, ps, flag, "one-pass")
    b, cb, near = call(ps, ps, flag, log=log)
    if n == 9001:
        assert near > 1 << 24
    if logging:
        assert log.count == near and bool((log.iterations[:near] >= 0).all())
        # a particle with itself takes no steps
        assert int((log.iterations[:near] == 0).sum()) <= n
    assert vec_rel_err(b[:3], a[:3]) <= 1e-12
    assert vec_rel_err(b[3:], a[3:]) <= 1e-12
    if flag in (-1, 1):
        assert ca[:4] == cb[:4]


def test_flag_zero_leaves_the_pairs():
    ps = system(5200, list(range(30)))
    out, cnt, near = call(ps, ps, 0)
    assert near == 0 and cnt[0] == 0
    assert all(np.all(o == 0) for o in out)


def test_graph_form_beyond_the_symmetric_list_bound():
    from tupan_amd import _native
    from tupan_amd.lib.hip_backend import current_stream_handle
    n = 5200
    ps = system(n, list(range(100)))
    ref, _, near = call(ps, ps)
    fields = _native.ptr_array([getattr(ps, f).data_ptr() for f in FIELDS])
    for cap in (near, (1 << 26) + 1):
        outs = [torch.zeros(n, dtype=torch.float64, device="cuda:0")
                for _ in range(6)]
        status = torch.zeros(1, dtype=torch.int32, device="cuda:0")
        _native.check(_native.lib().tupan_sakura_graph(
            n, fields, n, fields, 1.0 / 64, -1,
            _native.ptr_array([o.data_ptr() for o in outs]), cap, None,
            status.data_ptr(), current_stream_handle()),
            "tupan_sakura_graph")
        assert int(status.item()) == 0
        got = [o.cpu().numpy() for o in outs]
        if cap == near:
            assert all(np.array_equal(x, y) for x, y in zip(got, ref))
        assert vec_rel_err(got[:3], ref[:3]) <= 1e-12
        assert vec_rel_err(got[3:], ref[3:]) <= 1e-12
