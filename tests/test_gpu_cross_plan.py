"""Few i against many j: launch plans with more than 64 j-splits (one per
whole tile) and chunk lengths picked to even out the workgroups per CU.
Sizes below one tile, at whole tiles, one particle past them, and past the
64-split limit; rows against the oracle (FP64 1e-13 of the row's vector,
split-FP32 8 x 2^-24 of the row's contribution magnitudes), ieee64 within
FP64 rounding (its splits change the sum order)."""
import numpy as np
import pytest

from conftest import vec_rel_err

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def state(n, seed):
    rng = np.random.default_rng(seed)
    d = {k: rng.standard_normal(n) for k in ("rx", "ry", "rz", "vx", "vy",
                                             "vz")}
    d["mass"] = rng.uniform(0.5, 1.5, n) / n
    d["eps2"] = np.full(n, 1e-6)
    return d


@pytest.mark.parametrize("mode", ["fp64", "split32", "ieee64"])
@pytest.mark.parametrize("ni,nj", [(1, 511), (3, 512), (65, 513),
                                   (30, 32768), (513, 33281), (2501, 60001),
                                   (1025, 131073)])
def test_rows_vs_oracle(ni, nj, mode):
    from oracle import Oracle
    from tupan_amd.lib import extensions
    from tupan_amd.particles import ParticleSystem
    print(ni, nj, mode, flush=True)
    di, dj = state(ni, 1), state(nj, 2)
    ips = ParticleSystem.from_numpy(di, device="cuda:0")
    jps = ParticleSystem.from_numpy(dj, device="cuda:0")
    out = extensions.Acc("HIP", "float64", mode=mode).calc(ips, jps)
    rows = np.unique([r for r in (0, 1, 63, 64, 511, 512, 1024, ni - 1)
                      if r < ni])
    got = [o.cpu().numpy()[rows] for o in out]
    i = {k: v[rows] for k, v in di.items()}
    ref = Oracle("float64").acc(i, dj)
    if mode != "split32":
        assert vec_rel_err(got, ref) <= 1e-13
        return
    r2 = sum((i[k][:, None] - dj[k][None, :])**2 for k in ("rx", "ry", "rz"))
    w = (dj["mass"] * np.sqrt(r2) / (r2 + 2e-6)**1.5).sum(1)
    err = np.sqrt(sum((g - r)**2 for g, r in zip(got, ref)))
    assert np.max(err / w) <= 8 * 2.0**-24


@pytest.mark.parametrize("mode", ["fp64", "split32", "ieee64"])
@pytest.mark.parametrize("ni,nj", [(1024, 32767), (1024, 32768),
                                   (300, 500001), (1025, 1048576),
                                   (1300, 1048577), (1024, 1048575)])
def test_bucket_edges_and_padded_rows_vs_oracle(ni, nj, mode):
    """Both sides of the table's pair-count lines (2^25, 2^30) and sets whose
    rows fill a quarter to nine tenths of the tuned shape's workgroup, which
    take the one-wave shape: same tolerances."""
    test_rows_vs_oracle(ni, nj, mode)
