"""The symmetric engine's four-particles-per-lane form in FP32 arithmetic,
whose j sums change lanes four times per 64 particles (sym.h: sym_pass): on
both sides of its bound (131072 | 131073, the latter with a last block of one
particle) and past it with a ragged block, every FP32 kernel; and a set whose
partial sums pass the engine's limit, which the tile engine takes.  States,
rows and bars as in test_gpu_symmetric.py."""
import numpy as np
import pytest

from conftest import vec_rel_err

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

from test_gpu_symmetric import (oracle_rows, rows_of, run, state,  # noqa: E402
                                system)


def acc_bar(d, rows, got, ref):
    """Error of the accelerations over the sum of their contributions'
    magnitudes."""
    dr = [d[k][rows][:, None] - d[k][None, :] for k in ("rx", "ry", "rz")]
    r2 = sum(x * x for x in dr)
    R2 = r2 + d["eps2"][rows][:, None] + d["eps2"][None, :]
    w = np.where(r2 > 0, d["mass"] * np.sqrt(r2)
                 / np.where(r2 > 0, R2, 1.0)**1.5, 0.0).sum(1)
    err = np.sqrt(sum((g - r)**2 for g, r in zip(got[:3], ref[:3])))
    return np.max(err / w)


KERNELS = ([(k, "split32") for k in ("acc", "acc_jerk", "tstep")]
           + [(k, "float") for k in ("acc", "acc_jerk", "tstep",
                                     "snap_crackle", "phi")])


@pytest.mark.parametrize("kernel,mode,n", [
    (k, m, n) for k, m in KERNELS for n in (131072, 131073, 133800)
    if n == 131073 or k in ("acc_jerk", "tstep")])
def test_four_per_lane_fp32(kernel, mode, n):
    print(kernel, mode, n, flush=True)
    d = state(n, n, "uniform")
    if mode == "float":
        d = {k: v.astype(np.float32).astype(np.float64)
             for k, v in d.items()}
    ps = system(d, torch.float32 if mode == "float" else torch.float64)
    rows = np.unique(np.concatenate([rows_of(n), [1088, n - 1025, n - 700]]))
    got = [g[rows].astype(np.float64) for g in run(kernel, mode, ps)]
    ref = oracle_rows(kernel, d, rows)
    if kernel == "tstep":
        for g, r in zip(got, ref):
            assert np.max(np.abs(g / r - 1)) <= 1e-6
        return
    if kernel == "phi":
        assert np.max(np.abs(got[0] / ref[0] - 1)) <= 2e-5
        return
    if kernel in ("acc", "acc_jerk"):
        assert acc_bar(d, rows, got, ref) <= 8 * 2.0**-24
    for a in range(0, len(got), 3):
        assert vec_rel_err(got[a:a + 3], ref[a:a + 3]) <= \
            (2e-5 if mode == "float" else 1e-5)


def test_partial_sums_past_the_limit():
    n = 450001
    d = state(n, 7, "uniform")
    ps = system(d, torch.float64)
    rows = np.array([0, 1024, n // 2, n - 1])
    got = [g[rows] for g in run("acc_jerk", "fp64", ps)]
    ref = oracle_rows("acc_jerk", d, rows)
    assert vec_rel_err(got[:3], ref[:3]) <= 1e-13
    assert vec_rel_err(got[3:], ref[3:]) <= 1e-13
