"""The symmetric engine (sym.h): a set against itself above a few thousand
particles, each unordered pair once.

Sizes where it can go wrong: the first it takes in each arithmetic (2049 in
FP64, 4097 in FP32), one particle past a whole block, the last and first
sizes of neighbouring shapes (9216 | 9217: one and two particles per lane;
36864 | 36865: two and four in FP64), odd and even block counts.  Rows at
block edges are checked against the oracle, on views that start at an odd
element (arrays aligned to 8 bytes only), with coincident particles.

Bars: FP64 1e-13 of the row's vector; split-FP32 and the float build 8 FP32
roundings (8 x 2^-24) of the row's sum of contribution magnitudes, formed
here in FP64, for the accelerations (as test_gpu_pairwise.py), and 2e-5 of
the row's vector for the float build's other outputs; Tstep 1e-6 in FP32
arithmetic.
"""
import numpy as np
import pytest

from conftest import vec_rel_err

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

ETA = 1.0 / 64
CLASSES = {"acc": "Acc", "acc_jerk": "AccJerk", "tstep": "Tstep",
           "snap_crackle": "SnapCrackle", "phi": "Phi"}


def state(n, seed, soft):
    rng = np.random.default_rng(seed)
    d = {k: rng.standard_normal(n) for k in
         ("rx", "ry", "rz", "vx", "vy", "vz", "ax", "ay", "az", "jx", "jy",
          "jz")}
    d["mass"] = rng.uniform(0.5, 1.5, n) / n
    d["eps2"] = np.full(n, 1e-6) if soft == "uniform" else \
        rng.uniform(0.0, 2e-6, n)
    # two particles of different blocks at one position, at rest to each
    # other in no component
    for k in ("rx", "ry", "rz"):
        d[k][n - 1] = d[k][3]
    return d


def system(d, dtype, offset=1):
    """Device system whose arrays start `offset` elements into a buffer."""
    from tupan_amd.particles import ParticleSystem
    ps = ParticleSystem.from_numpy(d, device="cuda:0")
    for k, v in list(ps.arrays().items()):
        if v.dtype == torch.float64:
            ps.__dict__[k] = v.to(dtype)
    for k in d:
        v = torch.as_tensor(d[k], device="cuda:0").to(dtype)
        buf = torch.empty(v.numel() + offset, dtype=dtype, device="cuda:0")
        buf[offset:] = v
        ps.__dict__[k] = buf[offset:]
    return ps


def rows_of(n):
    edges = [0, 3, 63, 64, 255, 256, 511, 512, 1023, 1024, n // 2, n - 2,
             n - 1]
    return np.unique([r for r in edges if r < n])


def oracle_rows(kernel, d, rows, prec="float64"):
    from oracle import Oracle
    o = Oracle(prec)
    i = {k: v[rows] for k, v in d.items()}
    fn = getattr(o, kernel)
    return fn(i, d, ETA) if kernel == "tstep" else fn(i, d)


def run(kernel, mode, ps):
    from tupan_amd.lib import extensions
    prec = "float32" if mode == "float" else "float64"
    ext = getattr(extensions, CLASSES[kernel])(
        "HIP", prec, mode="fp64" if mode == "float" else mode)
    args = (ETA,) if kernel == "tstep" else ()
    out = ext.calc(ps, ps, *args)
    torch.cuda.synchronize()
    return [r.detach().cpu().numpy() for r in out]


FP64 = (2049, 2304, 2305, 9216, 9217, 36864, 36865)
FP32 = (4097, 4353, 9216, 9217)
CASES = ([(k, "fp64", n) for k in ("acc", "acc_jerk", "tstep", "snap_crackle")
          for n in FP64 if k == "acc_jerk" or n in (2049, 9217, 36865)]
         + [(k, "split32", n) for k in ("acc", "acc_jerk", "tstep")
            for n in FP32 if k == "acc_jerk" or n in (4097, 9217)]
         + [("phi", "fp64", n) for n in (32768, 32769, 36865)]
         + [(k, "float", n) for k in CLASSES for n in (4097, 9217)])


@pytest.mark.parametrize("soft", ["uniform", "mixed"])
@pytest.mark.parametrize("kernel,mode,n", CASES)
def test_rows_vs_oracle(kernel, mode, n, soft):
    print(kernel, mode, n, soft, flush=True)
    d = state(n, n, soft)
    if mode == "float":
        d = {k: v.astype(np.float32).astype(np.float64)
             for k, v in d.items()}
    ps = system(d, torch.float32 if mode == "float" else torch.float64)
    rows = rows_of(n)
    got = [g[rows].astype(np.float64) for g in run(kernel, mode, ps)]
    ref = oracle_rows(kernel, d, rows)
    if kernel == "tstep":
        bar = 1e-13 if mode == "fp64" else 1e-6
        for g, r in zip(got, ref):
            assert np.max(np.abs(g / r - 1)) <= bar
        return
    if kernel == "phi":
        assert np.max(np.abs(got[0] / ref[0] - 1)) <= \
            (1e-13 if mode == "fp64" else 2e-5)
        return
    if mode == "fp64":
        assert vec_rel_err(got[:3], ref[:3]) <= 1e-13
        if len(got) > 3:
            assert vec_rel_err(got[3:], ref[3:]) <= 1e-13
        return
    # accelerations: FP32 roundings of the contributions' magnitudes
    if kernel in ("acc", "acc_jerk"):
        dr = [d[k][rows][:, None] - d[k][None, :] for k in ("rx", "ry", "rz")]
        r2 = sum(x * x for x in dr)
        R2 = r2 + d["eps2"][rows][:, None] + d["eps2"][None, :]
        w = np.where(r2 > 0, d["mass"] * np.sqrt(r2) / np.where(
            r2 > 0, R2, 1.0)**1.5, 0.0).sum(1)
        err = np.sqrt(sum((g - r)**2 for g, r in zip(got[:3], ref[:3])))
        assert np.max(err / w) <= 8 * 2.0**-24
    for a in range(0, len(got), 3):
        assert vec_rel_err(got[a:a + 3], ref[a:a + 3]) <= \
            (2e-5 if mode == "float" else 1e-5)


@pytest.mark.parametrize("kernel", ["acc", "acc_jerk", "tstep"])
def test_split32_overflow_falls_back_to_fp64(kernel):
    """An unsoftened pair 1e-15 apart overflows FP32; both particles' rows
    are evaluated again in FP64 by the reduction."""
    n = 5003
    d = state(n, 5, "uniform")
    d["eps2"][:] = 0.0
    for k in ("rx", "ry", "rz"):
        d[k][n - 1] += 3.0
    i, j = 70, 4100
    for k in ("rx", "ry", "rz"):
        d[k][i] = d[k][j] = 0.0
    d["rx"][j] = 1e-15
    ps = system(d, torch.float64)
    rows = np.array([i, j, 0, n - 1])
    got = [g[rows] for g in run(kernel, "split32", ps)]
    ref = oracle_rows(kernel, d, rows)
    for g, r in zip(got, ref):
        assert np.all(np.isfinite(g))
        assert np.max(np.abs(g[:2] - r[:2]) / np.abs(r[:2]).max()) <= 1e-12
        assert np.max(np.abs(g[2:] / r[2:] - 1)) <= 1e-4


def test_repeated_calls_and_streams_are_bitwise_equal():
    """The sums are added in a fixed order: repeated calls, and calls on a
    second stream, give the same bits."""
    ps = system(state(9301, 9, "uniform"), torch.float64)
    first = run("acc_jerk", "fp64", ps)
    again = run("acc_jerk", "fp64", ps)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        other = run("acc_jerk", "fp64", ps)
    for a, b, c in zip(first, again, other):
        assert np.array_equal(a, b) and np.array_equal(a, c)
