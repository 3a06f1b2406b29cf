"""Autotuner: ``python -m tupan_amd.tune [--quick]`` on the target GPU.

For every pairwise kernel and arithmetic mode it times each compiled tile
shape at 2, 4, 8 and 16 workgroups per CU on calls between two random
clusters of a few sizes per size bucket (few i against many j, square, many i
against few j), and keeps the entry with the smallest mean of time over the
best time of that size (GPU time of the whole call, combine included).  For
the ensemble plan it times each lanes-per-system packing on the 4096-system
workload.  The choices go to tupan_amd/tune/cache.json, which the library
applies when it loads.
"""
import argparse
import json
import sys
import time

import numpy as np
import torch

from .. import _native
from . import CACHE, load, save

KERNELS = {  # name -> (kernel id, modes)
    "phi": (_native.K_PHI, ("fp64", "float32")),
    "acc": (_native.K_ACC, ("fp64", "split32", "float32")),
    "acc_jerk": (_native.K_ACC_JERK, ("fp64", "split32", "ieee64",
                                      "float32")),
    "snap_crackle": (_native.K_SNAP_CRACKLE, ("fp64", "float32")),
    "tstep": (_native.K_TSTEP, ("fp64", "split32", "float32")),
    "nreg_x": (_native.K_NREG_X, ("fp64", "float32")),
    "nreg_v": (_native.K_NREG_V, ("fp64", "float32")),
    "pnacc": (_native.K_PNACC, ("fp64", "split32", "float32")),
}
# (ni, nj) of the calls timed, each in its kernel's size bucket
SETS = ((200, 3000), (64, 16000), (4000, 700), (2000, 2100), (300, 50000),
        (16000, 700), (4000, 4096), (3000, 50000), (6000, 6000), (9000, 7000),
        (15000, 15500), (60000, 2500), (30000, 31000), (20000, 60000),
        (65000, 66000))


def size_bucket(name, ni, nj):
    """The library's bucket of a call (engine.h: size_bucket)."""
    pairs = ni * nj
    low = name == "pnacc" or (name == "snap_crackle" and ni >= 16384)
    if pairs < (1 << 22 if low else 1 << 25):
        return 0
    return 1 if pairs < 1 << 30 else 2


def cluster(n, seed=0, dtype=torch.float64):
    from ..particles import ParticleSystem
    rng = np.random.default_rng(seed)
    d = {k: rng.normal(0, 1, n) for k in ("rx", "ry", "rz", "vx", "vy",
                                         "vz", "ax", "ay", "az", "jx", "jy",
                                         "jz")}
    d["mass"] = np.full(n, 1.0 / n)
    d["eps2"] = np.full(n, 1e-8)
    ps = ParticleSystem.from_numpy(d, device="cuda:0")
    if dtype != torch.float64:
        for k, v in list(ps.arrays().items()):
            if v.dtype == torch.float64:
                ps.__dict__[k] = v.to(dtype)
    return ps


def queued_ms(fn, reps, hold):
    """GPU time of one fn() in a run of `reps` behind a product of the
    square matrix `hold`, which keeps the GPU busy while the host queues the
    run: kernels and the gaps between them, no host time.  Best of 2."""
    best = None
    for _ in range(2):
        t0 = torch.cuda.Event(enable_timing=True)
        t1 = torch.cuda.Event(enable_timing=True)
        torch.mm(hold, hold)
        t0.record()
        for _ in range(reps):
            fn()
        t1.record()
        t1.synchronize()
        t = t0.elapsed_time(t1) / reps
        best = t if best is None else min(best, t)
    return best


def time_call(fn, reps):
    """Best of `reps` GPU times of fn(), from events on the launch stream
    around the whole call (all-pairs kernel, split combine and the gaps
    between their launches)."""
    fn()
    torch.cuda.synchronize()
    best = None
    for _ in range(reps):
        t0 = torch.cuda.Event(enable_timing=True)
        t1 = torch.cuda.Event(enable_timing=True)
        t0.record()
        fn()
        t1.record()
        t1.synchronize()
        t = t0.elapsed_time(t1)
        best = t if best is None else min(best, t)
    return best


def tune_pairwise(quick, names, pinned=()):
    from . import SLOTS
    from ..lib import extensions
    lib = _native.lib()
    out = []
    # PNAcc at the reference's own test values (order 7, c = 128)
    extensions.clight.pn_order, extensions.clight.clight = 7, 128.0
    hold = torch.ones(2048, 2048, dtype=torch.float64, device="cuda:0")
    classes = {"phi": extensions.Phi, "acc": extensions.Acc,
               "acc_jerk": extensions.AccJerk,
               "snap_crackle": extensions.SnapCrackle,
               "tstep": extensions.Tstep, "nreg_x": extensions.NREG_X,
               "nreg_v": extensions.NREG_V, "pnacc": extensions.PNAcc}
    for b in range(2 if quick else 3):
        for name, (kid, modes) in KERNELS.items():
            if name not in names:
                continue
            sets = [s for s in SETS if size_bucket(name, *s) == b]
            for mode in modes:
                if (name, mode) in pinned:
                    continue
                flt = mode == "float32"
                ext = (classes[name]("HIP", "float32") if flt else
                       classes[name]("HIP", "float64", mode=mode))
                args = (0.01,) if name in ("tstep", "nreg_x", "nreg_v") else ()
                times = {}
                for ni, nj in sets:
                    dt = torch.float32 if flt else torch.float64
                    ips, jps = cluster(ni, 0, dt), cluster(nj, 1, dt)
                    reps = 10 if b == 0 else 2
                    ext.calc(ips, jps, *args)
                    for shape in range(6):
                        for wg in (2, 4, 8, 16):
                            _native.check(
                                lib.tupan_tune_set(kid, SLOTS[mode], b, shape,
                                                   wg), "tupan_tune_set")
                            times.setdefault((shape, wg), []).append(queued_ms(
                                lambda: ext.calc(ips, jps, *args), reps, hold))
                best = [min(t[q] for t in times.values())
                        for q in range(len(sets))]
                score = {k: sum(x / y for x, y in zip(t, best)) / len(sets)
                         for k, t in times.items()}
                shape, wg = min(score, key=score.get)
                _native.check(lib.tupan_tune_set(kid, SLOTS[mode], b, shape,
                                                 wg), "tupan_tune_set")
                out.append({"kernel": name, "mode": mode, "bucket": b,
                            "shape": shape, "wg_per_cu": wg,
                            "over_best": round(score[shape, wg], 3),
                            "default_over_best": round(score[0, 4], 3)})
                print("%-12s %-7s bucket %d shape %d wg/cu %2d  %.3f x best "
                      "(default %.3f)" % (name, mode, b, shape, wg,
                                          score[shape, wg], score[0, 4]),
                      flush=True)
    return out


def tune_ensemble(nsys):
    from ..ics.ensemble import make_ensemble
    from ..lib.ensemble import Ensemble
    ps, ens = make_ensemble(nsys=nsys, nmin=3, nmax=64, seed=1,
                            device="cuda:0")
    res = []
    for lanes in (8, 16, 32, 64):
        e = Ensemble(ens.offsets, min_lanes=lanes)
        t = time_call(lambda: e.sakura(ps, 1.0 / 64, -1), 3)
        res.append((t, lanes))
        print("ensemble min_lanes %2d  %.3f ms" % (lanes, t), flush=True)
    res.sort()
    return {"min_lanes": res[0][1], "ms": res[0][0],
            "all": {str(L): t for t, L in res}}


def main(argv=None):
    ap = argparse.ArgumentParser()
    ap.add_argument("--quick", action="store_true")
    ap.add_argument("--ensemble-systems", type=int, default=4096)
    ap.add_argument("--kernels", default=",".join(KERNELS),
                    help="comma-separated subset; the cache keeps the other "
                         "kernels' entries")
    args = ap.parse_args(argv)
    assert torch.cuda.is_available(), "the autotuner runs on the GPU"
    names = [k for k in args.kernels.split(",") if k]
    for k in names:
        if k not in KERNELS:
            raise SystemExit("unknown kernel %r" % k)
    cu, _ = _native.device_info()
    t0 = time.time()
    old = load()
    # a pinned entry (FP64 phi: the summation order behind a seed's initial
    # conditions) stays
    keep = [e for e in old.get("pairwise", [])
            if e.get("kernel") not in names or e.get("pinned")]
    pinned = {(e["kernel"], e["mode"]) for e in keep if e.get("pinned")}
    data = {"device": {"cu": cu, "name": torch.cuda.get_device_name(0)},
            "pairwise": keep + tune_pairwise(args.quick, names, pinned)}
    if args.ensemble_systems > 0:
        data["ensemble"] = tune_ensemble(args.ensemble_systems)
    elif "ensemble" in old:
        data["ensemble"] = old["ensemble"]
    data["seconds"] = time.time() - t0
    save(data)
    print("wrote", CACHE)
    return 0


if __name__ == "__main__":
    sys.exit(main())
