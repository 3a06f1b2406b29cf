"""tupan_sia_split and tupan_sia_update against the array operations they
replace: bit for bit, at sizes around the partition's blocks (1024 particles
each, 256 of them summed at once), with all, none and some particles slow,
NaN and signed zero steps, on views that start inside a larger array, and
the routes that keep the array operations (float32, non-contiguous)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def system(n, seed, offset):
    from tupan_amd.particles import ParticleSystem
    rng = np.random.default_rng(seed)
    d = {k: rng.standard_normal(n + offset) for k in
         ("mass", "eps2", "rx", "ry", "rz", "vx", "vy", "vz", "time",
          "tstep")}
    d["id"] = rng.permutation(n + offset)
    d["nstep"] = rng.integers(0, 9, n + offset)
    ps = ParticleSystem.from_numpy(d, device="cuda:0")
    for k in ("ax", "ay", "az"):
        ps.register_auxiliary_attribute(k, "real")
        getattr(ps, k).copy_(torch.as_tensor(rng.standard_normal(n + offset)))
    return ps


def same(a, b):
    for k, v in a.arrays().items():
        w = b.arrays()[k]
        assert torch.equal(v.view(torch.int64), w.view(torch.int64)), k


@pytest.mark.parametrize("n", [3, 64, 1023, 1024, 1025, 5000, 262145 + 1024])
@pytest.mark.parametrize("threshold", [0.7, -1.0, 1e300])
def test_partition_matches_array_operations(n, threshold):
    from tupan_amd.integrator import sia
    whole = system(n, n, 7)
    whole.tstep[8] = float("nan")
    whole.tstep[9] = -0.0
    other = whole.copy()
    a, b = whole[7:7 + n], other[7:7 + n]
    slow, fast = sia.partition_level(a, threshold)
    rslow, rfast = sia.partition(b, abs(b.tstep) > threshold)
    assert (slow.n, fast.n) == (rslow.n, rfast.n)
    same(whole, other)


@pytest.mark.parametrize("n", [1, 255, 257, 70001])
def test_updates_match_array_operations(n):
    from tupan_amd.integrator import sia
    from tupan_amd.integrator.device_update import BOOK, device_update
    ps = system(n, 3, 1)
    other = ps.copy()
    a, b = ps[1:1 + n], other[1:1 + n]
    h = 0.1 / 3
    sia.drift(a, h)
    sia.kick_n(a, -h)
    assert device_update(BOOK, (a.tstep, a.time, a.nstep), h)
    for x, v in (("rx", "vx"), ("ry", "vy"), ("rz", "vz")):
        t = getattr(b, x)
        t += getattr(b, v) * h
    for x, v in (("vx", "ax"), ("vy", "ay"), ("vz", "az")):
        t = getattr(b, x)
        t += getattr(b, v) * -h
    b.tstep[...] = h
    b.time += h
    b.nstep += 1
    same(ps, other)


@pytest.mark.parametrize("n", [1, 256, 70001])
def test_sakura_updates_match_array_operations(n):
    from tupan_amd.integrator import device_update as du
    ps = system(n, 4, 0)
    for k in ("drx", "dry", "drz", "dvx", "dvy", "dvz"):
        ps.register_auxiliary_attribute(k, "real")
        getattr(ps, k).copy_(ps.rx * 0.3 + ps.vy)
    other = ps.copy()
    tau = 0.1 / 3
    du.half_drift(ps, tau)
    du.apply_pair_drift(ps)
    for x in "xyz":
        t = getattr(other, "r" + x)
        t += getattr(other, "v" + x) * tau / 2
    for k in ("rx", "ry", "rz", "vx", "vy", "vz"):
        t = getattr(other, k)
        t += getattr(other, "d" + k)
    same(ps, other)


def test_other_arrays_keep_the_array_operations():
    from tupan_amd.integrator.device_update import DRIFT, device_update
    x = [torch.ones(8, device="cuda:0") for _ in range(6)]
    assert not device_update(DRIFT, x, 0.5)
    y = [torch.ones(16, dtype=torch.float64, device="cuda:0")[::2]
         for _ in range(6)]
    assert not device_update(DRIFT, y, 0.5)
    assert not device_update(DRIFT, [t.cpu() for t in y], 0.5)


@pytest.mark.parametrize("narr", [1, 3, 4, 5, 16, 31, 32])
@pytest.mark.parametrize("n", [7, 1025])
def test_partition_moves_every_array(n, narr):
    """Array counts around the four that a block moves, the first array the
    step sizes themselves: order and bits of a stable partition."""
    import ctypes as C
    from tupan_amd import _native
    g = torch.Generator(device="cuda:0").manual_seed(n + narr)
    arrs = [torch.rand(n, dtype=torch.float64, device="cuda:0", generator=g)
            for _ in range(narr)]
    slow = arrs[0] > 0.4
    ref = [torch.cat((a[slow], a[~slow])) for a in arrs]
    ptrs = (C.c_void_p * narr)(*[a.data_ptr() for a in arrs])
    out = (C.c_int * 2)()
    _native.check(_native.lib().tupan_sia_split(
        n, ptrs, narr, arrs[0].data_ptr(), 0.4, None, out,
        torch.cuda.current_stream().cuda_stream), "tupan_sia_split")
    assert out[0] == int(slow.sum()) and out[1] == 0
    for a, r in zip(arrs, ref):
        assert torch.equal(a, r)
