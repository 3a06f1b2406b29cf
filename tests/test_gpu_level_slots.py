"""Slots of the device-scheduled SIA levels: the workers a slot launches are
those a call of a set of n can reach, so its launches are counted in a
captured graph, at sizes with and without the symmetric engine's shapes and
the table's second size bucket; and a step over each of them equals the host
driver's bit for bit (no call is left without its worker)."""
import ctypes
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

MODES = ("fp64", "split32")


def integrator(n, mode, **kw):
    from tupan_amd.integrator import Integrator
    from tupan_amd.lib import extensions
    from tupan_amd.particles import ParticleSystem
    extensions.install("HIP", "float64", mode=mode)
    rng = np.random.default_rng(n)
    d = {k: rng.standard_normal(n) for k in ("rx", "ry", "rz", "vx", "vy",
                                             "vz")}
    d["mass"] = rng.uniform(0.1, 2.0, n)**2 / n
    d["eps2"] = np.full(n, 1e-6)
    ps = ParticleSystem.from_numpy(d, device="cuda:0")
    type(ps).t_curr = 0.0
    return Integrator(2.0**-9, 0.0, ps, method="sia21h.dkd", **kw), ps


@pytest.fixture(autouse=True)
def default_extensions():
    yield
    from tupan_amd.lib import extensions
    extensions.install("HIP", "float64")


def hip_runtime():
    """The HIP runtime this process runs on."""
    for line in open("/proc/self/maps"):
        m = re.search(r"(/\S*libamdhip64\.so\S*)", line)
        if m:
            return ctypes.CDLL(m.group(1))
    raise RuntimeError("no HIP runtime mapped")


# launches besides the pair workers: the scheduler, four partition passes,
# updates, subtree, few-body
OTHER = 8


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n,pair", [
    # Tstep and Acc: tile shape and small-set kernel each; one combine
    (500, 5), (2000, 5),
    # and the symmetric engine with its reduction (from 2049 or 4097 on)
    (5000, 8),
    # a second symmetric shape each, Acc's second tile shape
    (12000, 11)])
def test_launches_per_slot(n, pair, mode):
    it, ps = integrator(n, mode, device_levels=True)
    it.initialize(1.0)
    lv = it.integrator._device_levels()
    nodes = []
    for slots in (1, 5):
        lv.slots = slots
        g = torch.cuda.CUDAGraph(keep_graph=True)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            with torch.cuda.graph(g, stream=side):
                lv.enqueue(False)
        torch.cuda.current_stream().wait_stream(side)
        count = ctypes.c_size_t(0)
        rc = hip_runtime().hipGraphGetNodes(
            ctypes.c_void_p(g.raw_cuda_graph()), None, ctypes.byref(count))
        assert rc == 0
        nodes.append(count.value)
    assert nodes[1] - nodes[0] <= 4 * (OTHER + pair), nodes
    lv.close()


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n", [257, 2000, 5000, 12000])
def test_step_equals_host_levels(n, mode):
    got = []
    for kw in ({}, {"device_levels": True}):
        it, ps = integrator(n, mode, **kw)
        it.evolve_step(1.0)
        order = torch.argsort(ps.id)
        got.append([getattr(ps, k)[order].cpu().numpy()
                    for k in ("rx", "ry", "rz", "vx", "vy", "vz")])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
