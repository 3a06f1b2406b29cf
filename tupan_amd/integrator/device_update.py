"""Elementwise updates of device-resident particle arrays in one launch
(libtupan_hip: tupan_sia_update), shared by the host-driven steps."""
import torch

DRIFT, BOOK, HALF_DRIFT, ADD = range(4)


def on_current_device(t):
    return t.is_cuda and t.get_device() == torch.cuda.current_device()


def device_update(kind, tensors, h=0.0):
    """One update of ``tensors`` (tupan_sia_update's arrays, in its order):
    DRIFT x += v h, BOOK, HALF_DRIFT x += (v h) / 2, ADD x += d.  The values
    are the array operations', bit for bit.  False, and nothing done, unless
    they are contiguous float64 arrays (BOOK's third: int64) of one size on
    the current device: the caller then runs the same operations array by
    array."""
    if not on_current_device(tensors[0]):
        return False
    n = tensors[0].numel()
    for k, t in enumerate(tensors):
        dtype = torch.int64 if kind == BOOK and k == 2 else torch.float64
        if not (t.is_cuda and t.dtype == dtype and t.is_contiguous()
                and t.numel() == n and not t.requires_grad):
            return False
    from .. import _native
    from ..lib.hip_backend import current_stream_handle
    _native.check(_native.lib().tupan_sia_update(
        kind, n, _native.ptr_array([t.data_ptr() for t in tensors]), h,
        current_stream_handle()), "tupan_sia_update")
    return True


def half_drift(ps, tau):
    """r += v tau / 2."""
    if not device_update(HALF_DRIFT, (ps.rx, ps.ry, ps.rz, ps.vx, ps.vy,
                                      ps.vz), tau):
        ps.rx += ps.vx * tau / 2
        ps.ry += ps.vy * tau / 2
        ps.rz += ps.vz * tau / 2


def apply_pair_drift(ps):
    """r += dr, v += dv of the Sakura pair drift."""
    if not device_update(ADD, (ps.rx, ps.ry, ps.rz, ps.vx, ps.vy, ps.vz,
                               ps.drx, ps.dry, ps.drz, ps.dvx, ps.dvy,
                               ps.dvz)):
        ps.rx += ps.drx
        ps.ry += ps.dry
        ps.rz += ps.drz
        ps.vx += ps.dvx
        ps.vy += ps.dvy
        ps.vz += ps.dvz
