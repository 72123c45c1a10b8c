"""``PyLB.stream`` and ``PyLB.stream_and_bounce_back`` on the GPU.

``stream(f_ikl)`` replaces ``PyLB/Streaming.py:33-46``: periodic streaming of
a ``(9, nx, ny)`` array in place, channel ``i`` moved by ``c_i``
(``PyLB/Streaming.py:28-29``).  As with the reference's ``np.roll`` loop the
values are only permuted, so any dtype of 1, 2, 4 or 8 bytes is accepted and
the result is bit-exact.

``stream_and_bounce_back(f_ikl, u0=0.1)`` replaces the cavity drivers' wall
function (``cavity_opt1.py:177-245``, ``cavity_opt2.py:109-177``): streaming,
half-way bounce-back on the bottom (l = 0), left (k = 0) and right
(k = nx-1) walls, and a lid at l = ny-1 moving with ``u0`` in +x; float32 or
float64.

numpy arguments are modified in place through a device round trip; torch
tensors on a ROCm device are processed on the device.
"""

import numpy as np
import torch
from torch.autograd import forward_ad

from latticeboltzmann_amd import kernels
from . import _staging

# Channel velocities, as PyLB/Streaming.py:28-29 exposes them.
c_ic = np.array([[0, 1, 0, -1, 0, 1, -1, -1, 1],
                 [0, 0, 1, 0, -1, 1, 1, -1, -1]]).T


def _check_populations(f, name):
    if isinstance(f, np.ndarray):
        if not f.flags.writeable:
            raise ValueError("%s(): array is read-only" % name)
    elif not _staging.is_device_tensor(f):
        raise TypeError("%s(): expected a numpy array or a ROCm device tensor" % name)
    if f.ndim != 3 or f.shape[0] != 9:
        raise ValueError("%s(): populations must have shape (9, nx, ny), got %s"
                         % (name, tuple(f.shape)))
    return f.shape[1] > 0 and f.shape[2] > 0


# Streaming in place moves half the bytes of a second array and a copy back, but a
# thread moves one value at a time down 16 rows and one block shifts a whole row, so
# it needs wide values, rows that fill their blocks, and rows enough to fill the GPU
# or short enough to be quick.  us a call in place against the second array:
#   1- and 2-byte values: uint8 3000 x 2000 57.6 / 41.8, FP16 6000 x 200 22.1 / 18.0
#     (2048^2 42.9 / 47.4): second array;
#   FP64 2048^2 105 / 235, FP32 2048^2 52 / 122, 1500 x 700 17.1 / 26.7;
#   rows of 512 bytes, FP64 6000 x 64 16.8 / 19.3, FP32 6000 x 128 18.0 / 19.4; FP32
#     6000 x 64 15.8 / 15.5, FP64 100000 x 10 186 / 73;
#   few long rows: FP32 64 x 20000 40.5 / 30.7, FP64 3 x 500000 760 / 64, but FP32
#     256 x 100000 644 / 687 and 64 x 6000 13.2 / 15.7.
# Small arrays are bound by the host, where the second array costs less (512^2, a
# call: FP32, 9.4 MB, 15.3 / 14.6, FP64 15.3 / 16.8).  The cavity form takes three
# launches against two and its side walls touch a cache line per row: it wants 48 MB
# (43 MB 30.8 / 29.8, 54 MB 31 / 37) and rows of 1024 bytes (FP64 100000 x 128
# 557 / 708, FP32 100000 x 128 361 / 343).
_IN_PLACE, _WALLS_IN_PLACE = 12 << 20, 48 << 20
_ROW_BYTES, _WALLS_ROW_BYTES = 512, 1024
_MANY_ROWS, _SHORT_ROW = 256, 6144


def _in_place(f, walls):
    if f.nbytes < (_WALLS_IN_PLACE if walls else _IN_PLACE):
        return False
    size, (_, nx, ny) = f.element_size(), f.shape
    # blocks of 256 threads of a launch, at most: 2.4 a row segment of 256 values
    return (size >= 4 and (nx >= _MANY_ROWS or ny <= _SHORT_ROW) and 3 * nx * (ny // 256 + 1) < 1 << 24
            and ny * size >= (_WALLS_ROW_BYTES if walls else _ROW_BYTES) and _plain(f))


def _plain(f):
    """A tensor whose memory the kernels may rewrite as it lies; the others
    (views, autograd leaves, lazily conjugated or negated ones, inference tensors
    outside inference mode, tensors with a forward-mode tangent) go through a
    second array and torch's own copy_ with its rules."""
    return (type(f) is torch.Tensor and f.is_contiguous() and not f.requires_grad
            and not f.is_conj() and not f.is_neg()
            and (torch.is_inference_mode_enabled() or not f.is_inference())
            and forward_ad.unpack_dual(f).tangent is None)


def stream(f_ikl):
    """Propagate channel occupations by one cell, periodic, in place."""
    if not _check_populations(f_ikl, "stream"):
        return
    itemsize = f_ikl.itemsize if isinstance(f_ikl, np.ndarray) else f_ikl.element_size()
    if itemsize not in (1, 2, 4, 8):
        raise TypeError("stream(): element size must be 1, 2, 4 or 8 bytes")
    if isinstance(f_ikl, np.ndarray):
        out = kernels.stream(_staging.to_device(f_ikl))
        _staging.write_back(f_ikl, out)
    elif _in_place(f_ikl, False):
        kernels.stream_in_place(f_ikl)
        _staging.written(f_ikl)
    else:
        src = f_ikl.contiguous()
        out = kernels.stream(src)
        f_ikl.copy_(out)


def stream_and_bounce_back(f_ikl, u0=0.1):
    """Stream and apply the cavity's no-slip walls and moving lid, in place."""
    if not _check_populations(f_ikl, "stream_and_bounce_back"):
        return
    if isinstance(f_ikl, np.ndarray):
        ok = f_ikl.dtype in (np.dtype(np.float32), np.dtype(np.float64))
    else:
        ok = f_ikl.dtype in (torch.float32, torch.float64)
    if not ok:
        raise TypeError("stream_and_bounce_back(): dtype must be float32 or float64")
    if isinstance(f_ikl, np.ndarray):
        out = kernels.stream_bounce_back(_staging.to_device(f_ikl), float(u0))
        _staging.write_back(f_ikl, out)
    elif _in_place(f_ikl, True):
        kernels.stream_in_place(f_ikl, float(u0))
        _staging.written(f_ikl)
    else:
        out = kernels.stream_bounce_back(f_ikl.contiguous(), float(u0))
        f_ikl.copy_(out)
