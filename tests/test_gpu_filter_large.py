"""The density filter and the OC sensitivity filter on a cell of more than
2^30 nodes, whose byte offsets need more than 32 bits: the planes past that
point against the same filter on a slab of them (whose kernels and order of
sums per output are the same, so the bits are)."""
import ctypes

import numpy as np
import pytest

import opentm_amd as otm
from opentm_amd import _capi

pytestmark = pytest.mark.gpu

NX, NY, NZ, PERIOD = 1031, 1025, 1027, 79  # plane z holds chunk[z % PERIOD]; 2^30 nodes are 1016 planes and a part
PLANE = NX * NY
Z0, MARGIN = 1005, 6  # first plane compared; a slab's outer planes are cut off (twice the reach at most)
RESO = (ctypes.c_int * 3)(NX, NY, NZ)


def chunk(seed):
    return np.random.default_rng(seed).random((PERIOD, NY, NX), dtype=np.float32) * np.float32(0.9) + np.float32(0.1)


def field(planes):
    lib = _capi.load()
    buf = otm.DeviceBuffer(PLANE * NZ)
    for z in range(0, NZ, PERIOD):
        _capi.check(lib.otm_memcpy(ctypes.c_void_p(buf.ptr.value + 4 * PLANE * z), planes.ctypes.data_as(ctypes.c_void_p),
                                   4 * planes.size, _capi.OTM_DEVICE, _capi.OTM_HOST), "otm_memcpy")
    return buf


def top(buf):
    out = np.empty((NZ - Z0, NY, NX), np.float32)
    _capi.check(_capi.load().otm_memcpy(out.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(buf.ptr.value + 4 * PLANE * Z0),
                                        4 * out.size, _capi.OTM_HOST, _capi.OTM_DEVICE), "otm_memcpy")
    return out


def test_cells_beyond_32_bit_offsets():
    assert PLANE * NZ > 1 << 30 and NZ % PERIOD == 0
    lib = _capi.load()
    x = chunk(1)
    din, dout = field(x), otm.DeviceBuffer(PLANE * NZ)
    slab = x[np.arange(Z0 - MARGIN, NZ) % PERIOD]
    for radius in (1.5, 3.4):
        for adjoint in (0, 1):
            _capi.check(lib.otm_conv_filter(RESO, 0, radius, 0, adjoint, din.ptr, dout.ptr, _capi.OTM_DEVICE),
                        "otm_conv_filter")
            ref = otm.conv_filter(slab, 0, radius, False, adjoint=bool(adjoint))[MARGIN:]
            same = np.array_equal(top(dout), ref)
            print("[case] filter radius", radius, "adjoint", adjoint, "same", same, flush=True)
            assert same


def test_sensitivity_filter_beyond_32_bit_offsets():
    s, r = chunk(2), chunk(3)
    dsens, drho = field(s), field(r)
    oc = otm.OCOptimizer(PLANE * NZ, 0.001, 0.02, 0.5)
    oc.filterSens(dsens, drho, NX, (NX, NY, NZ), 2.5)
    oc.close()
    planes = np.arange(Z0 - MARGIN, NZ + MARGIN) % NZ % PERIOD  # periodic: plane NZ is plane 0
    ss, rr = s[planes], r[planes]
    small = otm.OCOptimizer(ss.size, 0.001, 0.02, 0.5)
    small.filterSens(ss, rr, NX, (NX, NY, len(planes)), 2.5)
    small.close()
    same = np.array_equal(top(dsens), ss[MARGIN:-MARGIN])
    print("[case] sensitivity filter same", same, flush=True)
    assert same
