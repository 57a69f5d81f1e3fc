"""The fractal heightmap with one and with two pixels a thread: the oracle's bits for maps below, at and past
the size where the launch changes, with ragged edges, and with the most rows of a grid of one pixel a thread."""
import ctypes as C

import numpy as np
import pytest

from superterrainplus_amd import capi, workloads as W

from helpers import log

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,rows", [(1, 1), (65, 7), (63, 129), (1024, 512), (1024, 513), (727, 723), (1, 262144), (1, 300001)])
def test_heightmap_bit_exact(gpu, oracle, width, rows):
    log(f"heightmap {width}x{rows}")
    table = capi.PermutationTable(42, W.DISTRIBUTION, W.GRADIENT_OFFSET, W.ENGINE_MT19937)
    info = capi.FractalInformation(0.5, 2.0, 3, 200.0, (C.c_float * 2)(64.0, -32.0), (C.c_float * 2)(width / 2, rows / 2), 1.0, 1.0)
    out = capi.DeviceArray((rows, width), np.float32)
    capi.call("stp_simplex_heightmap", C.byref(table.view), C.byref(info), 1.0, 0.0, out.vp, width, rows, None)
    capi.synchronize()
    perm, g32, _ = oracle.permutation(42, W.DISTRIBUTION, W.GRADIENT_OFFSET, W.ENGINE_MT19937)
    d = oracle.FractalDesc(0.5, 2.0, 3, 200.0, 64.0, -32.0, width / 2, rows / 2, 1.0, 1.0)
    assert out.download().tobytes() == oracle.fractal_map(perm, g32, d, width, rows).tobytes()
