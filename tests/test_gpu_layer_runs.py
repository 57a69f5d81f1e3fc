"""Layer chains whose coarse nodes run several to a launch, and Voronoi tiles aligned to the lattice: the
oracle's maps bit for bit for widths and heights around the tiles, origins at every place in a lattice
cell (negative ones too), few and many maps, and maps so large that some coarse nodes get launches of
their own."""
import ctypes as C

import numpy as np
import pytest

from superterrainplus_amd import capi

from helpers import log
from test_gpu_layer import registry_tuple

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,origins", [
    (1, 1, [(0, 0), (-1, -1), (2, 3)]), (17, 5, [(x, z) for x in (-3, -2, -1, 0) for z in (-6, -5, -4, -3)]),
    (64, 16, [(2, 2), (-62, 18)]), (65, 33, [(1001, -777)]), (130, 67, [(-12345, 6789), (12, 34)]), (300, 1, [(7, 9)]), (3, 400, [(-9, 11)]),
    (1500, 900, [(-700, 123)])])
def test_layer_maps_bit_exact(gpu, oracle, width, height, origins):
    log(f"layer runs {width}x{height} maps={len(origins)}")
    nodes, registry = capi.demo_layer_program(), capi.demo_biome_registry()
    factory = C.c_void_p()
    capi.call("stp_layer_factory_create", (capi.LayerNode * len(nodes))(*nodes), len(nodes), 77, C.byref(registry), width, height,
              C.byref(factory))
    try:
        out = capi.DeviceArray((len(origins), height, width), np.uint16)
        flat = (C.c_int32 * (2 * len(origins)))(*[v for o in origins for v in o])
        capi.call("stp_layer_factory_generate_device", factory, out.vp, flat, len(origins), None)
        capi.synchronize()
        got, status = out.download(), C.c_uint32()
        capi.call("stp_layer_factory_status", factory, C.byref(status))
        assert status.value == 0
    finally:
        capi.lib().stp_layer_factory_destroy(factory)
    chain = [oracle.layer_node(n.Kind, n.Salt, [p for p in n.Parent if p >= 0], n.Param, n.CacheSize) for n in nodes]
    assert (got == oracle.layer_biomemap(chain, 77, registry_tuple(registry), origins, width, height)).all()


LOW, HIGH = -2 ** 31, 2 ** 31 - 1


@pytest.mark.parametrize("origin,ok", [((LOW, 0), False), ((0, LOW + 1), False), ((LOW + 2, LOW + 2), True), ((HIGH - 4, HIGH - 3), True),
                                       ((HIGH - 3, 0), False)])
def test_layer_coordinate_ends(gpu, oracle, origin, ok):
    """Where a Voronoi root's own arithmetic would leave int (x - 2), and where its last column does, the
    map is refused on the host."""
    log(f"layer coordinates {origin}")
    # a continent node (0), a Voronoi node (4) on it
    nodes = [capi.LayerNode(0, 0, (C.c_int32 * 2)(-1, -1), 5, 32), capi.LayerNode(4, 0, (C.c_int32 * 2)(0, -1), 7, 32)]
    registry, factory = capi.demo_biome_registry(), C.c_void_p()
    capi.call("stp_layer_factory_create", (capi.LayerNode * 2)(*nodes), 2, 77, C.byref(registry), 5, 4, C.byref(factory))
    try:
        out = capi.DeviceArray((4, 5), np.uint16)
        go = lambda: capi.call("stp_layer_factory_generate_device", factory, out.vp, (C.c_int32 * 2)(*origin), 1, None)  # noqa: E731
        if not ok:
            with pytest.raises(capi.STPError):
                go()
            return
        go()
        capi.synchronize()
        got = out.download()
    finally:
        capi.lib().stp_layer_factory_destroy(factory)
    chain = [oracle.layer_node(n.Kind, n.Salt, [p for p in n.Parent if p >= 0], n.Param, n.CacheSize) for n in nodes]
    assert (got[None] == oracle.layer_biomemap(chain, 77, registry_tuple(registry), [origin], 5, 4)).all()
