"""The generator's serialized erosion with independent drops run at the same time: the oracle's heights
bit for bit over two erosions (the stream id advances), from maps where every drop is in every other
one's way to sparse ones, at the edges of a chunk of steps, of the brush sizes and of the range the
ordered passes take (a lifetime of 1 to 256 steps, a brush radius of up to 16, more than one drop; the
others run drop by drop)."""
import ctypes as C

import numpy as np
import pytest

from superterrainplus_amd import capi, workloads as W

from helpers import log, oracle_rain

pytestmark = pytest.mark.gpu

NOISE = capi.SimplexNoiseSetting(42, W.DISTRIBUTION, W.GRADIENT_OFFSET, W.ENGINE_MT19937)


def rain_setting(drops, radius, lifetime, **kw):
    s = W.erosion_setting(drops, seed=7, lifetime=lifetime)
    s.ErosionBrushRadius = radius
    for k, v in kw.items():
        setattr(s, k, v)
    return s


def erode(gpu_chunks, mx, my, nn, rain, calls):
    c = capi.ChunkSetting()
    c.ChunkSize[:] = c.MapSize[:] = [mx, my]
    c.ChunkScale[:] = [1.0, 1.0]
    c.DiversityNearestNeighbour[:] = c.SplatNearestNeighbour[:] = [1, 1]
    c.ErosionNearestNeighbour[:] = [nn, nn]
    c.RenderDistance[:] = [3, 3]
    plugin, gen = C.c_void_p(), C.c_void_p()
    capi.call("stp_diversity_simplex_create", C.byref(NOISE), C.byref(capi.BiomeProperty(*W.Fractal().biome())),
              (C.c_uint32 * 2)(mx, my), C.byref(plugin))
    try:
        capi.call("stp_heightfield_generator_create", C.byref(c), C.byref(rain), plugin, C.byref(gen))
        capi.call("stp_heightfield_generator_set_erosion_mode", gen, 1)
        fixed = [np.zeros((my, mx), np.uint16) for _ in gpu_chunks]
        for _ in range(calls):
            capi.call("stp_heightfield_erode", gen, (C.c_void_p * len(gpu_chunks))(*[a.ctypes.data for a in gpu_chunks]),
                      (C.c_void_p * len(fixed))(*[a.ctypes.data for a in fixed]))
        return fixed
    finally:
        capi.lib().stp_heightfield_generator_destroy(gen)
        capi.lib().stp_diversity_destroy(plugin)


CASES = [(64, 64, 1, 1500, 3, 30, {}), (256, 192, 1, 1200, 3, 30, {}), (96, 96, 3, 2000, 3, 30, {}), (128, 128, 1, 600, 2, 6, {}),
         (128, 128, 1, 600, 4, 7, {}), (200, 100, 1, 500, 1, 13, {}), (160, 160, 1, 300, 6, 30, {}), (150, 170, 1, 150, 16, 12, {}),
         (100, 100, 1, 700, 3, 1, {}), (150, 150, 1, 200, 3, 256, {}), (90, 90, 1, 2, 3, 30, {}), (90, 90, 1, 1, 3, 30, {}),
         (90, 90, 1, 60, 3, 257, {}), (90, 90, 1, 60, 17, 20, {}), (128, 128, 1, 500, 3, 40, {"minWaterVolume": 0.9}),
         (128, 128, 1, 500, 3, 40, {"minWaterVolume": 2.0, "initWaterVolume": 1.0})]


@pytest.mark.parametrize("mx,my,nn,drops,radius,lifetime,kw", CASES)
def test_ordered_erosion_bit_exact(gpu, oracle, mx, my, nn, drops, radius, lifetime, kw):
    log(f"ordered erosion {mx}x{my} nn={nn} drops={drops} r={radius} lifetime={lifetime} {kw}")
    rng = np.random.default_rng(mx + 3 * my + drops)
    # hills with a plateau (drops that stop at once) and a step (steep slopes, deposits)
    y, x = np.mgrid[0:my * nn, 0:mx * nn].astype(np.float64)
    h = 0.5 + 0.2 * np.sin(x / 11.0) * np.cos(y / 17.0) + 0.02 * rng.random((my * nn, mx * nn))
    h[:my // 4, :mx // 3] = 0.6
    h[my // 2:, mx // 2:] += 0.15
    merged = h.astype(np.float32)
    chunks = [np.ascontiguousarray(c) for c in oracle.nn_unmerge(merged, (nn, nn), (mx, my))]
    rain = rain_setting(drops, radius, lifetime, **kw)
    for call in range(2):
        oracle.erode(merged, (nn, nn), (mx, my), oracle_rain(oracle, rain), drops, rain.Seed, stream_id=call)
    fixed = erode(chunks, mx, my, nn, rain, 2)
    want = oracle.nn_unmerge(merged, (nn, nn), (mx, my))
    assert all(c.tobytes() == w.tobytes() for c, w in zip(chunks, want))
    assert all((f == w).all() for f, w in zip(fixed, oracle.nn_unmerge(oracle.format_heightmap(merged), (nn, nn), (mx, my))))


def ordered(merged, mx, my, nn, rain, poll_limit):
    """The heights of the ordered passes alone and whether they gave up."""
    d = capi.DeviceArray.from_host(merged)
    idx, w = capi.brush(mx * nn, rain.ErosionBrushRadius)
    d_idx, d_w = capi.DeviceArray.from_host(idx), capi.DeviceArray.from_host(w)
    gave_up = C.c_int(-1)
    capi.call("stp_hydraulic_erosion_ordered", d.vp, C.byref(capi.nn_info((mx, my), (nn, nn))), C.byref(rain), d_idx.vp, d_w.vp,
              idx.size, 0, poll_limit, C.byref(gave_up), None)
    return d.download(), gave_up.value


WAYS = [(64, 64, 1, 1500, 3, 30, {}), (96, 96, 3, 2000, 3, 30, {}), (128, 128, 1, 600, 2, 6, {}), (150, 170, 1, 150, 16, 12, {}),
        (150, 150, 1, 200, 3, 256, {})]


@pytest.mark.parametrize("limit", [1 << 22, 0])
@pytest.mark.parametrize("mx,my,nn,drops,radius,lifetime,kw", WAYS)
def test_ordered_passes_and_their_way_out(gpu, oracle, mx, my, nn, drops, radius, lifetime, kw, limit):
    """The ordered passes come to their end by themselves. With no patience at all the first wave in another
    one's way gives up, and the serialized kernel erodes the saved map. The oracle's bits both times."""
    log(f"ordered passes {mx}x{my} nn={nn} drops={drops} r={radius} lifetime={lifetime} limit={limit}")
    y, x = np.mgrid[0:my * nn, 0:mx * nn].astype(np.float64)
    before = (0.5 + 0.2 * np.sin(x / 11.0) * np.cos(y / 17.0)).astype(np.float32)
    rain = rain_setting(drops, radius, lifetime, **kw)
    want = before.copy()
    oracle.erode(want, (nn, nn), (mx, my), oracle_rain(oracle, rain), drops, rain.Seed, stream_id=0)
    got, gave_up = ordered(before, mx, my, nn, rain, limit)
    assert gave_up == (1 if limit == 0 else 0)
    assert got.tobytes() == want.tobytes()


@pytest.mark.parametrize("drops,radius,lifetime", [(1, 3, 30), (60, 17, 30), (60, 3, 257)])
def test_ordered_passes_refuse(gpu, drops, radius, lifetime):
    with pytest.raises(capi.STPError):
        ordered(np.full((90, 90), 0.5, np.float32), 90, 90, 1, rain_setting(drops, radius, lifetime), 1 << 22)
