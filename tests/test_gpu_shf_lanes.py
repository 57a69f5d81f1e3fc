"""The single histogram filter's lane-per-item passes against the oracle, bit for bit: items, bin order,
weights and offsets at the edges of their groups (16, 32 and 64 items), segments (64 outputs) and
column blocks (16 columns), windows longer and shorter than a segment, ids over the whole 16-bit
range, more items than lanes (the line-by-line passes take over), and the capacity rule."""
import ctypes as C

import numpy as np
import pytest

from superterrainplus_amd import capi

from helpers import log
from test_gpu_shf import BIN, FilterBuffer, device_filter, host_filter

pytestmark = pytest.mark.gpu


def sample_map(seed, w, h, ids, patch, spread):
    """3 x 3 maps of ids in patch x patch squares; `spread` scatters them over 16 bits."""
    rng = np.random.default_rng(seed)
    m = rng.integers(0, ids, (-(-3 * h // patch), -(-3 * w // patch)))
    m = np.repeat(np.repeat(m, patch, 0), patch, 1)[:3 * h, :3 * w]
    return (m * 40503 % 65536 if spread else m).astype(np.uint16)


@pytest.mark.parametrize("w,h,r,ids,patch,cap,spread", [
    (2, 3, 2, 3, 1, 3, False), (63, 65, 2, 5, 1, 8, True), (64, 64, 8, 16, 1, 16, False), (65, 63, 8, 17, 1, 17, True),
    (17, 129, 16, 32, 1, 32, False), (130, 67, 16, 33, 1, 40, True), (81, 70, 32, 64, 1, 64, True),
    (200, 129, 2, 9, 7, 9, False), (257, 66, 6, 40, 13, 40, True), (150, 140, 140, 12, 3, 12, False), (72, 90, 20, 90, 9, 64, True),
    (300, 260, 4, 4, 64, 4, False)])
def test_lane_filter_matches_oracle(gpu, oracle, w, h, r, ids, patch, cap, spread):
    log(f"lane filter {w}x{h} r={r} ids={ids} patch={patch}")
    sample = sample_map(w * 1000 + h, w, h, ids, patch, spread)
    item, weight, off = oracle.shf_window(sample, (w, h), (w, h), r)
    buf = FilterBuffer(cap)
    # the second map runs in the same buffer, on what the first left there
    for m in (sample, sample[::-1].copy()):
        if m is not sample:
            item, weight, off = oracle.shf_window(m, (w, h), (w, h), r)
        gi, gw, go = host_filter(buf, m, (3, 3), (w, h), r)
        assert (go == off).all() and (gi == item).all() and gw.tobytes() == weight.tobytes()


@pytest.mark.parametrize("cap,ok", [(7, False), (8, False), (9, True)])
def test_lane_filter_capacity(gpu, oracle, cap, ok):
    """Columns of one id each, nine ids in turn: every window of 2r + 1 = 9 columns holds all nine."""
    log(f"lane filter capacity {cap}")
    w, h, r = 40, 24, 4
    ids = np.arange(3 * w) % 9
    sample = np.repeat(ids[None, :], 3 * h, 0).astype(np.uint16)
    buf = FilterBuffer(cap)
    if ok:
        item, weight, off = oracle.shf_window(sample, (w, h), (w, h), r)
        gi, gw, go = host_filter(buf, sample, (3, 3), (w, h), r)
        assert (go == off).all() and (gi == item).all() and gw.tobytes() == weight.tobytes()
    else:
        with pytest.raises(capi.STPError) as e:
            host_filter(buf, sample, (3, 3), (w, h), r)
        assert e.value.code == 4


def lane_path(out, w, h):
    """Whether the lane-per-item passes made this histogram: their bins lie right after their offsets (256-byte
    aligned), the line-by-line passes have a scan's sums between."""
    return out.Bin - out.HistogramStartOffset == (4 * (w * h + 1) + 255) // 256 * 256


def check_device(oracle, buf, m, w, h, r):
    item, weight, off = oracle.shf_window(m, (w, h), (w, h), r)
    d = capi.DeviceArray.from_host(m)
    out, n = device_filter(buf, d, (3, 3), (w, h), r)
    bins, offset = np.zeros(n, BIN), np.zeros(w * h + 1, np.uint32)
    capi.call("stp_memcpy_async", capi.ptr(bins), C.c_void_p(out.Bin), bins.nbytes, None)
    capi.call("stp_memcpy_async", capi.ptr(offset), C.c_void_p(out.HistogramStartOffset), offset.nbytes, None)
    capi.synchronize()
    assert (offset == off).all() and (bins["item"] == item).all() and bins["weight"].tobytes() == weight.tobytes()
    return lane_path(out, w, h)


@pytest.mark.parametrize("ids,cap,lanes", [(5, 8, True), (40, 8, True), (64, 12, True), (65, 12, False)])
def test_lane_filter_path(gpu, oracle, ids, cap, lanes):
    """Which passes take a map depends on its items, not on the bin capacity."""
    log(f"lane filter path ids={ids} cap={cap}")
    w, h, r = 48, 40, 2
    m = np.zeros((3 * h, 3 * w), np.uint16)
    # every id once in the window of samples, far enough apart that a pixel sees few
    for k in range(ids):
        m[h + 4 * (k // 11), w + 4 * (k % 11)] = k * 997 % 65536
    assert check_device(oracle, FilterBuffer(cap), m, w, h, r) == lanes


def test_lane_filter_after_a_crowded_map(gpu, oracle):
    """A buffer whose last map held too many items goes line by line until a map would have fitted."""
    w, h, r = 70, 50, 4
    crowded, plain = sample_map(3, w, h, 400, 4, True), sample_map(4, w, h, 6, 4, True)
    buf, way = FilterBuffer(40), []
    for k, m in enumerate((plain, crowded, crowded, plain, plain, crowded, plain)):
        log(f"lane filter after a crowded map {k}")
        way.append(check_device(oracle, buf, m, w, h, r))
    assert way == [True, False, False, False, True, False, False]
