"""Sizes, offsets and rules that the host works out for the kernels, at the
ends of their ranges.  All CPU; no GPU calls."""
import ctypes

import pytest


@pytest.mark.parametrize("x,y,w", [
    (0, 0, 1), (46339, 46340, 46341), (46399, 46399, 46400), (65534, 32767, 65535), (0, 65534, 65535),
    (65534, 65534, 65535)])
def test_de_kernel_index_offset_past_2_31_cells(prod_lib, x, y, w):
    """Byte offset of a cell's kernel index in the density estimation's gather:
    two bytes a cell, beyond 32 bits from 2^31 cells on."""
    f = prod_lib.fl3k_de_findex_offset
    f.argtypes = [ctypes.c_int] * 3
    f.restype = ctypes.c_ulonglong
    assert f(x, y, w) == 2 * (x + y * w)


def test_deferred_counts_say_whether_they_failed(prod_lib):
    """fl3d_deferred_badvals returns its status beside the count, so that a
    failed wait is not a count of zero; nothing deferred is neither."""
    f = prod_lib.fl3d_deferred_badvals
    f.argtypes = [ctypes.POINTER(ctypes.c_double)]
    f.restype = ctypes.c_int
    n = ctypes.c_double(-1.0)
    assert f(ctypes.byref(n)) == 0 and n.value == 0.0


@pytest.mark.parametrize("rgb,per_item", [(1, 65536), (0, 81920)])
@pytest.mark.parametrize("records,chunk", [(1 << 28, 1 << 17), (1 << 31, 1 << 18), (32768, 16384)])
def test_partial_sums_are_those_of_the_accumulation_tiles(prod_lib, rgb, per_item, records, chunk):
    """Partial sums hold 4096 cells an item (16 bytes a cell, 20 with alphas),
    whatever tiles the walkers count: a 7716x4356 still of 2^28 records takes
    0.3 GB."""
    f = prod_lib.fl3k_bin_partial_bytes
    f.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_longlong]
    f.restype = ctypes.c_size_t
    assert f(rgb, chunk, records) == per_item * (2 * records // chunk + 1)


@pytest.mark.parametrize("records", [32768, 1 << 22, 8 << 20, 1 << 26, 1 << 28, 1 << 31])
@pytest.mark.parametrize("rgb", [0, 1])
def test_partial_sums_of_ordinary_items_have_room(prod_lib, rgb, records):
    """Items of 2^14 to 2^18 records as the launch's size sets them on 256 CUs;
    shorter ones (entries too bright for more) only while their sums take no more
    than 256 MiB and 8 bytes a record."""
    f = prod_lib.fl3k_bin_partial_bytes
    f.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_longlong]
    f.restype = ctypes.c_size_t
    chunk = min(max(records // 512 // 8192 * 8192, 16384), 1 << 18 if records > 1 << 30 else 1 << 17)
    room = (256 << 20) + 8 * records
    assert 0 < f(rgb, chunk, records) <= room
    for few in (1, 171, 5000):
        want = (81920, 65536)[rgb] * (2 * records // few + 1)
        assert f(rgb, few, records) in ((0, want) if abs(want / room - 1) < 0.01 else (want if want < room else 0,))


@pytest.mark.parametrize("lds,walkers", [
    (1000, 4096), (32767, 4096), (32769, 3072), (50000, 2048), (73728, 2048), (73729, 1024), (100000, 1024),
    (160000, 1024)])
def test_walkers_that_run_one_per_wavefront(prod_lib, lds, walkers):
    """fl3h_iterate takes a wavefront per walker up to four rounds (two beyond the
    classic variations) of those that a 256-CU chip of 160 KB LDS holds, at most four
    a CU (8 KB of LDS each beside the genome's)."""
    f = prod_lib.fl3k_lone_walkers
    f.argtypes = [ctypes.c_size_t, ctypes.c_size_t, ctypes.c_int, ctypes.c_int]
    f.restype = ctypes.c_int
    assert f(lds, 160 << 10, 256, 0) == walkers
    for tier in (1, 6):
        assert f(lds, 160 << 10, 256, tier) == walkers // 2


@pytest.mark.parametrize("k1,k2,finite", [
    (1068.0, 1 / 2000.0, 1), (-1068.0, 1 / 2000.0, 1), (0.0, 0.0, 1), (1e25, 1e10, 1), (1e27, 1e10, 0),
    (1068.0, -1 / 2000.0, 0), (1068.0, float("inf"), 0), (0.0, float("inf"), 0), (float("nan"), 1.0, 0),
    (1.0, float("nan"), 0), (float("inf"), 1.0, 0)])
def test_values_that_the_float_gather_may_multiply_by_zero(prod_lib, k1, k2, finite):
    """A 32-bit cell adds at most 2^32 k1 log(1 + 2^32 k2) to a channel: the
    production gather takes those below 1e38 only (1e25 and 1e10 give 1.9e36,
    100 times that is too much)."""
    f = prod_lib.fl3k_de_values_finite
    f.argtypes = [ctypes.c_double] * 2
    f.restype = ctypes.c_int
    assert f(k1, k2) == finite


@pytest.mark.parametrize("width,height,ok", [
    ((1 << 24) - 1, 2, 1), (1 << 24, 2, 0), (2, (1 << 24) - 1, 1), (1, 1 << 24, 0), (65535, 65535, 1), (1, 1, 1)])
def test_sides_that_records_can_hold(prod_lib, width, height, ok):
    """A record's cell is a 24-bit product of the width and the row: longer sides
    take direct deposits."""
    assert prod_lib.fl3k_record_sides(width, height) == ok
    low = (1 << 24) - 1
    assert ok == ((width & low) * (height & low) == width * height)


@pytest.mark.parametrize("rounds,njobs,tables,wave,samples", [
    (0, 1, 0, 1, 1 << 15), (0, 1000, 0, 1, 1 << 15), (0, 32, 1, 1, 1 << 15), (0, 33, 1, 1, 1 << 20),
    (0, 1000, 1, 1, 1 << 20), (1, 1, 0, 1, 1 << 20), (1, 1000, 1, 0, 1 << 20), (0, 1, 0, 0, 1 << 17),
    (0, 1000, 0, 0, 1 << 17), (0, 2, 1, 0, 1 << 20), (0, 33, 1, 0, 1 << 20)])
def test_samples_from_which_deposits_are_sorted(prod_lib, rounds, njobs, tables, wave, samples):
    """Launches of many jobs with a palette each, or of any with xaos, keep to the
    line of 2^20 samples; xaos and one palette to 2^17."""
    f = prod_lib.fl3k_bin_min_samples
    f.argtypes = [ctypes.c_int] * 4
    f.restype = ctypes.c_longlong
    assert f(rounds, njobs, tables, wave) == samples


@pytest.mark.parametrize("cap,need,fits", [
    (0, 1, 0), (4096, 4096, 1), (4096, 4097, 0), (128 << 20, 1, 1), ((128 << 20) + 1, 1, 0),
    (900 << 20, 64 << 20, 0), (900 << 20, (64 << 20) + 1, 1), (900 << 20, 900 << 20, 1), (900 << 20, 901 << 20, 0)])
def test_pinned_memory_is_given_back(prod_lib, cap, need, fits):
    """Pinned memory beyond 128 MiB lives until a call needs no more than half of that."""
    f = prod_lib.fl3k_pin_fits
    f.argtypes = [ctypes.c_size_t] * 2
    f.restype = ctypes.c_int
    assert f(cap, need) == fits
