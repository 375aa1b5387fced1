"""The key sort at the sizes where its plan changes: the edges of a tile (2048 and 4096 keys), of the tile counts
that are added up without group sums (64 tiles) and of whole groups of 32, of the small tiles (1,572,864 keys) and
of the two-launch passes (2^22 keys), with key widths of one to eight passes, keys that all fall into one digit,
and bits above key_n_bits that must not count."""
import ctypes as C

import numpy as np
import pytest

import splatx_hip as sh
from test_zz_no_alloc import Hip, tile_depth_keys

pytestmark = pytest.mark.gpu


def check(gpu, keys, bits):
    vals = np.arange(keys.size, dtype=np.int32)
    ks, vs = gpu.sort_isect(keys, vals, bits)
    low = keys if bits == 64 else keys & np.uint64((1 << bits) - 1)
    order = np.argsort(low, kind="stable")
    assert np.array_equal(vs, order.astype(np.int32))
    assert np.array_equal(ks, keys[order])


@pytest.mark.parametrize("n", [1, 2, 511, 2047, 2048, 2049, 4097, 131071, 131072, 131073, 133121, 196609])
@pytest.mark.parametrize("bits", [1, 3, 9, 10, 33, 45, 64])
def test_tile_and_group_edges(gpu, n, bits):
    print(f"n {n}, bits {bits}", flush=True)
    rng = np.random.Generator(np.random.PCG64(n * 64 + bits))
    check(gpu, rng.integers(0, 1 << 63, n, dtype=np.uint64) * np.uint64(2) + rng.integers(0, 2, n, dtype=np.uint64), bits)


@pytest.mark.parametrize("n", [1572864, 1572865, 1 << 22, (1 << 22) + 1])
def test_plan_edges(gpu, n):
    print(f"n {n}", flush=True)
    rng = np.random.Generator(np.random.PCG64(n))
    tiles = rng.integers(0, 4346, n, dtype=np.uint64)
    depths = rng.uniform(0.5, 50.0, n).astype(np.float32).view(np.uint32).astype(np.uint64)
    check(gpu, (tiles << np.uint64(32)) | depths, 45)


@pytest.mark.parametrize("n", [5000, 140000])
def test_one_digit(gpu, n):
    print(f"n {n}", flush=True)
    check(gpu, np.full(n, 0x123456789ABC, np.uint64), 48)
    keys = np.full(n, 7, np.uint64)
    keys[n // 2] = 3
    check(gpu, keys, 32)


@pytest.mark.parametrize("bits", [45, 36])  # five passes and four: each buffer is read by some pass
@pytest.mark.parametrize("n", [1, 3, 2047, 2048, 2049, 131_073, 1_572_865])
def test_device_buffers_at_any_element(gpu, n, bits):
    """The allocation-free sort on arrays that begin one element into their allocations: aligned to a key and to a value,
    and to nothing more."""
    print(f"n {n}, bits {bits}", flush=True)
    hip = Hip()
    keys, vals = tile_depth_keys(np.random.Generator(np.random.PCG64(n)), n, bits)
    want_k, want_v = gpu.sort_isect(keys, vals, bits)
    f = gpu.lib.sxh_sort_isect_noalloc
    f.restype = C.c_int32
    f.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_int64, C.c_uint32, C.c_void_p, C.c_void_p]
    for shift in ((1, 1, 1, 1), (1, 0, 0, 0), (0, 0, 1, 0), (0, 1, 0, 1)):
        bufs = [hip.alloc(a.nbytes + 64) for a in (keys, vals, keys, vals)]
        try:
            at = [C.c_void_p(p.value + s * a.itemsize) for p, s, a in zip(bufs, shift, (keys, vals, keys, vals))]
            hip.h2d(at[0], keys)
            hip.h2d(at[1], vals)
            assert f(gpu.handle, at[0], at[1], n, bits, at[2], at[3]) == sh.SXH_OK, gpu.lib.sxh_last_error()
            ks, vs = np.zeros_like(keys), np.zeros_like(vals)
            hip.d2h(ks, at[2])
            hip.d2h(vs, at[3])
            assert np.array_equal(ks, want_k) and np.array_equal(vs, want_v), shift
        finally:
            for p in bufs:
                hip.free(p)
