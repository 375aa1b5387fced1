"""The key sort at the sizes where its plan changes: the edges of a tile (2048 and 4096 keys), of the tile counts
that are added up without group sums (64 tiles) and of whole groups of 32, of the small tiles (1,572,864 keys) and
of the two-launch passes (2^22 keys), with key widths of one to eight passes, keys that all fall into one digit,
and bits above key_n_bits that must not count."""
import numpy as np
import pytest

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
