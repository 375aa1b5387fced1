"""Copies between host arrays and the device: sizes around the pinned ring's chunks (512 KiB, 1 MiB, 4 MiB) and around
the sizes where it changes its way (2, 8, 24 and 32 MiB), byte arrays of odd lengths, host memory the runtime already
knows (pinned), and transfers that follow one another through the same ring."""
import ctypes
import threading

import numpy as np
import pytest

import scene
import splatx_hip as sh

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.mark.parametrize("nbytes", [4, 12, 512 * 1024 - 4, 512 * 1024, 512 * 1024 + 4, 2 * MIB - 4, 2 * MIB, 2 * MIB + 4,
                                    8 * MIB - 4, 8 * MIB + 4, 24 * MIB - 4, 24 * MIB + 4, 32 * MIB - 4, 33 * MIB + 4])
def test_scan_of_size(gpu, nbytes):
    # 4 B per element to the device, 8 B back
    print(f"bytes {nbytes}", flush=True)
    x = np.random.Generator(np.random.PCG64(nbytes)).integers(0, 100, nbytes // 4, dtype=np.int32)
    for _ in range(2):
        assert np.array_equal(gpu.prefix_scan_i64(x), np.cumsum(x, dtype=np.int64))
        x = x[::-1].copy()


@pytest.mark.parametrize("n", [1, 5, 1021, 524289])
def test_byte_masks(gpu, oracle, n):
    print(f"masks {n}", flush=True)
    rng = np.random.Generator(np.random.PCG64(n))
    dirs = rng.standard_normal((n, 3)).astype(np.float32)
    co = rng.standard_normal((n, 1, 3)).astype(np.float32)
    masks = (rng.random(n) < 0.5).astype(np.uint8)
    got = gpu.sh_fwd(dirs, co, 0, masks=masks)
    assert np.array_equal(got, oracle.sh_fwd(dirs, co, 0, masks=masks))


@pytest.mark.parametrize("rows", [5001, 30001, 65536, 65537, 70001, 200003])
def test_large_groups_and_pinned(gpu, rows):
    """Parameters and moments in one exchange, some of them in pinned memory, above and below the size at which the
    groups are staged together (65,536 rows), from a few MB on (copying threads, a copy engine)."""
    hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime the library has loaded
    pinned = []

    def empty(d, pin):
        if not pin:
            return np.empty((rows, d), np.float32)
        p = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(rows * d * 4), 0) == 0
        pinned.append(p)
        return np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_float)), (rows, d))

    print(f"rows {rows}", flush=True)
    dims = scene.group_dims(2)
    rng = np.random.Generator(np.random.PCG64(rows))
    ex = gpu.make_train_step_executor(arena_rows=rows, sh_degree=2)

    def arrays(fill):
        out = []
        for k in range(3):
            group = []
            for g, d in enumerate(dims):
                a = empty(d, (g + k) % 3 == 0)
                a[:] = rng.standard_normal((rows, d)) if fill else 0.0
                group.append(a)
            out.append(group)
        return out

    for _ in range(2):
        up, down = arrays(True), arrays(False)
        ex.upload_params(*up, rows)
        ex.download_params(*down, rows)
        for a, b in zip(up, down):
            for x, y in zip(a, b):
                assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
    ex.close()
    for p in pinned:
        hip.hipHostFree(p)


def test_null_group_is_refused_before_anything_moves(gpu):
    sc = scene.make_scene(n=300, sh_degree=1, width=64, height=48, fx=60.0, seed=3)
    ex = gpu.make_train_step_executor(arena_rows=sc.n, sh_degree=1)
    p, m, v = scene.copy_state(sc)
    ex.upload_params(p, m, v, sc.n)
    with pytest.raises(sh.SxInvalidArgument):
        ex.upload_params([x + 1 for x in p], m, [*v[:5], None], sc.n)
    got = scene.copy_state(sc)
    ex.download_params(*got, sc.n)
    ex.close()
    assert all(np.array_equal(x, y) for x, y in zip(got[0], p))


def test_backends_on_several_threads():
    """Backends of their own on three host threads at once: every ring, its threads and its kept buffers are its backend's."""
    n = 40_003
    dims = scene.group_dims(2)
    failed = []

    def work(seed):
        try:
            rng = np.random.Generator(np.random.PCG64(seed))
            b = sh.Backend(0)
            ex = b.make_train_step_executor(arena_rows=n, sh_degree=2)
            for k in range(4):
                up = [[rng.standard_normal((n, d)).astype(np.float32) for d in dims] for _ in range(3)]
                down = [[np.zeros((n, d), np.float32) for d in dims] for _ in range(3)]
                ex.upload_params(*up, n)
                x = rng.integers(0, 100, 300_007 * (seed + k + 1), dtype=np.int32)
                assert np.array_equal(b.prefix_scan_i64(x), np.cumsum(x, dtype=np.int64))
                ex.download_params(*down, n)
                for a, c in zip(up, down):
                    for y, z in zip(a, c):
                        assert np.array_equal(y.view(np.uint32), z.view(np.uint32))
            ex.close()
            b.close()
        except Exception as e:  # noqa: BLE001 (told by the test's thread)
            failed.append((seed, repr(e)))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
