"""The step's tile sort (u16 tile ids, positions as values, depths carried) where its plan changes: room for 65,536
intersections (tile counts without and with group sums), for 2^20 (tiles of 1024 and of 2048 keys) and for 2^22 (two
launches per pass, or a scanned count matrix), each on both sides, over images of 240 tiles (one pass, which leaves the
tile offsets), 256 and 272 (two passes). The steps fill that room to the last entry, pass it by one (the buffers grow),
and take a handful of entries and none in it."""
import numpy as np
import pytest

import oracle_py
import scene
import splatx_hip as sh

pytestmark = pytest.mark.gpu


def rows_of(sizes, tw, th, seed):
    """One row per entry of sizes: tw * th for a splat over the whole image, 1 for one within a tile."""
    n, w, h = len(sizes), 16 * tw, 16 * th
    p = scene.make_params(n, 0, seed)
    rng = np.random.Generator(np.random.PCG64(seed))
    z = rng.uniform(2.0, 6.0, n)
    z[rng.random(n) < 0.3] = 3.0  # equal depths go by the row
    one = np.asarray(sizes) == 1
    fx = 200.0
    px = np.where(one, 16 * rng.integers(0, tw, n) + 8.0, w / 2.0)
    py = np.where(one, 16 * rng.integers(0, th, n) + 8.0, h / 2.0)
    p[0][:] = np.stack([(px - w / 2.0) * z / fx, (py - h / 2.0) * z / fx, z], 1)
    p[2][:] = np.where(one, np.log(1e-3), np.log(600.0 * z / fx))[:, None]
    p[3][:] = -3.5
    return p, scene.pinhole(fx, fx, w / 2.0, h / 2.0)


def split(total, tiles, rng):
    """Sizes that add up to total, as few rows as there can be, mixed."""
    s = np.array([tiles] * (total // tiles) + [1] * (total % tiles))
    return list(rng.permutation(s))


@pytest.mark.parametrize("tw,th", [(16, 15), (16, 16), (17, 16)])
@pytest.mark.parametrize("first", [43_691, 43_692, 699_051, 699_052, 2_796_203, 2_796_204])
def test_capacity_edges(gpu, first, tw, th):
    print(f"first {first}, tiles {tw * th}", flush=True)
    tiles, w, h = tw * th, 16 * tw, 16 * th
    room = first + first // 2  # what the first step's growth leaves (65,536 at least)
    rng = np.random.Generator(np.random.PCG64(first))
    a = split(first, tiles, rng)
    b = split(room - first, tiles, rng)
    sizes = a + b + [1]
    n = len(sizes)
    p, K = rows_of(sizes, tw, th, first)
    gt = rng.uniform(0.0, 1.0, (h, w, 3)).astype(np.float32)
    at, away = scene.identity_view(), scene.identity_view()
    away[2, 3] = -30.0
    zero = [np.zeros_like(x) for x in p]
    base = dict(K=K, width=w, height=h, degrees_to_use=0, lr=[0.0] * 6, gt_rgb=gt)
    res = []
    for order in (sh.SXH_ISECT_ORDER_INDEX_FIRST, sh.SXH_ISECT_ORDER_DEPTH_FIRST):
        ex = gpu.make_train_step_executor(arena_rows=n, sh_degree=0, ssim_weight=0.0, isect_mode=sh.SXH_ISECT_AABB)
        ex.set_isect_order(order)
        ex.upload_params(p, zero, zero, n)
        out = []
        for count, vm in ((len(a), at), (len(a) + len(b), at), (3, at), (len(a), at), (len(a), away), (len(a) + len(b), at),
                          (n, at)):
            r = ex.step(want_render=True, viewmat=vm, count=count, **base)
            out.append((r["n_isects"], r["n_visible"], r["loss"], r["render_colors"].copy()))
        state = [[np.zeros_like(x) for x in p] for _ in range(3)]
        ex.download_params(*state, n)
        ex.close()
        res.append((out, state))
    (oa, sa), (ob, sb) = res
    want = [first, room, sum(sizes[:3]), first, 0, room, room + 1]
    assert [x[0] for x in oa] == want and [x[0] for x in ob] == want
    for x, y in zip(oa, ob):
        assert x[1:3] == y[1:3] and np.array_equal(x[3].view(np.uint32), y[3].view(np.uint32))
    for ga, gb in zip(sa, sb):
        for x, y in zip(ga, gb):
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
    assert np.abs(sa[1][0]).max() > 0
    ro = oracle_py.Oracle(libm=False).train_step(*[[x.copy() for x in g] for g in (p, zero, zero)], len(a), 0,
                                                 scene.identity_view(), K, w, h, gt, 0, [0.0] * 6, ssim_weight=0.0,
                                                 isect_mode=sh.SXH_ISECT_AABB, forward_only=True)
    assert ro["n_isects"] == first
    for k in (0, 3):
        assert np.array_equal(oa[k][3].view(np.uint32), ro["render_colors"].view(np.uint32))


@pytest.mark.parametrize("n", [900, 12_000])
def test_more_tiles_than_16_bits_hold(gpu, n):
    """65,792 tiles: the tile ids are u32 (17 bits, three passes, offsets by a pass of their own), with room for fewer
    intersections than the group sums begin at and for more."""
    w, h = 4112, 4096
    sc = scene.make_scene(n=n, sh_degree=0, width=w, height=h, fx=3700.0, seed=5, gt=None)
    p, m, v = scene.copy_state(sc)
    kw = scene.step_kwargs(sc)
    ro = oracle_py.Oracle(libm=False).train_step(p, m, v, n, 0, sc.viewmat, sc.K, w, h, None, 0, kw["lr"], forward_only=True)
    assert (ro["n_isects"] < 65_536) == (n == 900)
    for order in (sh.SXH_ISECT_ORDER_INDEX_FIRST, sh.SXH_ISECT_ORDER_DEPTH_FIRST):
        print(f"rows {n}, order {order}", flush=True)
        ex = gpu.make_train_step_executor(arena_rows=n, sh_degree=0, ssim_weight=0.2)
        ex.set_isect_order(order)
        ex.upload_params(p, m, v, n)
        for _ in range(2):
            r = ex.step(want_render=True, forward_only=True, **kw)
            assert r["n_isects"] == ro["n_isects"]
            assert np.array_equal(r["render_colors"].view(np.uint32), ro["render_colors"].view(np.uint32))
        ex.close()
