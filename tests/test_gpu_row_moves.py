"""Rows moved between the arena's columns and the caller's row-major arrays: every group width (SH degrees 0 to 3)
at row counts around the moving kernels' blocks (64 and 256 rows), and a download from an arena in spatial order,
which puts each row in its caller's place and leaves the arena's order as it is."""
import numpy as np
import pytest

import scene
import splatx_hip as sh

pytestmark = pytest.mark.gpu


def bits(groups):
    return [np.asarray(x).view(np.uint32) for x in groups]


@pytest.mark.parametrize("deg", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [1, 63, 65, 256, 257, 1000])
def test_upload_download_round_trip(gpu, deg, n):
    print(f"rows {n}, degree {deg}", flush=True)
    rng = np.random.Generator(np.random.PCG64(n * 4 + deg))
    dims = scene.group_dims(deg)
    ex = gpu.make_train_step_executor(arena_rows=n + 7, sh_degree=deg)
    up = [[rng.standard_normal((n, d)).astype(np.float32) for d in dims] for _ in range(3)]
    ex.upload_params(*up, n)
    down = [[np.full((n + 7, d), np.nan, np.float32) for d in dims] for _ in range(3)]
    ex.download_params(*down, n)
    ex.close()
    for a, b in zip(up, down):
        for x, y in zip(bits(a), b):
            assert np.array_equal(x, y[:n].view(np.uint32))
            assert np.isnan(y[n:]).all()


@pytest.mark.parametrize("rows", [2500, 3000, 3100])
def test_download_from_spatial_order(gpu, rows):
    """A download of fewer rows than the live ones, of all, and of more, between steps: the same rows as from an
    arena in the caller's order, and the steps after it (and an upload over some or all of the rows) too."""
    sc = scene.make_scene(n=3100, sh_degree=2, width=96, height=64, fx=90.0, seed=71)
    n = 3000
    res = []
    for order in (sh.SXH_ROW_ORDER_ORIGINAL, sh.SXH_ROW_ORDER_SPATIAL):
        print(f"row order {order}, rows {rows}", flush=True)
        ex = gpu.make_train_step_executor(arena_rows=sc.n, sh_degree=sc.sh_degree, ssim_weight=0.2)
        ex.set_row_order(order)
        ex.upload_params(*scene.copy_state(sc), sc.n)
        kw = dict(scene.step_kwargs(sc), gt_rgb=sc.gt, count=n)
        out = []
        for k in range(3):
            ex.step(**kw)
            got = scene.copy_state(sc)
            for group in got:
                for x in group:
                    x[:] = 7.0
            ex.download_params(*got, rows)
            out.append(got)
        ex.upload_params(*scene.copy_state(sc), rows)
        ex.step(**kw)
        got = scene.copy_state(sc)
        ex.download_params(*got, sc.n)
        out.append(got)
        ex.close()
        res.append(out)
    for a, b in zip(*res):
        for ga, gb in zip(a, b):
            for x, y in zip(bits(ga), bits(gb)):
                assert np.array_equal(x, y)
