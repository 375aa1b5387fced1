"""Index-first steps of up to 1024 preprocess blocks (262,144 rows) do the block scan in the emit's launch; larger clouds
and depth-first steps launch it. Around that count, and for a single block, both orders must give the same counts,
losses and arena bit for bit, through a step that overflows the intersection buffers and one without any."""
import numpy as np
import pytest

import scene
import splatx_hip as sh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 257, 262144, 262145])
def test_fold_matches_scan(gpu, n):
    print(f"rows {n}", flush=True)
    sc = scene.make_scene(n=n, sh_degree=0, width=80, height=64, fx=70.0, seed=n)
    away = scene.identity_view()
    away[2, 3] = -30.0
    res = []
    for order in (sh.SXH_ISECT_ORDER_INDEX_FIRST, sh.SXH_ISECT_ORDER_DEPTH_FIRST):
        ex = gpu.make_train_step_executor(arena_rows=n, sh_degree=0, ssim_weight=0.2)
        ex.set_isect_order(order)
        ex.upload_params(*scene.copy_state(sc), n)
        out = []
        for vm in (scene.identity_view(), away, scene.identity_view()):
            r = ex.step(**dict(scene.step_kwargs(sc), viewmat=vm, gt_rgb=sc.gt))
            out.append((r["loss"], r["n_isects"], r["n_visible"]))
        state = scene.copy_state(sc)
        ex.download_params(*state, n)
        ex.close()
        res.append((out, state))
    (oa, sa), (ob, sb) = res
    assert oa == ob and oa[1][1] == 0
    for ga, gb in zip(sa, sb):
        for x, y in zip(ga, gb):
            assert np.array_equal(x.view(np.uint32), y.view(np.uint32))
