"""A render session keeps clouds of 65,536 rows or more in spatial order: its frames against an executor's in the caller's
order, byte for byte, with many equal depths (ties go by the caller's row), below, at and above that size, first (depth
first) and later frames (index first), in both antialiasing modes."""
import numpy as np
import pytest

import scene
import splatx_hip as sh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,aa", [(65_535, False), (65_536, True), (70_001, False)])
def test_session_frames_in_spatial_order(gpu, tmp_path, n, aa):
    w, h, fx = 203, 117, 180.0
    sc = scene.make_scene(n=n, sh_degree=1, width=w, height=h, fx=fx, seed=3)
    p, m, v = scene.copy_state(sc)
    p[0][: n // 3, 2] = 4.0
    ex = gpu.make_train_step_executor(arena_rows=n, sh_degree=1, antialiased=aa)
    ex.upload_params(p, m, v, n)
    path = str(tmp_path / "cloud.ply")
    ex.export_ply(n, path, min_opacity=0.0, pad_sh_full=False)
    cl = sh.ply_read(path)  # (what the session reads)
    assert cl["count"] == n
    ex.upload_params([x.copy() for x in cl["params"]], m, v, n)
    session = gpu.render_session(path, antialiased=aa)
    try:
        rng = np.random.Generator(np.random.PCG64(1))
        for k in range(3):
            # the first view along the depth axis: the tied rows keep one depth
            vm = np.eye(4, dtype=np.float32) if k == 0 else scene.jittered_view(rng)
            K = scene.pinhole(fx, fx, w / 2.0, h / 2.0)
            for _ in range(2):
                r = ex.step(want_render=True, viewmat=vm, K=K, width=w, height=h, count=n, degrees_to_use=1,
                            lr=[0.0] * 6, forward_only=True)["render_colors"].reshape(h, w, 3)
                want = np.rint(np.where(r > 0, np.minimum(r, np.float32(1.0)), np.float32(0.0)) * np.float32(255.0))
                frame = session.frame(vm, fx, fx, w / 2.0, h / 2.0, w, h)
                assert np.array_equal(frame[..., :3], want.astype(np.uint8))
    finally:
        session.close()
        ex.close()
