"""The workloads whose speed this framework is measured by, through its public entry points.

Four kinds of work, over the sizes and options a program uses them with:

- `train`: a training segment. The cloud's rows and moments go to the executor, the caller loop runs
  `steps` iterations over the cameras (every target resident), and the rows and moments come back: what a
  trainer does between two events that need the cloud on the host. With `cap` the segment begins with the
  device MCMC refine and every step injects noise.
- `frames`: a render session's frames along a camera path, as RGBA8 images.
- `sort`: the allocation-free (tile, depth) key sort on device buffers.
- `ops`: the forward and backward of one view through the per-op entry points, on host arrays.

Scenes have the generators' distributions of the benchmark configurations: `plain` (a small or medium cloud in
front of the camera), `wide` (a large scene, many rows outside the view, splats of a few pixels), `dense`
(large splats, thousands of entries per tile, most of them behind opaque ones).
"""
from __future__ import annotations

import ctypes
import math
import os
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "splatx-metal_amd", "python"))

import scene  # noqa: E402
import splatx_hip as sh  # noqa: E402

# means x, y ~ U[-xy, xy], z ~ U[z0, z1]; log-scales ~ N(ln mu, sd); a share of means at one depth (tie);
# opacity logits ~ N(0, logit)
FAMILIES = {
    "plain": dict(xy=2.0, z0=2.0, z1=10.0, mu=0.02, sd=0.5, tie=0.0),
    "wide": dict(xy=4.0, z0=1.5, z1=20.0, mu=0.01, sd=0.7, tie=0.0),
    "dense": dict(xy=2.8, z0=2.0, z1=4.0, mu=0.08, sd=0.5, tie=0.1),
}


def listed():
    return [
        # a first look at a capture: a few thousand points, a thumbnail of odd size; launches are all of it
        dict(name="train_2k_97x61", kind="train", family="plain", n=2000, sh=1, w=97, h=61, fx=90.0, aabb=True,
             aa=False, ssim=0.2, cap=0, steps=50),
        # a small cloud, colour only, L1 loss
        dict(name="train_10k_256", kind="train", family="plain", n=10_000, sh=0, w=256, h=256, fx=230.0, aabb=True,
             aa=False, ssim=0.0, cap=0, steps=30),
        # an object capture
        dict(name="train_100k_800", kind="train", family="plain", n=100_000, sh=3, w=800, h=800, fx=720.0, aabb=True,
             aa=False, ssim=0.2, cap=0, steps=80),
        # a scene at full size, the headline configuration
        dict(name="train_1m_1297x840", kind="train", family="wide", n=1_000_000, sh=3, w=1297, h=840, fx=1150.0,
             aabb=False, aa=False, ssim=0.2, cap=0, steps=60),
        # the same with MCMC: 3 M of 4 M rows live, one refine and the steps after it, noise in each
        dict(name="train_mcmc_3m", kind="train", family="wide", n=3_000_000, sh=3, w=1297, h=840, fx=1150.0,
             aabb=False, aa=False, ssim=0.2, cap=4_000_000, steps=40),
        # large overlapping splats at full HD, antialiased, about 20 thousand entries per tile
        dict(name="train_dense_2m_1080p", kind="train", family="dense", n=2_000_000, sh=3, w=1920, h=1080, fx=1600.0,
             aabb=False, aa=True, ssim=0.2, cap=0, steps=30),
        # the viewer: an object at a window's size, and a full scene
        dict(name="frames_60k_641x479", kind="frames", family="plain", n=60_000, sh=3, w=641, h=479, fx=560.0, aa=False,
             frames=20),
        dict(name="frames_1m_1297x840", kind="frames", family="wide", n=1_000_000, sh=3, w=1297, h=840, fx=1150.0,
             aa=True, frames=10),
        # a serving loop's sort: a small view's entries, and near the entry point's limit
        dict(name="sort_70k", kind="sort", n=70_001, tiles=260),
        dict(name="sort_2m", kind="sort", n=2_000_000, tiles=4346),
        # a host trainer that calls op by op
        dict(name="ops_40k_640x360", kind="ops", family="plain", n=40_000, sh=3, w=640, h=360, fx=560.0, aabb=False,
             aa=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("train", "train", "train", "train", "frames", "sort", "ops"))
    if kind == "sort":
        return dict(kind="sort", n=_log(rng, 500, 2_000_000), tiles=_log(rng, 16, 8000))
    family = rng.choice(("plain", "wide", "dense")) if kind == "train" else rng.choice(("plain", "wide"))
    most = {"plain": 300_000, "wide": 1_500_000, "dense": 1_000_000}[family]
    if kind == "ops":
        most = 60_000
    n = _log(rng, 2000, most)
    w = _log(rng, 64, 720 if kind == "ops" else 1600)
    h = max(48, int(w * rng.uniform(0.45, 0.95)))
    c = dict(kind=kind, family=family, n=n, sh=rng.choice((0, 1, 2, 3, 3)), w=w, h=h, fx=round(w * rng.uniform(0.8, 1.0), 1),
             aa=rng.random() < 0.4)
    if kind == "frames":
        return dict(c, frames=10)
    c["aabb"] = rng.random() < 0.3
    if kind == "ops":
        return c
    mcmc = family != "dense" and rng.random() < 0.25
    return dict(c, ssim=rng.choice((0.0, 0.2, 0.2)), cap=int(n * 1.3) if mcmc else 0, steps=rng.randrange(20, 61) if family != "dense" else 20)


# ---- inputs --------------------------------------------------------------------------------------------

def _cloud(case, seed):
    """The six parameter groups as host arrays, drawn on the GPU."""
    f = FAMILIES[case["family"]]
    n = case["n"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=g)

    means = torch.rand(n, 3, device="cuda", generator=g)
    means[:, :2] = (means[:, :2] * 2.0 - 1.0) * f["xy"]
    means[:, 2] = f["z0"] + means[:, 2] * (f["z1"] - f["z0"])
    if f["tie"]:
        means[: int(n * f["tie"]), 2] = 0.5 * (f["z0"] + f["z1"])
    quats = normal(n, 4)
    quats /= quats.norm(dim=1, keepdim=True)
    # with MCMC a wider spread of opacities: about 5 % of the rows are dead
    groups = [means, quats, math.log(f["mu"]) + f["sd"] * normal(n, 3), normal(n) * (3.2 if case.get("cap") else 1.0),
              0.5 * normal(n, 3), 0.05 * normal(n, ((case["sh"] + 1) ** 2 - 1) * 3)]
    return [x.float().cpu().numpy() for x in groups]


def _views(seed, count):
    rng = np.random.Generator(np.random.PCG64(seed))
    return [scene.jittered_view(rng) for _ in range(count)]


N_VIEWS = 8
_backend = None


def _get_backend():
    global _backend
    if _backend is None:
        _backend = sh.Backend(0)
    return _backend


class _Owner(dict):
    """A state whose executor or session is given back with it."""

    def __del__(self):
        for k in ("ex", "session"):
            if self.get(k) is not None:
                self[k].close()


def _executor(case, rows):
    return _get_backend().make_train_step_executor(
        arena_rows=rows, sh_degree=case["sh"], ssim_weight=case.get("ssim", 0.2), antialiased=case["aa"],
        isect_mode=sh.SXH_ISECT_AABB if case.get("aabb") else sh.SXH_ISECT_ACCUTILE)


def _schedule(case, ex):
    """A 30,000-iteration run past its SH ramp: full degree, the default learning rates."""
    s = ex.train_schedule_defaults()
    s.total_iters = 30_000
    if case["cap"]:
        s.mcmc_enabled = 1
        s.cap_max = case["cap"]
        s.opacity_reg = s.scale_reg = 1e-2
    return s


START_ITER = 7001  # the steps between two refines (one every 100 iterations)


def _prepare_train(case, seed):
    n, w, h = case["n"], case["w"], case["h"]
    rows = max(case["cap"], n)
    ex = _executor(case, rows)
    K = scene.pinhole(case["fx"], case["fx"], w / 2.0, h / 2.0)
    views = _views(seed, N_VIEWS)
    # the targets: another cloud of the same family seen from the same cameras
    ex.set_gt_cache(np.zeros((N_VIEWS, h, w, 3), np.float32))
    p = _cloud(case, seed + 500_009)
    dims = scene.group_dims(case["sh"])
    pad = [np.zeros((rows, d), np.float32) for d in dims]
    m, v = [x.copy() for x in pad], [x.copy() for x in pad]
    ex.upload_params(p, m, v, n)
    for k, vm in enumerate(views):
        ex.render_to_gt_cache(k, viewmat=vm, K=K, width=w, height=h, count=n, degrees_to_use=case["sh"], lr=[0.0] * 6)
    out = [[x.copy() for x in pad] for _ in range(3)]
    s = _Owner(case=case, ex=ex, p=_cloud(case, seed), m=m, v=v, out=out,
               cams=[sh.TrainCamera.make(vm, K, w, h, k) for k, vm in enumerate(views)], sched=_schedule(case, ex))
    if case["cap"]:
        s["binoms"] = _get_backend().make_binoms_lut(51)
        s["rng0"] = _get_backend().mt64_seed(seed)
    return s


def _run_train(s):
    case, ex = s["case"], s["ex"]
    n = case["n"]
    ex.upload_params(s["p"], s["m"], s["v"], n)
    more = {}
    if case["cap"]:
        rng = s["rng0"].copy()
        r = ex.mcmc_refine(n, case["cap"], rng, s["binoms"], inject_noise=True, noise_seed=42, noise_offset=START_ITER - 1,
                           noise_scale=1.6e-4 * 5e5 * 0.01 ** (START_ITER / 30_000))
        n = r["count"]
        more = dict(rng=rng, binoms=s["binoms"])
    r = ex.train_loop(s["cams"], START_ITER, START_ITER + case["steps"], n, s["sched"], **more)
    p, m, v = s["out"]
    ex.download_params(p, m, v, n)
    live = [[x[:n] for x in group] for group in (p, m, v)]
    return dict(count=n, first_loss=r["first_loss"], last_loss=r["last_loss"], params=live[0], exp_avg=live[1],
                exp_avg_sq=live[2])


def _prepare_frames(case, seed):
    n = case["n"]
    ex = _executor(case, n)
    p = _cloud(case, seed)
    zero = [np.zeros_like(x) for x in p]
    ex.upload_params(p, zero, zero, n)
    with tempfile.TemporaryDirectory(prefix="splatx_frames_") as d:
        path = os.path.join(d, "cloud.ply")
        ex.export_ply(n, path, pad_sh_full=False)
        ex.close()
        session = _get_backend().render_session(path, antialiased=case["aa"])
    return _Owner(case=case, session=session, views=_views(seed, case["frames"]))


def _run_frames(s):
    c = s["case"]
    return [s["session"].frame(vm, c["fx"], c["fx"], c["w"] / 2.0, c["h"] / 2.0, c["w"], c["h"]) for vm in s["views"]]


def _prepare_sort(case, seed):
    n = case["n"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    # a Gaussian's tiles lie side by side: runs of neighbouring tile ids with one depth, index order
    start = torch.randint(0, case["tiles"], (n,), device="cuda", generator=g)
    run = torch.cumsum((torch.rand(n, device="cuda", generator=g) < 0.35).long(), 0)
    step = torch.arange(n, device="cuda") - torch.searchsorted(run, run)
    tile = (start[run] + step) % case["tiles"]
    depth = (1.5 + 18.5 * torch.rand(n, device="cuda", generator=g))[run].view(torch.int32).long()
    keys = (tile << 32) | depth
    values = torch.arange(n, device="cuda", dtype=torch.int32)
    f = _get_backend().lib.sxh_sort_isect_noalloc
    f.restype = ctypes.c_int32
    f.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int64, ctypes.c_uint32, ctypes.c_void_p,
                  ctypes.c_void_p]
    torch.cuda.synchronize()
    return dict(case=case, f=f, keys=keys, values=values, keys_out=torch.empty_like(keys),
                values_out=torch.empty_like(values), bits=32 + sh.bits_for_count(case["tiles"]))


def _run_sort(s):
    rc = s["f"](_get_backend().handle, s["keys"].data_ptr(), s["values"].data_ptr(), s["keys"].numel(), s["bits"],
                s["keys_out"].data_ptr(), s["values_out"].data_ptr())
    if rc != 0:
        raise RuntimeError(_get_backend().lib.sxh_last_error().decode())
    return s["keys_out"], s["values_out"]


def _prepare_ops(case, seed):
    p = _cloud(case, seed)
    n, w, h = case["n"], case["w"], case["h"]
    g = np.random.Generator(np.random.PCG64(seed))
    y, x = np.mgrid[0:h, 0:w]
    gt = np.stack([0.5 + 0.4 * np.sin(x * g.uniform(0.01, 0.2) + y * g.uniform(0.01, 0.2) + g.uniform(0, 6))
                   for _ in range(3)], -1).astype(np.float32)
    return dict(case=case, means=p[0], quats=p[1], scales=np.exp(p[2]), opacities=1.0 / (1.0 + np.exp(-p[3])),
                coeffs=np.concatenate([p[4][:, None, :], p[5].reshape(n, -1, 3)], 1), view=_views(seed, 1)[0],
                K=scene.pinhole(case["fx"], case["fx"], w / 2.0, h / 2.0), gt=gt[None])


def _run_ops(s):
    c, b = s["case"], _get_backend()
    n, w, h = c["n"], c["w"], c["h"]
    tw, th = (w + 15) // 16, (h + 15) // 16
    cam = dict(means=s["means"], quats=s["quats"], scales=s["scales"], viewmats=s["view"], Ks=s["K"], width=w, height=h,
               calc_compensations=c["aa"])
    pr = b.projection_fused_fwd(opacities=s["opacities"], **cam)
    valid = (pr["radii"][0].min(-1) > 0).astype(np.uint8)
    vm = s["view"]
    dirs = s["means"] - (-(vm[:3, :3].T @ vm[:3, 3])).astype(np.float32)
    pre = b.sh_fwd(dirs, s["coeffs"], c["sh"], masks=valid) + np.float32(0.5)
    colors = np.maximum(pre, np.float32(0.0))
    op = s["opacities"] * pr["compensations"][0] if c["aa"] else s["opacities"]
    tight = {} if c["aabb"] else dict(conics=pr["conics"], opacities=op)
    it = b.isect_tiles(pr["means2d"], pr["radii"], pr["depths"], 1, n, tw, th, **tight)
    keys, ids = b.sort_isect(it["isect_ids"], it["flatten_ids"], 32 + it["tile_n_bits"])
    offsets = b.isect_offset_encode(keys, 1, tw, th)
    rk = dict(means2d=pr["means2d"], conics=pr["conics"], colors=colors, opacities=op, isect_offsets=offsets,
              flatten_ids=ids, I=1, N=n, n_isects=ids.size, width=w, height=h, tile_width=tw, tile_height=th)
    r = b.rasterize_fwd(**rk)
    ss = b.ssim_fwd(r["render_colors"], s["gt"], need_coeffs=True)
    v_render = b.ssim_bwd(r["render_colors"], s["gt"], ss["coeff_mu"], ss["coeff_sigma"], ss["coeff_cross"])
    g = b.rasterize_bwd(r["render_alphas"], r["last_ids"], v_render, np.zeros_like(r["render_alphas"]), **rk)
    sg = b.sh_bwd(dirs, s["coeffs"], c["sh"], g["v_colors"] * (pre > 0), masks=valid)
    more, v_op = {}, g["v_opacities"]
    if c["aa"]:
        more = dict(compensations=pr["compensations"], v_compensations=v_op[None] * s["opacities"])
        v_op = v_op * pr["compensations"][0]
    pg = b.projection_fused_bwd(radii=pr["radii"], conics=pr["conics"], v_means2d=g["v_means2d"][None],
                                v_depths=np.zeros((1, n), np.float32), v_conics=g["v_conics"][None], **more, **cam)
    return dict(render=r["render_colors"][0], alpha=r["render_alphas"][0, ..., 0], ssim=ss["ssim"], v_render=v_render[0],
                v_means=pg["v_means"] + sg["v_dirs"], v_quats=pg["v_quats"], v_scales=pg["v_scales"], v_opacities=v_op,
                v_coeffs=sg["v_coeffs"])


def prepare(case, seed):
    return {"train": _prepare_train, "frames": _prepare_frames, "sort": _prepare_sort, "ops": _prepare_ops}[case["kind"]](
        case, seed)


def run(state):
    return {"train": _run_train, "frames": _run_frames, "sort": _run_sort, "ops": _run_ops}[state["case"]["kind"]](state)


# ---- what a pass cannot do without ------------------------------------------------------------------------

def _shares(case):
    """(share of the rows in view, intersections per row in view): the families' geometry in closed form, the
    splat's cutoff box against the tiles."""
    f = FAMILIES[case["family"]]
    seen, tiles, zs = 0.0, 0.0, 32
    for k in range(zs):
        z = f["z0"] + (k + 0.5) / zs * (f["z1"] - f["z0"])
        s = min(1.0, 0.5 * case["w"] / case["fx"] * z / f["xy"]) * min(1.0, 0.5 * case["h"] / case["fx"] * z / f["xy"])
        r = 2.5 * case["fx"] * f["mu"] * math.exp(0.5 * f["sd"] ** 2) / z + 0.5
        seen += s / zs
        tiles += s / zs * (2.0 * r / 16.0 + 1.0) ** 2
    return seen, tiles / seen * (0.9 if case.get("aabb") else 0.7)


def work(case):
    if case["kind"] == "sort":
        return {"bytes": 24.0 * case["n"], "flops": 0.0}
    n, px = case["n"], case["w"] * case["h"]
    seen, per = _shares(case)
    coeffs = 3 * (case["sh"] + 1) ** 2
    floats = 11 + coeffs
    isects = n * seen * per
    if case["kind"] == "frames":
        # every row's geometry, the colours of those in view, a list entry written and read per intersection
        one = 44.0 * n + n * seen * 4.0 * coeffs + 12.0 * min(isects, 1000.0 * px / 256) + 4.0 * px
        return {"bytes": case["frames"] * one, "flops": case["frames"] * 600.0 * min(isects, 1000.0 * px / 256)}
    if case["kind"] == "ops":
        return {"bytes": 4.0 * n * floats * 2 + 24.0 * isects + 100.0 * px, "flops": 3000.0 * isects}
    rows = n * 1.05 if case["cap"] else n
    # per step: parameters and moments of the rows in view (of all rows with noise: their geometry) read and
    # written, a list entry and its gradient per intersection that any pixel reaches, the image and its target
    reach = min(isects, 1000.0 * px / 256)
    one = 24.0 * floats * rows * seen + 44.0 * rows + 48.0 * reach + 60.0 * px
    return {"bytes": case["steps"] * one + 24.0 * floats * n, "flops": case["steps"] * 3000.0 * reach}


def tolerance(case):
    if case["kind"] in ("frames", "sort"):
        return "exact"
    if case["kind"] == "ops":
        # against 64 bits: 1.2e-4 in the SSIM gradient (differences of nearly equal sums), 1e-5 to 5e-5 elsewhere; in
        # another order of the gradients' sums 3e-7
        return {"rel": 5e-4, "max": 0.1}
    # Adam's step has the size of the learning rate whatever the gradient's, so where a gradient is near zero its
    # rounding decides the step, and a segment carries that on. With one unit in the last place on the log-scales and
    # logits at its start, the outputs after 40 steps are off by up to 0.006 (10 thousand rows), 0.003 (1 million), and by
    # 0.001 to 0.04 after 20 to 40 steps of the dense scene (its first moments), single values by their own size.
    return {"rel": 0.03, "max": 0.99}


# ---- the same in 64 bits ----------------------------------------------------------------------------------

def _sh64(deg, d, co):
    x, y, z = (d / d.norm(dim=1, keepdim=True)).unbind(1)
    b = [torch.full_like(x, 0.28209479177387814)]
    if deg >= 1:
        c = 0.4886025119029199
        b += [-c * y, c * z, -c * x]
    if deg >= 2:
        b += [1.0925484305920792 * x * y, -1.0925484305920792 * y * z, 0.31539156525252005 * (3 * z * z - 1),
              -1.0925484305920792 * x * z, 0.5462742152960396 * (x * x - y * y)]
    if deg >= 3:
        b += [-0.5900435899266435 * y * (3 * x * x - y * y), 2.890611442640554 * x * y * z,
              -0.4570457994644658 * y * (5 * z * z - 1), 0.3731763325901154 * z * (5 * z * z - 3),
              -0.4570457994644658 * x * (5 * z * z - 1), 1.445305721320277 * z * (x * x - y * y),
              -0.5900435899266435 * x * (x * x - 3 * y * y)]
    return (torch.stack(b, 1)[:, :, None] * co[:, : len(b)]).sum(1)


def _project64(case, vm, K, means, quats, scales, op):
    """means2d, conic, raster opacity, depth, radii (0: not in view)."""
    w, h = case["w"], case["h"]
    fx, fy, cx, cy = K[0, 0], K[1, 1], K[0, 2], K[1, 2]
    q = quats / quats.norm(dim=1, keepdim=True)
    qw, qx, qy, qz = q.unbind(1)
    R = torch.stack([1 - 2 * (qy * qy + qz * qz), 2 * (qx * qy - qw * qz), 2 * (qx * qz + qw * qy),
                     2 * (qx * qy + qw * qz), 1 - 2 * (qx * qx + qz * qz), 2 * (qy * qz - qw * qx),
                     2 * (qx * qz - qw * qy), 2 * (qy * qz + qw * qx), 1 - 2 * (qx * qx + qy * qy)], 1).reshape(-1, 3, 3)
    M = vm[:3, :3] @ (R * scales[:, None, :])
    t = means @ vm[:3, :3].T + vm[:3, 3]
    x, y, z = t.unbind(1)
    safe = torch.where(z > 0.01, z, torch.ones_like(z))
    limx, limy = 0.15 * w / fx, 0.15 * h / fy
    tx = safe * (x / safe).clamp(-(cx / fx + limx), (w - cx) / fx + limx)
    ty = safe * (y / safe).clamp(-(cy / fy + limy), (h - cy) / fy + limy)
    zero = torch.zeros_like(safe)
    J = torch.stack([fx / safe, zero, -fx * tx / safe ** 2, zero, fy / safe, -fy * ty / safe ** 2], 1).reshape(-1, 2, 3)
    V = J @ M
    c00, c01, c11 = (V[:, 0] ** 2).sum(1), (V[:, 0] * V[:, 1]).sum(1), (V[:, 1] ** 2).sum(1)
    det0 = c00 * c11 - c01 * c01
    c00, c11 = c00 + 0.3, c11 + 0.3
    det = c00 * c11 - c01 * c01
    if case["aa"]:
        op = op * (det0 / det).clamp(min=0.005 ** 2).sqrt()
    m2 = torch.stack([fx * x / safe + cx, fy * y / safe + cy], 1)
    conic = torch.stack([c11 / det, -c01 / det, c00 / det], 1)
    with torch.no_grad():
        ext = torch.sqrt(2 * torch.log((op * 255).clamp(min=1.0))).clamp(max=3.33)
        rad = torch.stack([torch.ceil(ext * c00.sqrt()), torch.ceil(ext * c11.sqrt())], 1)
        size = torch.tensor([w, h], device=m2.device, dtype=m2.dtype)
        ok = (z >= 0.01) & (op * 255 >= 1) & (rad.min(1).values > 0) & ((m2 + rad > 0) & (m2 - rad < size)).all(1)
        rad = torch.where(ok[:, None], rad, torch.zeros_like(rad))
    return m2, conic, op, z, rad


def _batches64(case, m2, z, rad):
    """Tiles with their rows in depth order, in batches padded to one length: (tile ids, rows, real)."""
    tw, th = (case["w"] + 15) // 16, (case["h"] + 15) // 16
    top = torch.tensor([tw, th], device=m2.device)
    rows = torch.argsort(z, stable=True)
    rows = rows[rad[rows, 0] > 0]
    lo = torch.minimum(((m2[rows] - rad[rows]) / 16).floor().long().clamp(min=0), top)
    hi = torch.minimum(((m2[rows] + rad[rows]) / 16).ceil().long().clamp(min=0), top)
    wide, count = hi[:, 0] - lo[:, 0], (hi - lo).prod(1)
    first = torch.cumsum(count, 0) - count
    own = torch.repeat_interleave(torch.arange(rows.numel(), device=m2.device), count)
    k = torch.arange(own.numel(), device=m2.device) - first[own]
    tile = (lo[own, 1] + k // wide[own]) * tw + lo[own, 0] + k % wide[own]
    order = torch.argsort(tile, stable=True)
    ids, tile = rows[own[order]], tile[order]
    n_of = torch.bincount(tile, minlength=tw * th)
    start = torch.cumsum(n_of, 0) - n_of
    by = torch.argsort(n_of, descending=True)
    sizes = n_of[by].tolist()
    at = 0
    while at < len(sizes) and sizes[at] > 0:
        size = sizes[at]
        many = max(1, 120_000 // size)
        t = by[at: at + many]
        j = torch.arange(size, device=m2.device)[None]
        real = j < n_of[t][:, None]
        yield t, ids[torch.where(real, start[t][:, None] + j, torch.zeros_like(j))], real
        at += many


def _tiles64(case, t, rows, real, m2, conic, op, color):
    """(colour, alpha) of the pixels of tiles t, 256 each."""
    tw = (case["w"] + 15) // 16
    k = torch.arange(256, device=m2.device)
    px = (t % tw)[:, None] * 16 + k % 16 + 0.5
    py = torch.div(t, tw, rounding_mode="floor")[:, None] * 16 + torch.div(k, 16, rounding_mode="floor") + 0.5
    dx = m2[rows, 0][:, None, :] - px[:, :, None]
    dy = m2[rows, 1][:, None, :] - py[:, :, None]
    c = conic[rows]
    sigma = 0.5 * (c[:, None, :, 0] * dx * dx + c[:, None, :, 2] * dy * dy) + c[:, None, :, 1] * dx * dy
    alpha = (op[rows][:, None, :] * torch.exp(-sigma)).clamp(max=0.99)
    alpha = torch.where((sigma >= 0) & (alpha >= 1.0 / 255.0) & real[:, None, :], alpha, torch.zeros_like(alpha))
    after = torch.cumsum(torch.log1p(-alpha), 2)
    kept = torch.where(after > math.log(1e-4), alpha, torch.zeros_like(alpha))
    before = torch.cat([torch.zeros_like(after[:, :, :1]), after[:, :, :-1]], 2)
    weight = kept * torch.exp(before)
    return weight @ color[rows], weight.sum(2)


def _tile_image(case, img):
    """An image [h, w, c] as [tiles, 256, c], zero outside."""
    tw, th = (case["w"] + 15) // 16, (case["h"] + 15) // 16
    full = img.new_zeros(th * 16, tw * 16, img.shape[2])
    full[: case["h"], : case["w"]] = img
    return full.reshape(th, 16, tw, 16, -1).transpose(1, 2).reshape(th * tw, 256, -1)


def _image_of(case, tiles):
    tw, th = (case["w"] + 15) // 16, (case["h"] + 15) // 16
    return tiles.reshape(th, tw, 16, 16, -1).transpose(1, 2).reshape(th * 16, tw * 16, -1)[: case["h"], : case["w"]]


def _ssim64(a, b):
    k = torch.arange(11, device=a.device, dtype=a.dtype) - 5
    g = torch.exp(-k * k / (2 * 1.5 ** 2))
    g = g / g.sum()

    def blur(x):
        x = x.permute(2, 0, 1)[:, None]
        return torch.nn.functional.conv2d(torch.nn.functional.conv2d(x, g.reshape(1, 1, 1, 11)), g.reshape(1, 1, 11, 1))

    ma, mb = blur(a), blur(b)
    va, vb, vab = blur(a * a) - ma * ma, blur(b * b) - mb * mb, blur(a * b) - ma * mb
    return ((2 * ma * mb + 1e-4) * (2 * vab + 9e-4) / ((ma * ma + mb * mb + 1e-4) * (va + vb + 9e-4))).mean()


def _view64(case, vm, K, leaves, loss_of):
    """One view in 64 bits: the render and what `loss_of(render)` leaves in the gradients of `leaves` = (means, quats,
    linear scales, activated opacities, SH coefficients). loss_of None: forward only."""
    means, quats, scales, op, co = leaves
    m2, conic, rop, z, rad = _project64(case, vm, K, means, quats, scales, op)
    campos = -(vm[:3, :3].T @ vm[:3, 3])
    color = (_sh64(case["sh"], means - campos, co) + 0.5).clamp(min=0)
    flat = [x.detach().requires_grad_(loss_of is not None) for x in (m2, conic, rop, color)]
    tiles = (case["w"] + 15) // 16 * ((case["h"] + 15) // 16)
    rgb, alpha = m2.new_zeros(tiles, 256, 3), m2.new_zeros(tiles, 256, 1)
    batches = list(_batches64(case, m2.detach(), z.detach(), rad))
    with torch.no_grad():
        for t, rows, real in batches:
            rgb[t], a = _tiles64(case, t, rows, real, *flat)
            alpha[t] = a[:, :, None]
    img = _image_of(case, rgb).clone().requires_grad_(loss_of is not None)
    alpha = _image_of(case, alpha)[..., 0]
    if loss_of is None:
        return img, alpha, None, None, rad
    loss = loss_of(img)
    loss.backward()
    v = _tile_image(case, img.grad)
    for t, rows, real in batches:
        _tiles64(case, t, rows, real, *flat)[0].backward(v[t])
    torch.autograd.backward([m2, conic, rop, color], [x.grad if x.grad is not None else torch.zeros_like(x) for x in flat])
    return img.detach(), alpha, loss.detach(), img.grad, rad


def _exact_train(case, seed):
    f = FAMILIES[case["family"]]
    pairs = 256.0 * case["n"] * _shares(case)[0] * _shares(case)[1]
    if case["cap"] or f["tie"] or pairs * case["steps"] > 6e9:
        return None
    up = lambda x: torch.tensor(np.asarray(x), device="cuda", dtype=torch.float64)  # noqa: E731
    K = up(scene.pinhole(case["fx"], case["fx"], case["w"] / 2.0, case["h"] / 2.0))
    views = [up(v) for v in _views(seed, N_VIEWS)]
    n = case["n"]

    def leaves(p):
        return p[0], p[1], torch.exp(p[2]), torch.sigmoid(p[3]), torch.cat([p[4][:, None, :], p[5].reshape(n, -1, 3)], 1)

    with torch.no_grad():
        target = [up(x) for x in _cloud(case, seed + 500_009)]
        gts = [_view64(case, vm, K, leaves(target), None)[0] for vm in views]
    p = [up(x) for x in _cloud(case, seed)]
    m, v = [torch.zeros_like(x) for x in p], [torch.zeros_like(x) for x in p]
    lam = case["ssim"]
    losses = []
    for it in range(START_ITER, START_ITER + case["steps"]):
        gt = gts[it % N_VIEWS]

        def loss_of(img, gt=gt):
            one = (img - gt).abs().mean()
            return one if lam == 0 else (1 - lam) * one + lam * (1 - _ssim64(img, gt))

        q = [x.detach().requires_grad_(True) for x in p]
        _, _, loss, _, rad = _view64(case, views[it % N_VIEWS], K, leaves(q), loss_of)
        losses.append(float(loss))
        lr = [1.6e-4 * 0.01 ** (it / 30_000), 1e-3, 5e-3, 5e-2, 2.5e-3, 2.5e-3 / 20]
        seen = rad[:, 0] > 0
        with torch.no_grad():
            for g in range(6):
                if p[g].numel() == 0:
                    continue
                grad = q[g].grad
                s = seen if p[g].dim() == 1 else seen[:, None]
                m[g] = torch.where(s, 0.9 * m[g] + 0.1 * grad, m[g])
                v[g] = torch.where(s, 0.999 * v[g] + 0.001 * grad * grad, v[g])
                p[g] = torch.where(s, p[g] - lr[g] * m[g] / (v[g].sqrt() + 1e-15), p[g])
    host = lambda xs: [(x[:, None] if x.dim() == 1 else x).cpu().numpy() for x in xs]  # noqa: E731
    return dict(count=None, first_loss=losses[0], last_loss=losses[-1], params=host(p), exp_avg=host(m), exp_avg_sq=host(v))


def _exact_ops(case, seed):
    s = _prepare_ops(case, seed)
    up = lambda x: torch.tensor(np.asarray(x), device="cuda", dtype=torch.float64)  # noqa: E731
    q = [up(s[k]).requires_grad_(True) for k in ("means", "quats", "scales", "opacities", "coeffs")]
    gt = up(s["gt"][0])
    img, alpha, loss, v_render, _ = _view64(case, up(s["view"]), up(s["K"]), q, lambda i: 1 - _ssim64(i, gt))
    host = lambda x: x.detach().cpu().numpy()  # noqa: E731
    return dict(render=host(img), alpha=host(alpha), ssim=1.0 - float(loss), v_render=host(v_render), v_means=host(q[0].grad),
                v_quats=host(q[1].grad), v_scales=host(q[2].grad), v_opacities=host(q[3].grad), v_coeffs=host(q[4].grad))


def exact(case, seed):
    if case["kind"] == "train":
        return _exact_train(case, seed)
    return _exact_ops(case, seed) if case["kind"] == "ops" else None
