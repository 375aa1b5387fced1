"""The rasterisers on images of few tiles (the forward has a wave per 4x4 pixel block there) and around the tile count
where it changes to four waves a tile (512): lists around the batch (512 entries) and chunk (4) edges, where a pixel's
transmittance is spent within a chunk, colours that a zero weight would not cancel, masks, backgrounds and several
images."""
import numpy as np
import pytest

import inputs
from test_gpu_ops import extreme_splats, rel_l2, same_bits

pytestmark = pytest.mark.gpu


def check(gpu, oracle, kw, grads=True):
    a, b = gpu.rasterize_fwd(**kw), oracle.rasterize_fwd(**kw)
    for k in ("render_colors", "render_alphas", "last_ids"):
        assert same_bits(a[k], b[k]), k
    if not grads:
        return
    r = inputs.rng(5)
    gin = dict(render_alphas=b["render_alphas"], last_ids=b["last_ids"],
               v_render_colors=r.standard_normal(b["render_colors"].shape).astype(np.float32),
               v_render_alphas=r.standard_normal(b["render_alphas"].shape).astype(np.float32))
    ga, gb = gpu.rasterize_bwd(**gin, **kw), oracle.rasterize_bwd(**gin, **kw)
    for k in ("v_means2d", "v_conics", "v_colors", "v_opacities"):
        assert rel_l2(ga[k], gb[k]) <= 1e-4, (k, rel_l2(ga[k], gb[k]))


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 31, 33, 255, 257, 511, 512, 513, 1025])
def test_list_lengths(gpu, oracle, n):
    print(f"entries {n}", flush=True)
    check(gpu, oracle, extreme_splats(50 + n, n=n, width=37, height=21))


@pytest.mark.parametrize("size", [(512, 256), (513, 256), (432, 304)])  # 512, 528 and 513 tiles
def test_tile_counts(gpu, oracle, size):
    print(f"size {size}", flush=True)
    check(gpu, oracle, extreme_splats(7, n=150, width=size[0], height=size[1]))


@pytest.mark.parametrize("opacity", [0.3, 0.9, 0.99])
def test_spent_within_a_chunk(gpu, oracle, opacity):
    """Opaque splats over every pixel: T runs out after a number of entries that differs between pixels."""
    kw = extreme_splats(8, n=600, width=40, height=24)
    kw["opacities"] = np.full_like(kw["opacities"], opacity)
    kw["conics"] = np.tile(np.array([0.002, 0.0005, 0.003], np.float32), (1, 600, 1))
    check(gpu, oracle, kw)


@pytest.mark.parametrize("n", [63, 64, 65, 127, 129, 255, 256, 257, 321])
def test_backward_segments(gpu, oracle, n):
    """Faint splats over every pixel: each block's list holds all entries, around two segments (32 each) and
    the batch (256) of the backward. The sums run over 16 pixels and 16 blocks in 32 bits, T over n factors: below 1e-4."""
    kw = extreme_splats(20 + n, n=n, width=33, height=18)
    kw["opacities"] = np.full_like(kw["opacities"], 0.02)
    kw["conics"] = np.tile(np.array([0.002, 0.0005, 0.003], np.float32), (1, n, 1))
    check(gpu, oracle, kw)


def test_colours_not_finite(gpu, oracle):
    kw = extreme_splats(9, n=300, width=48, height=32)
    c = kw["colors"].copy()
    c[0, 10:40:6, 0], c[0, 12:60:9, 1], c[0, 11:60:4, 2] = np.inf, -np.inf, np.nan
    kw["colors"] = c
    a, b = gpu.rasterize_fwd(**kw), oracle.rasterize_fwd(**kw)
    assert same_bits(a["render_alphas"], b["render_alphas"]) and same_bits(a["last_ids"], b["last_ids"])
    x, y = a["render_colors"], b["render_colors"]
    assert np.isnan(y).any() and np.isinf(y).any() and np.isfinite(y).any()
    assert np.array_equal(np.isnan(x), np.isnan(y))
    assert same_bits(np.nan_to_num(x, nan=0.0), np.nan_to_num(y, nan=0.0))


def test_images_masks_backgrounds(gpu, oracle):
    check(gpu, oracle, inputs.raster_kwargs(oracle, n=900, seed=11, I=2, width=75, height=45, backgrounds=True, masks=True))


@pytest.mark.parametrize("n", [1, 3, 5, 63, 65, 300, 1000])
def test_same_bits_among_many_images(gpu, n):
    """One image of six tiles, and the same image 100 times in one call (600 tiles): the forward and the gradients of an
    image do not depend on the tiles beside it, bit for bit. Each tile lists splats of its own, so that every gradient
    is one sum of one tile and no order of atomic adds enters."""
    print(f"entries {n}", flush=True)
    many, w, h, tiles = 100, 44, 29, 6
    one = extreme_splats(70 + n, n=tiles * n, width=w, height=h)
    one["flatten_ids"] = np.arange(tiles * n, dtype=np.int32)
    one["isect_offsets"] = (np.arange(tiles, dtype=np.int32) * n).reshape(1, 2, 3)
    one["n_isects"] = tiles * n
    all_ = dict(one, I=many, n_isects=many * tiles * n)
    for k in ("means2d", "conics", "colors", "opacities"):
        all_[k] = np.repeat(one[k], many, 0)
    for k in ("flatten_ids", "isect_offsets"):
        step = np.arange(many, dtype=np.int32) * (tiles * n)
        all_[k] = (one[k].reshape(1, -1) + step[:, None]).astype(np.int32)
    all_["flatten_ids"] = all_["flatten_ids"].ravel()
    all_["isect_offsets"] = all_["isect_offsets"].reshape(many, 2, 3)
    a, b = gpu.rasterize_fwd(**one), gpu.rasterize_fwd(**all_)
    r = inputs.rng(5)
    v_c = r.standard_normal(a["render_colors"].shape).astype(np.float32)
    v_a = r.standard_normal(a["render_alphas"].shape).astype(np.float32)
    ga = gpu.rasterize_bwd(a["render_alphas"], a["last_ids"], v_c, v_a, **one)
    gb = gpu.rasterize_bwd(b["render_alphas"], b["last_ids"], np.repeat(v_c, many, 0), np.repeat(v_a, many, 0), **all_)
    assert np.abs(ga["v_means2d"]).max() > 0
    for k in range(many):
        assert same_bits(a["render_colors"][0], b["render_colors"][k]) and same_bits(a["render_alphas"][0], b["render_alphas"][k])
        # (positions in the list, from the image's first; a pixel no splat reached reads 0 in every image)
        assert np.array_equal(np.where(a["render_alphas"][0, ..., 0] > 0, a["last_ids"][0] + k * tiles * n, 0), b["last_ids"][k])
    for k in ("v_means2d", "v_conics", "v_colors", "v_opacities"):
        x = gb[k].reshape(many, *ga[k].shape)
        for q in range(many):
            assert same_bits(ga[k], x[q]), (k, q)


def test_backward_far_into_the_list(gpu):
    """A tile whose list begins past entry 2^27 of the intersections (the entries before it belong to a masked tile, which
    is skipped): the same gradients, bit for bit, as with the list at the start. The image cuts through its 4x4 blocks,
    whose pixels outside must take no part."""
    n, far, w, h = 300, (1 << 27) + 5, 18, 11
    kw = extreme_splats(12, n=n, width=w, height=h)
    kw.update(masks=np.array([[[0, 1]]], np.uint8), isect_offsets=np.zeros((1, 1, 2), np.int32),
              flatten_ids=np.arange(n, dtype=np.int32), n_isects=n)
    ids = np.zeros(far + n, np.int32)
    ids[far:] = kw["flatten_ids"]
    moved = dict(kw, isect_offsets=np.array([[[0, far]]], np.int32), flatten_ids=ids, n_isects=far + n)
    r = inputs.rng(5)
    v_c, v_a = r.standard_normal((1, h, w, 3)).astype(np.float32), r.standard_normal((1, h, w, 1)).astype(np.float32)
    g = []
    for k in (kw, moved):
        f = gpu.rasterize_fwd(**k)
        g.append((f, gpu.rasterize_bwd(f["render_alphas"], f["last_ids"], v_c, v_a, **k)))
    assert same_bits(g[0][0]["render_colors"], g[1][0]["render_colors"])
    assert np.abs(g[0][1]["v_means2d"]).max() > 0
    for k in ("v_means2d", "v_conics", "v_colors", "v_opacities"):
        assert same_bits(g[0][1][k], g[1][1][k]), k
