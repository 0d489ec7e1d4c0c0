"""Block lists at the sizes where row generation changes path: bins just below and at the
high-bin limit (1024 list positions), blocks at and beyond the promotion threshold (256),
sorting rounds of 1024 positions with a remainder, triangles from a fraction of a pixel to the
whole bin, and bins cut by the image edge. Bins, lists and fragment counts bit-exact, colours
within 1/255, as everywhere."""

import numpy as np
import pytest

from lucid_amd import _lib, scenes

from test_gpu_parity import _check, _render_both

pytestmark = pytest.mark.gpu


def _soup(n, w, h, size_px, seed):
    """n soup triangles inside the first bin (or the image), vertex offsets of size_px."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(1.0, min(31.0, w - 1, h - 1), (n, 1, 2))
    off = rng.normal(0.0, 1.0, (n, 3, 2)) * size_px
    ndc = (c + off + 0.5) / np.array([w, h]) * 2.0 - 1.0
    return scenes.soup_scene(w, h, ndc, rng.uniform(1.0, 90.0, n), rng.uniform(0, 1, (n, 3, 3)),
                             rng.uniform(0.05, 0.4, n), name=f"bin_{n}_{size_px}")


@pytest.mark.parametrize("opts", [0, _lib.OPT_FP32_SAMPLES])
@pytest.mark.parametrize("n,w,h,size_px", [
    (1, 8, 8, 40.0), (63, 33, 31, 12.0), (65, 40, 17, 0.6), (511, 32, 32, 2.0),
    (512, 32, 32, 2.0), (513, 37, 45, 6.0), (1025, 35, 33, 1.5), (5003, 41, 39, 3.0),
    (600, 64, 64, 60.0)])
def test_bin_sizes(oracle_mod, n, w, h, size_px, opts):
    sc = _soup(n, w, h, size_px, seed=n)
    r, gpu, ref = _render_both(sc, oracle_mod, opts=opts)
    _check(sc, gpu, ref, oracle_mod)


@pytest.mark.parametrize("n", [255, 256, 257, 300])
def test_promotion_threshold(oracle_mod, n):
    """n triangles that all cover one block of a low bin."""
    sc = scenes.block_stack(48, 40, n, center_px=(12, 12), size_px=6.0, seed=n)
    r, gpu, ref = _render_both(sc, oracle_mod)
    _check(sc, gpu, ref, oracle_mod)


@pytest.mark.parametrize("n", [64, 65, 128, 129, 512, 513, 2048, 2049, 4097])
def test_sort_lengths(oracle_mod, n):
    """n triangles over one block, at the lengths where its sort takes another path: one, two and
    four keys per lane, one 256-key chunk, several, and the long-list pass."""
    sc = scenes.block_stack(48, 40, n, center_px=(12, 12), size_px=6.0, seed=n)
    r, gpu, ref = _render_both(sc, oracle_mod)
    _check(sc, gpu, ref, oracle_mod)


@pytest.mark.parametrize("opts", [0, _lib.OPT_FP32_SAMPLES])
@pytest.mark.parametrize("w,h", [(1024, 1024), (1025, 1024)])
def test_raster_launch_threshold(oracle_mod, w, h, opts):
    """Frames at and just beyond the bin count up to which both kinds of blocks share a launch
    (1024 bins), with register-sorted and pre-sorted blocks: two stacks of different heights."""
    a = scenes.block_stack(w, h, 90, center_px=(500, 300), size_px=30.0, seed=1)
    b = scenes.block_stack(w, h, 1500, center_px=(w - 9, h - 9), size_px=9.0, seed=2)
    n = a.num_verts
    sc = scenes.block_stack(w, h, 1590, seed=3)
    sc.positions = np.concatenate([a.positions, b.positions])
    sc.colors_rgb = np.concatenate([a.colors_rgb, b.colors_rgb])
    sc.tri_alpha = np.concatenate([a.tri_alpha, b.tri_alpha])
    assert n + b.num_verts == sc.num_verts
    r, gpu, ref = _render_both(sc, oracle_mod, opts=opts)
    _check(sc, gpu, ref, oracle_mod)


def _stacks(w, h, per_bin, counts, seed):
    """`counts[i]` triangles over one block in the middle of bin i (row-major, 32 x 32 pixels)."""
    rng = np.random.default_rng(seed)
    bins = np.repeat(np.arange(len(counts)), counts)
    nbx = (w + 31) // 32
    c = np.stack([bins % nbx, bins // nbx], -1)[:, None] * 32.0 + 12.0
    off = np.array([[-3.0, -3.0], [4.0, -3.0], [-3.0, 4.0]]) + rng.uniform(-0.4, 0.4, (len(bins), 3, 2))
    ndc = (c + off + 0.5) / np.array([w, h]) * 2.0 - 1.0
    n = len(bins)
    return scenes.soup_scene(w, h, ndc, rng.uniform(1.0, 90.0, n), rng.uniform(0, 1, (n, 3, 3)),
                             rng.uniform(0.05, 0.4, n), name=f"stacks_{w}x{h}_{per_bin}")


def test_promoted_bins_overflow_the_lists(oracle_mod):
    """512 promoted bins, whose list space (16 lists of 1000 positions each) is more than a new
    renderer has: the frame is rendered again with larger lists."""
    sc = _stacks(1024, 512, 500, np.full(512, 500), seed=5)
    r, gpu, ref = _render_both(sc, oracle_mod)
    assert gpu["stats"]["high_bins"] >= 512
    _check(sc, gpu, ref, oracle_mod)


@pytest.mark.parametrize("w,h", [(2080, 1056), (1000, 37), (2500, 300)])
def test_many_bins(oracle_mod, w, h):
    """More bins than one step of the categorising work-group takes (2048), and rows of bins that
    end inside a step; empty, low, promoted and high bins mixed."""
    rng = np.random.default_rng(w)
    nb = ((w + 31) // 32) * (h // 32)
    counts = rng.choice([0, 1, 7, 300, 520], nb, p=[0.5, 0.2, 0.25, 0.03, 0.02])
    sc = _stacks(w, h, "mixed", counts, seed=w)
    r, gpu, ref = _render_both(sc, oracle_mod)
    _check(sc, gpu, ref, oracle_mod)


@pytest.mark.parametrize("make", [
    lambda: scenes.tilted_planes(2500, 2048, 3, seed=1),      # 79 x 64 bins, a wave per triangle
    lambda: scenes.tilted_planes(2560, 40, 5, seed=2),
    lambda: scenes.tilted_planes(40, 2000, 5, seed=3),
    lambda: scenes.config0(seed=8, num_tris=300, width=1000, height=700),
    lambda: scenes.config0(seed=9, num_tris=1024, width=700, height=500),
    lambda: scenes.config0(seed=9, num_tris=1025, width=700, height=500),  # two quads for some
    lambda: scenes.config0(seed=9, num_tris=8192, width=700, height=500),
    lambda: scenes.config0(seed=9, num_tris=30000, width=500, height=300),  # a thread per triangle
])
def test_large_triangles(oracle_mod, make):
    """Triangles over more than four bins, a few and many per work-group of the binning kernels,
    in frames of the most rows and columns of bins."""
    sc = make()
    r, gpu, ref = _render_both(sc, oracle_mod)
    _check(sc, gpu, ref, oracle_mod)


@pytest.mark.parametrize("opts", [0, _lib.OPT_FP32_SAMPLES])
@pytest.mark.parametrize("n", [2, 33, 63, 64, 65, 130])
def test_exact_pixel_lengths(oracle_mod, n, opts):
    """Pixels of n intersecting planes, around the length up to which their keys are sorted in
    registers (64)."""
    sc = scenes.tilted_planes(90, 60, n, seed=n)
    r, gpu, ref = _render_both(sc, oracle_mod, opts=opts)
    if n >= 63:
        assert gpu["stats"]["fallback_pixels"] > 0
    _check(sc, gpu, ref, oracle_mod)
