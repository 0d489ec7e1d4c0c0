"""The ordering windows decide only which pixels take the exact sort, never a result: fp32 frames
whose blocks are pre-sorted (their depth ranges are composited apart and chained), the window knob
on records that are not flat, and batches that mix frames with and without the alpha threshold."""

import numpy as np
import pytest

from lucid_amd import _lib, scenes

pytestmark = pytest.mark.gpu


def _planes(n, w, h, slope, alpha, seed, color_format="f32"):
    """n screen-filling quads at even depths, with slopes that make near neighbours cross. alpha: a
    range, or the alphas from the nearest on."""
    rng = np.random.default_rng(seed)
    corners = np.array([[-1.3, -1.2], [1.2, -1.3], [1.3, 1.2], [-1.2, 1.3]])
    ndc = np.repeat(corners[None], n, axis=0)
    k = rng.uniform(-slope, slope, (n, 2))
    rank = rng.permutation(n)
    depth = 10.0 + 0.05 * rank[:, None] + corners[:, 0] * k[:, :1] + corners[:, 1] * k[:, 1:]
    a = alpha[rank] if isinstance(alpha, np.ndarray) else rng.uniform(*alpha, n)
    return scenes.quad_soup_scene(w, h, ndc, depth, rng.uniform(0.0, 1.0, (n, 4, 3)), a,
                                  color_format=color_format, name=f"crossing_{n}")


def _render(sc, opts, window, runs=1):
    from lucid_amd.renderer import GpuScene, LucidRenderer
    print(f"\n[case] {sc.name} {sc.width}x{sc.height} opts={opts:#x} window={window}", flush=True)
    r = LucidRenderer((sc.width, sc.height), opts=opts)
    r.set_tuning(window=window)
    outs = []
    for _ in range(runs):
        out = r.render(GpuScene(sc), r.alloc_outputs(rgba8=True, rgba32f=True, counts=True))
        outs.append({k: v.cpu().numpy() for k, v in out.items()})
    return outs, r.get_stats()


@pytest.mark.parametrize("blend", [0, _lib.OPT_ADDITIVE_BLENDING])
@pytest.mark.parametrize("n,slope", [(320, 0.12), (700, 0.2)])
def test_fp32_presorted_blocks_keep_their_bits(n, slope, blend):
    """Blocks of more entries than the register sort takes, in which some pixels are out of order
    for one slot and not for four: the same bits with either window, and from run to run."""
    sc = _planes(n, 64, 48, slope, (0.4 / n, 2.0 / n), seed=n)
    opts = blend | _lib.OPT_FP32_SAMPLES
    (ref,), wide = _render(sc, opts, 4)
    assert wide["block_tris"] > 256 * 48 and wide["fallback_pixels"] < 64 * 48 // 2
    got, _ = _render(sc, opts, 1, runs=3)
    for g in got:
        for k in ref:
            assert np.array_equal(g[k].view(np.uint32), ref[k].view(np.uint32)), k


def _coplanar_pairs(n, w, h):
    """n parallel tilted layers, each of two triangles in exactly one plane (the second has the
    first one's corner and edges, one of them doubled, in dyadic coordinates, so that both depth
    planes have the same bits). In blocks that the first one's edge crosses their pixel masks, and
    so their centroids' depths, differ, and the first one comes first, as by its id."""
    p0 = np.stack([np.full(n, -32.0), np.full(n, -32.0), -(16.0 + np.arange(n) / 8.0)], -1)
    u, v = np.array([64.0, 0.0, -1.0]), np.array([0.0, 64.0, 0.0])
    pos = np.stack([p0, p0 + u, p0 + v, p0, p0 + 2 * u, p0 + v], 1).reshape(-1, 3)
    rng = np.random.default_rng(n)
    sc = scenes.soup_scene(w, h, np.zeros((2 * n, 3, 2)), np.ones(2 * n), rng.uniform(0, 1, (2 * n, 3, 3)),
                           rng.uniform(0.001, 0.01, 2 * n), name=f"coplanar_{n}")
    sc.positions = pos.astype(np.float32)
    assert np.array_equal(sc.positions, pos)
    return sc


@pytest.mark.parametrize("window", [1, 4])
@pytest.mark.parametrize("opts", [0, _lib.OPT_FP32_SAMPLES])
def test_equal_depths_in_two_ranges_are_ordered_by_id(oracle_mod, opts, window):
    """Equal depths on both sides of a depth range's end, in the order of their ids: exact, so no
    pixel takes the exact sort."""
    sc = _coplanar_pairs(300, 72, 64)
    (got,), stats = _render(sc, opts, window)
    assert stats["block_tris"] > 300 * 16 and stats["fragments"] > 300 * 1024
    assert stats["fallback_pixels"] == 0
    ref = oracle_mod.render(sc, opts=oracle_mod.OPT_FP32_SAMPLES if opts else 0)
    assert np.array_equal(got["frag_counts"].astype(np.uint32), ref["frag_counts"])
    assert np.abs(got["image"].astype(int) - ref["image"].astype(int)).max() <= 1


@pytest.mark.parametrize("other", ["bytes", "textured"])
def test_batch_of_mixed_frames_keeps_the_threshold_wide(other):
    """A flat frame with the alpha threshold batched with a byte-coloured or textured frame without
    it: the batch's records are then not flat, and the threshold, which looks at the samples that
    have left the window, needs the four slots whatever the tuning. After the first 64 of the 100
    layers the transmittance is below 1/128 with all but two of them blended, and not yet with all
    but four."""
    from lucid_amd.batch import LucidBatch
    from lucid_amd.renderer import GpuScene, LucidRenderer
    alpha = np.where(np.arange(100) % 2, 19.0, 20.0) / 255.0
    left = np.cumprod(1.0 - alpha)
    assert left[59] > 1.0 / 128.0 > left[61]
    flat = _planes(100, 40, 32, 0.0, alpha, seed=2)
    if other == "bytes":
        second = scenes.config0(seed=6, num_tris=500, width=64, height=40, color_format="rgba8")
    else:
        second = scenes.textured_planes(64, 40, 5, seed=7)
    images = {}
    for window in (4, 1):
        print(f"\n[case] batch of flat and {other}, window={window}", flush=True)
        rs = [LucidRenderer((40, 32), opts=_lib.OPT_ALPHA_THRESHOLD), LucidRenderer((64, 40))]
        for r in rs:
            r.set_tuning(window=window)
        outs = [r.alloc_outputs(rgba8=True, rgba32f=True, counts=True) for r in rs]
        LucidBatch(rs).render([GpuScene(flat), GpuScene(second)], outs)
        images[window] = [{k: v.cpu().numpy() for k, v in o.items()} for o in outs]
    for a, b in zip(images[1], images[4]):
        for k in a:
            assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), k


@pytest.mark.parametrize("blend", [0, _lib.OPT_ADDITIVE_BLENDING])
@pytest.mark.parametrize("kind", ["bytes", "textured", "fp32"])
def test_the_window_knob_is_for_flat_records(kind, blend):
    """Byte-coloured, textured and fp32 frames, whose surfaces cross: the narrow tuning sends no
    more of their pixels to the exact sort, and none when four slots can order them."""
    opts = blend
    if kind == "textured":
        sc = scenes.textured_planes(150, 97, 60, seed=7)
    else:
        sc = _planes(90, 72, 56, 0.25, (0.01, 0.1), seed=8, color_format="rgba8" if kind == "bytes" else "f32")
        opts |= _lib.OPT_FP32_SAMPLES if kind == "fp32" else 0
    (a,), narrow = _render(sc, opts, 1)
    (b,), wide = _render(sc, opts, 4)
    assert narrow["fallback_pixels"] == wide["fallback_pixels"]
    assert kind == "textured" or wide["fallback_pixels"] == 0
    for k in a:
        assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), k


@pytest.mark.parametrize("kind", ["bytes", "textured"])
def test_threshold_of_general_records(oracle_mod, kind):
    """The alpha threshold with the default (narrow) tuning on general and textured records: counts
    as in the oracle's exact frame, colours within the skipped remainder (below 1/128 per channel)
    and the 1/255 quantisation."""
    if kind == "bytes":
        sc = scenes.config0(num_tris=20000, width=128, height=128, seed=42, color_format="rgba8")
    else:
        sc = scenes.textured_planes(150, 97, 90, seed=9)
    (got,), _ = _render(sc, _lib.OPT_ALPHA_THRESHOLD, 1)
    ref = oracle_mod.render(sc)
    assert np.array_equal(got["frag_counts"].astype(np.uint32), ref["frag_counts"])
    assert np.abs(got["image"].astype(int) - ref["image"].astype(int)).max() <= 3
