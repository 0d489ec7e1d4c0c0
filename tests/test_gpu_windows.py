"""The ordering windows decide only which pixels take the exact sort, never a result: fp32 frames
whose blocks are pre-sorted (their depth ranges are composited apart and chained), narrow windows
of general and textured records where pixels do reach the exact sort, and batches that mix frames
with and without the alpha threshold."""

import numpy as np
import pytest

from lucid_amd import _lib, scenes

pytestmark = pytest.mark.gpu


def _planes(n, w, h, slope, alpha, seed, color_format="f32"):
    """n screen-filling quads at even depths, with slopes that make near neighbours cross."""
    rng = np.random.default_rng(seed)
    corners = np.array([[-1.3, -1.2], [1.2, -1.3], [1.3, 1.2], [-1.2, 1.3]])
    ndc = np.repeat(corners[None], n, axis=0)
    k = rng.uniform(-slope, slope, (n, 2))
    depth = 10.0 + 0.05 * rng.permutation(n)[:, None] + corners[:, 0] * k[:, :1] + corners[:, 1] * k[:, 1:]
    a = np.broadcast_to(alpha, n) if np.ndim(alpha) == 0 else rng.uniform(*alpha, n)
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
