"""Frames whose block lists do not fit: the space of the fixed high bins (at least 1024 list
positions) is decided before row generation, the space of promoted bins during it. Either way
the frame reports an overflow, the lists grow and the next frame equals the oracle's."""

import numpy as np
import pytest

from lucid_amd import _lib

from test_gpu_block_lists import _stacks
from test_gpu_parity import _check, _render_both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(1024, 512), (1056, 1056)])  # row generation in one launch, in two
def test_promoted_bins_overflow_beside_fixed_ones(oracle_mod, w, h):
    """100 fixed high bins (1200 list positions each), whose lists fit a new renderer, beside 380
    bins that are promoted (1000 positions each), whose lists do not."""
    from lucid_amd.renderer import GpuScene, LucidRenderer
    counts = np.zeros(((w + 31) // 32) * (h // 32), int)
    counts[:480] = 500
    counts[np.random.default_rng(3).choice(480, 100, replace=False)] = 600
    sc = _stacks(w, h, "fixed_promoted", counts, seed=6)
    print(f"\n[case] {sc.name} {len(counts)} bins, {sc.num_quads} quads", flush=True)
    r = LucidRenderer((w, h))
    out, gs = r.alloc_outputs(), GpuScene(sc)
    r.render_async(gs, out)
    assert r.finish() == _lib.LUCID_ERR_CAPACITY
    r.render(gs, out)  # (other pools may grow in between)
    assert r.get_stats()["high_bins"] == 480 and r.get_stats()["promoted_bins"] == 380
    r, gpu, ref = _render_both(sc, oracle_mod)
    _check(sc, gpu, ref, oracle_mod)


def test_more_list_positions_than_32_bits(oracle_mod):
    """840 k triangles over all 5120 bins of the largest frame: more list positions than the bins'
    32-bit offsets reach. The frame is refused, nothing is written at wrapped offsets, and the
    renderer goes on with the next scene."""
    from lucid_amd import scenes
    from lucid_amd.renderer import GpuScene, LucidRenderer
    w, h, n = 2560, 2048, 840_000
    assert n * 5120 > 2 ** 32
    ndc = np.broadcast_to(np.array([[-1.1, -1.2], [3.4, -1.3], [-1.2, 3.5]]), (n, 3, 2))
    sc = scenes.soup_scene(w, h, ndc, np.linspace(2.0, 90.0, n), np.full((n, 3, 3), 0.5, np.float32),
                           np.full(n, 0.5))
    print(f"\n[case] {n} full-screen triangles, {w}x{h}", flush=True)
    r = LucidRenderer((w, h))
    with pytest.raises(_lib.LucidError) as e:
        r.render(GpuScene(sc))
    assert e.value.code == _lib.LUCID_ERR_OUT_OF_MEMORY
    small = scenes.config0(seed=4, num_tris=3000, width=w, height=h)
    print("[case] the same renderer, 3000 triangles", flush=True)
    out = r.render(GpuScene(small))
    ref = oracle_mod.render(small)
    assert np.array_equal(out["frag_counts"].cpu().numpy().astype(np.uint32), ref["frag_counts"])
    assert np.abs(out["image"].cpu().numpy().astype(int) - ref["image"].astype(int)).max() <= 1
