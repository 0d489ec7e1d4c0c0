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
