"""What the stages of lucid_stage_times hold: row generation of low bins apart from that of high
bins, whose stage also has the sort, in frames of few bins as in large ones."""

import numpy as np
import pytest

from lucid_amd import _lib, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(512, 512), (1088, 1056)])
def test_high_bins_count_as_high(w, h):
    """Every bin is high: next to nothing of the row generation is the low bins'. The timed frame's
    image is the untimed one's."""
    from lucid_amd.renderer import GpuScene, LucidRenderer
    sc = scenes.config0(seed=12, num_tris=400_000, width=w, height=h, vertex_sigma=0.04)
    print(f"\n[case] {sc.name} {w}x{h}", flush=True)
    images, runs = [], []
    for opts in (_lib.OPT_TIMERS, 0):
        r = LucidRenderer((w, h), opts=opts)
        g, out = GpuScene(sc), r.alloc_outputs()
        for _ in range(5):
            r.render(g, out)
            if opts:
                runs.append(r.stage_times())
        assert r.get_stats()["low_bins"] == 0 and r.get_stats()["high_bins"] == r.bin_count
        images.append(out["image"].cpu().numpy())
    med = {k: float(np.median([t[k] for t in runs])) for k in runs[0]}
    print(med, flush=True)
    assert 0.0 < med["rowgen_low"] < 0.3 * med["rowgen_high_sort"]
    assert np.abs(images[0].astype(int) - images[1].astype(int)).max() <= 1
