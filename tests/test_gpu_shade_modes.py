"""The block rasterisers' shading modes and ordering windows give the same bits: plain records
(fp32 samples, fp32 vertex colours, unit lighting) against the general ones, which an instance
colour of white selects (a product with exactly 1), and narrow windows against the four-slot
window, on scenes in depth order and with planes that intersect, for each blend option. Gradients
likewise."""

import numpy as np
import pytest

from lucid_amd import _lib, scenes

pytestmark = pytest.mark.gpu

BLENDS = [0, _lib.OPT_ADDITIVE_BLENDING, _lib.OPT_ALPHA_THRESHOLD]


def _render(sc, opts, window):
    from lucid_amd.renderer import GpuScene, LucidRenderer
    print(f"\n[case] {sc.name} {sc.width}x{sc.height} opts={opts:#x} window={window}", flush=True)
    r = LucidRenderer((sc.width, sc.height), opts=opts)
    r.set_tuning(window=window)
    out = r.render(GpuScene(sc), r.alloc_outputs(rgba8=True, rgba32f=True, counts=True))
    return {k: v.cpu().numpy() for k, v in out.items()}


def _white(sc):
    """The same scene, shaded by the general records."""
    sc.instances["flags"] |= scenes.INST_HAS_COLOR
    sc.instance_colors = np.full(len(sc.instances), 0xffffffff, np.uint32)
    return sc


SCENES = {
    "soup": lambda: scenes.config0(seed=3, num_tris=4000, width=203, height=130),
    "deep": lambda: scenes.block_stack(70, 50, 1500, center_px=(20, 20), size_px=12.0, seed=4),
    "tilted": lambda: scenes.tilted_planes(170, 90, 24, seed=5),
}


@pytest.mark.parametrize("blend", BLENDS)
@pytest.mark.parametrize("scene", sorted(SCENES))
def test_plain_records(scene, blend):
    opts = blend | _lib.OPT_FP32_SAMPLES
    ref = _render(_white(SCENES[scene]()), opts, window=4)
    for window in (1, 4):
        for got in (_render(SCENES[scene](), opts, window), _render(_white(SCENES[scene]()), opts, window)):
            for k in ref:
                assert np.array_equal(got[k].view(np.uint32), ref[k].view(np.uint32)), (k, window)


@pytest.mark.parametrize("blend", BLENDS)
def test_narrow_windows_rgba8(blend):
    """Textured, and byte-coloured general records."""
    def bytes_scene():
        return scenes.config0(seed=6, num_tris=3000, width=150, height=97, color_format="rgba8")
    for make in (bytes_scene, lambda: scenes.textured_planes(150, 97, 30, seed=7)):
        a, b = _render(make(), blend, 1), _render(make(), blend, 4)
        for k in a:
            assert np.array_equal(a[k].view(np.uint32), b[k].view(np.uint32)), k


@pytest.mark.parametrize("window", [1, 4])
@pytest.mark.parametrize("scene", sorted(SCENES))
def test_plain_gradients(scene, window):
    import torch
    from lucid_amd.renderer import GpuScene, LucidRenderer
    grads = []
    for make in (SCENES[scene], lambda: _white(SCENES[scene]())):
        sc = make()
        print(f"\n[case] {sc.name} {sc.width}x{sc.height} window={window}", flush=True)
        r = LucidRenderer((sc.width, sc.height), opts=_lib.OPT_FP32_SAMPLES)
        r.set_tuning(window=window)
        g = torch.Generator().manual_seed(1)
        gi = (torch.randn((sc.height, sc.width, 4), generator=g) * 1e-3).cuda()
        grads.append([x.cpu().numpy() for x in r.backward(GpuScene(sc), gi)])
    assert np.abs(grads[0][0]).max() > 0
    for a, b in zip(*grads):
        assert np.array_equal(a, b)
