"""Setup at the sizes where its work-group handling can go wrong: the wave-wide instance search
(one instance, 64 and 65 probes, more than 64 * 64 instances, instances without quads) and the
wave's record staging (a last wave with one quad, waves with no visible triangle, both
triangles of a quad). Setup records bit-exact and frames against the oracle, as everywhere."""

import numpy as np
import pytest

from lucid_amd import scenes

from test_gpu_parity import _check, _render_both

pytestmark = pytest.mark.gpu


def _with_instances(sc, counts):
    """The scene's quads dealt to instances of the given sizes (their sum is the quad count)."""
    counts = np.asarray(counts, np.int64)
    assert counts.sum() == sc.num_quads
    inst = np.zeros(len(counts), scenes.INSTANCE_DTYPE)
    inst["index_offset"] = (np.cumsum(counts) - counts) * 4
    inst["num_quads"] = counts
    inst["flags"] = scenes.INST_HAS_VERTEX_COLORS
    sc.instances = inst
    sc.config = scenes.make_config(scenes.scene_camera(sc), len(inst))
    return sc


def _counts(num, quads, seed):
    """num instance sizes summing to `quads`, a third of them empty."""
    rng = np.random.default_rng(seed)
    w = rng.random(num) * (rng.random(num) > 0.33)
    w[rng.integers(0, num)] += 0.5
    return np.bincount(rng.choice(num, quads, p=w / w.sum()), minlength=num)


@pytest.mark.parametrize("num,quads", [(1, 1), (1, 65), (2, 257), (64, 700), (65, 700),
                                       (129, 1025), (4097, 3000)])
def test_instance_tables(oracle_mod, num, quads):
    sc = scenes.config0(num_tris=quads, width=96, height=64, seed=90 + num)
    sc = _with_instances(sc, _counts(num, quads, num))
    r, gpu, ref = _render_both(sc, oracle_mod)
    _check(sc, gpu, ref, oracle_mod)


@pytest.mark.parametrize("quads", [1, 31, 33, 64, 257])
def test_record_staging(oracle_mod, quads):
    """Mesh quads (two triangles each), some of them one-sided soup quads, with a run of 70
    rejected quads in the middle: every visible triangle's record as the oracle's."""
    rng = np.random.default_rng(quads)
    centre = rng.uniform(-0.9, 0.9, (quads, 1, 2))
    ndc = centre + rng.uniform(0.02, 0.2, (quads, 1, 1)) * np.array([[-1, -.9], [1, -1], [.9, 1], [-1, 1]])
    depth = np.repeat(rng.uniform(2.0, 50.0, (quads, 1)), 4, axis=1)
    sc = scenes.quad_soup_scene(96, 64, ndc, depth, rng.uniform(0, 1, (quads, 4, 3)),
                                rng.uniform(0.2, 0.8, quads))
    one = rng.random(quads) < 0.3
    sc.quad_indices[one, 3] = sc.quad_indices[one, 2]
    sc.quad_indices[90:160] = 0
    r, gpu, ref = _render_both(sc, oracle_mod)
    _check(sc, gpu, ref, oracle_mod)
    recs, aabb = r.read_setup(quads)
    assert np.array_equal(aabb, ref["quad_aabb"])
    live = np.zeros(2 * quads, bool)
    for s in range(2):
        live[s::2] = (aabb != 0xFFFFFFFF) & ((aabb >> (30 + s)) & 1 == 0)
    want = oracle_mod.render(sc, mode=oracle_mod.MODE_COUNTS)["tri_records"]
    assert np.array_equal(recs[live], want[live])
