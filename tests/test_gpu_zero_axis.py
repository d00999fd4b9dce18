"""Rays with zero direction components, and the launch rule of small batches, against the CPU oracle.

A ray that does not move along an axis is culled by boxes it cannot meet there, which the reference's slab
test lets through: the hits have to stay the oracle's bit for bit, also where triangles are large against
the scene (the cull's bound is then wider than the box) and where the caller's boxes do not hold their
triangles (the cull is then off).
"""
import numpy as np
import pytest

from gonzales_amd import abi, scenes
from gonzales_amd.accelerator import Primitives, Scene, TriangleMesh, build_bounding_hierarchy_gpu
from helpers import OracleView, random_rays, random_soup_hierarchy
from test_gpu_traversal import _assert_hits_equal, _device_any, _device_closest

pytestmark = pytest.mark.gpu


def _zero_axis_rays(n, seed, bh, scale=1.0):
    """Random rays, one or two direction components set to +0 or -0, a fifth with an origin coordinate on a
    vertex's own."""
    g = np.random.default_rng(seed)
    rays, tmax = random_rays(n, seed, lo=-0.2 * scale, hi=1.2 * scale, tmax=(0.1 * scale, 4.0 * scale))
    first = g.integers(0, 3, n)
    other = np.where(g.random(n) < 0.3, (first + 1) % 3, first)
    pts = np.concatenate([m.points[:, :3] for m in bh.scene.meshes])
    on = g.random(n) < 0.2
    for a, (o, d) in enumerate((("orgX", "dirX"), ("orgY", "dirY"), ("orgZ", "dirZ"))):
        z = (first == a) | (other == a)
        rays[d][z] = np.where(g.random(z.sum()) < 0.5, 0.0, -0.0)
        w = z & on
        rays[o][w] = pts[g.integers(0, len(pts), w.sum()), a]
    return rays, tmax


def test_zero_components_of_rays_that_are_not_finite(gpu):
    """NaN, infinite and huge origins or directions beside a zero component: tri_test accepts a NaN, so no
    box may be skipped."""
    bh = random_soup_hierarchy(5000, 13, scale=0.05)
    bh.upload_to_gpu()
    rays, tmax = _zero_axis_rays(20_000, 14, bh)
    g = np.random.default_rng(15)
    odd = np.asarray([np.nan, np.inf, -np.inf, 1e30, -3e38, 1e13], np.float32)
    for name in ("orgX", "orgY", "orgZ", "dirX", "dirY", "dirZ"):
        at = (g.random(len(rays)) < 0.1) & (rays[name] != 0.0)
        rays[name][at] = odd[g.integers(0, len(odd), at.sum())]
    ref, _ = OracleView(bh).closest(rays, tmax)
    hits, _ = _device_closest(bh, rays, tmax)
    assert np.array_equal(hits["prim"] >= 0, ref["hit"].astype(bool))
    finite = np.isfinite(ref["tHit"])
    for f, r in (("t", "tHit"), ("u", "u"), ("v", "v")):
        assert np.array_equal(np.isnan(hits[f]), np.isnan(ref[r]))
        assert np.array_equal(hits[f][finite], ref[r][finite], equal_nan=True)
    occ, _ = _device_any(bh, rays, tmax)
    assert np.array_equal(occ, ref["hit"].astype(bool))
    bh.free()


@pytest.mark.parametrize("n_tris,size,scale", [(40, 1.0, 1.0), (3000, 0.3, 1.0), (50_000, 0.02, 1.0),
                                               (20_000, 0.0005, 1.0), (5000, 30.0, 100.0)])
def test_zero_components_match_the_oracle(gpu, n_tris, size, scale):
    bh = random_soup_hierarchy(n_tris, n_tris, spread=scale, scale=size)
    bh.upload_to_gpu()
    rays, tmax = _zero_axis_rays(20_000, 5, bh, scale)
    ref, ref_st = OracleView(bh).closest(rays, tmax, stats=True)
    hits, _ = _device_closest(bh, rays, tmax)
    _assert_hits_equal(hits, ref)
    occ, _ = _device_any(bh, rays, tmax)
    assert np.array_equal(occ, ref["hit"].astype(bool))
    _, st = _device_closest(bh, rays, tmax, stats=True)  # the counting kernels count the reference's visits
    assert st.tobytes() == ref_st.tobytes()
    bh.free()


def test_zero_components_in_axis_aligned_planes(gpu):
    bh, _ = scenes.cornell_hierarchy()
    bh.upload_to_gpu()
    rays, tmax = _zero_axis_rays(20_000, 6, bh, 2.0)
    ref, _ = OracleView(bh).closest(rays, tmax)
    hits, _ = _device_closest(bh, rays, tmax)
    _assert_hits_equal(hits, ref)
    bh.free()


def test_boxes_that_do_not_hold_their_triangles(gpu):
    bh = random_soup_hierarchy(2000, 7, scale=0.2)
    lo = bh.nodes["boundsMinZ"].copy()
    bh.nodes["boundsMinZ"] = lo + 0.6 * (bh.nodes["boundsMaxZ"] - lo)
    bh.upload_to_gpu()
    rays, tmax = _zero_axis_rays(20_000, 8, bh)
    ref, _ = OracleView(bh).closest(rays, tmax)
    hits, _ = _device_closest(bh, rays, tmax)
    _assert_hits_equal(hits, ref)
    bh.free()


@pytest.mark.parametrize("sah", [False, True])
@pytest.mark.parametrize("broken", [0, 1, 60])
def test_hierarchies_built_on_the_device(gpu, sah, broken):
    """A vertex coordinate that is NaN leaves its triangle's box finite (minima and maxima drop it) and the
    triangle outside that box: tri_test accepts a NaN, so such a hierarchy culls nothing."""
    n = 3000
    g = np.random.default_rng(21)
    v = (g.random((n, 1, 3)) + 0.1 * (g.random((n, 3, 3)) - 0.5)).astype(np.float32)
    for k in g.permutation(n)[:broken]:
        v[k, g.integers(0, 3), g.integers(0, 3)] = np.nan
    mats = np.zeros(1, abi.MATERIAL)
    mats["type"] = 1
    scene = Scene([TriangleMesh.from_xyz(v.reshape(-1, 3), np.arange(3 * n, dtype=np.int64))], mats)
    bh = build_bounding_hierarchy_gpu(scene, Primitives.geometric(0, n, 0), sah=sah)
    rays, tmax = _zero_axis_rays(20_000, 22, bh)
    for f in ("orgX", "orgY", "orgZ"):  # origins taken from a vertex may be its NaN
        rays[f][np.isnan(rays[f])] = 0.5
    ref, _ = OracleView(bh).closest(rays, tmax)
    hits, _ = _device_closest(bh, rays, tmax)
    hit = ref["hit"].astype(bool)
    assert np.array_equal(hits["prim"] >= 0, hit)
    assert bool(np.isnan(ref["tHit"][hit]).any()) == (broken > 0)
    for f, r in (("t", "tHit"), ("u", "u"), ("v", "v")):
        assert np.array_equal(hits[f][hit], ref[r][hit], equal_nan=True)
    occ, _ = _device_any(bh, rays, tmax)
    assert np.array_equal(occ, hit)
    bh.free()


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 65_535, 65_536, 65_537, 131_072, 131_073])
def test_batches_at_the_edges_of_the_wave_sizes(gpu, n):
    bh = random_soup_hierarchy(500, 9, scale=0.1)
    bh.upload_to_gpu()
    rays, tmax = random_rays(n, 10)
    ref, _ = OracleView(bh).closest(rays, tmax)
    hits, _ = _device_closest(bh, rays, tmax)
    _assert_hits_equal(hits, ref)
    occ, _ = _device_any(bh, rays, tmax)
    assert np.array_equal(occ, ref["hit"].astype(bool))
    bh.free()


def test_default_rule_on_both_sides_of_its_line(gpu):
    bh = random_soup_hierarchy(500, 11, scale=0.1)
    bh.upload_to_gpu()
    rays, tmax = random_rays(1 << 22, 12)
    whole, _ = _device_closest(bh, rays, tmax)
    part, _ = _device_closest(bh, rays[:-1], tmax[:-1])
    assert whole[:-1].tobytes() == part.tobytes()
    sel = slice(0, 50_000)
    _assert_hits_equal(whole[sel], OracleView(bh).closest(rays[sel], tmax[sel])[0])
    bh.free()


@pytest.mark.parametrize("n_tris,binned", [(1 << 18, False), ((1 << 18) + 1, True)])
def test_large_default_batches_on_large_trees_are_binned(gpu, n_tris, binned):
    """Default batches of one lane per ray: on trees of more than 2^18 primitives binned from 3 x 2^20 rays on
    (the handle then keeps the binning's storage), with the hits of the given order."""
    bh = random_soup_hierarchy(n_tris, 13, scale=0.01)
    bh.upload_to_gpu()
    rays, tmax = random_rays(3 << 20, 14)
    part, _ = _device_closest(bh, rays[:-1], tmax[:-1])
    before = bh.info().deviceBytes
    whole, _ = _device_closest(bh, rays, tmax)
    assert (bh.info().deviceBytes > before) == binned
    assert whole[:-1].tobytes() == part.tobytes()
    occ, _ = _device_any(bh, rays, tmax)
    assert np.array_equal(occ, whole["prim"] >= 0)
    sel = slice(len(rays) - 50_000, None)
    _assert_hits_equal(whole[sel], OracleView(bh).closest(rays[sel], tmax[sel])[0])
    bh.free()
