"""The default launch of a path trace on both sides of its size rules: records equal, byte for byte, to one
launch per bounce over all paths (queued = 0)."""
import numpy as np
import pytest

from gonzales_amd import abi
from gonzales_amd.accelerator import BoundingHierarchy
from gonzales_amd.camera import cornell_camera
from gonzales_amd.integrator import (MisOptions, VolumePathIntegrator, coated_conductor_material, conductor_material,
                                     dielectric_material, diffuse_material)
from gonzales_amd import scenes

pytestmark = pytest.mark.gpu


def _integrator(diffuse):
    bh, _ = scenes.cornell_hierarchy()
    bh = BoundingHierarchy(bh.scene, bh.prim_ids, bh.nodes)
    bh.upload_to_gpu()
    cam = cornell_camera(res=512, spp=8, seed=3)
    opt = MisOptions(max_depth=4, zsobol_seed=cam.c.zsSeed, log2_spp=cam.c.zsLog2Spp, base4_digits=cam.c.zsBase4Digits)
    if diffuse:
        return VolumePathIntegrator(bh, opt), cam
    kinds = [diffuse_material((0.5, 0.4, 0.3)), dielectric_material(eta=1.5, roughness=0.2),
             conductor_material(roughness=0.3), coated_conductor_material(interface_roughness=0.1, conductor_roughness=0.3)]
    mats = abi.concat([kinds[k % 4] for k in range(len(bh.scene.materials))], abi.GZ_MATERIAL)
    return VolumePathIntegrator(bh, opt, materials=mats), cam


@pytest.mark.parametrize("diffuse,counts", [(True, (1, 63, 65, 4097, 1 << 19, (1 << 19) + 1)),
                                            (False, (1, 65, 4097, 1 << 20, (1 << 20) + 1))])
def test_default_launch_equals_the_full_relaunch(gpu, diffuse, counts):
    import torch

    integ, cam = _integrator(diffuse)
    assert cam.path_count > max(counts)
    got = []
    for n in counts:
        buf = torch.empty(n * abi.GZ_PATH.itemsize, dtype=torch.uint8, device="cuda")
        cam.paths_device(buf, 0, n)
        integ.trace(buf, n)
        got.append(buf.cpu().numpy())
    integ.bh.check_traversal()
    integ.set_launch(0)
    n = max(counts)
    buf = torch.empty(n * abi.GZ_PATH.itemsize, dtype=torch.uint8, device="cuda")
    cam.paths_device(buf, 0, n)
    integ.trace(buf, n)
    ref = buf.cpu().numpy()
    for n, g in zip(counts, got):
        assert np.array_equal(g, ref[:n * abi.GZ_PATH.itemsize]), n
    integ.bh.free()


def test_whole_rounds_of_a_batch_equal_its_levels(gpu):
    """The batch's default for small rounds against an explicit level-by-level launch: the same films."""
    from gonzales_amd.batch import BatchEntry, SceneBatch
    from gonzales_amd.camera import DeviceFilm

    pairs = [_integrator(True), _integrator(False)]
    entries = [BatchEntry(i, c, DeviceFilm(c)) for i, c in pairs]
    films = []
    for launch in (None, (256, 1, 64, 3, 3), (256, 1, 64, 0, 1)):
        batch = SceneBatch(entries, round_paths=700_001)
        if launch:
            batch.set_launch(*launch)
        batch.clear_films()
        batch.render()
        batch.check()
        films.append([t.clone() for e in entries for t in (e.film.light, e.film.weight, e.film.albedo, e.film.normal)])
        batch.close()
    for other in films[1:]:
        assert all((a == b).all() for a, b in zip(films[0], other))
    assert float(films[0][0].sum()) > 0 and float(films[0][4].sum()) > 0


def test_rounds_on_both_sides_of_the_wavefront_scenes_line(gpu):
    """Default rounds with 2^20 and with 2^20 + 8 paths of a scene that defaults to the wavefront (whole paths
    and levels): the films of an explicit level-by-level launch."""
    from gonzales_amd.batch import BatchEntry, SceneBatch
    from gonzales_amd.camera import DeviceFilm

    (mixed, cam), (diffuse, dcam) = _integrator(False), _integrator(True)
    entries = [BatchEntry(mixed, cam, DeviceFilm(cam)), BatchEntry(diffuse, dcam, DeviceFilm(dcam))]
    films = []
    for round_paths, launch in ((1 << 20, None), ((1 << 20) + 8, None), (1 << 20, (256, 1, 64, 0, 1))):
        batch = SceneBatch(entries, round_paths=round_paths)
        if launch:
            batch.set_launch(*launch)
        for use_graph in (True, False):
            batch.clear_films()
            batch.render(use_graph)
            batch.check()
            films.append([t.clone() for e in entries for t in (e.film.light, e.film.weight, e.film.albedo, e.film.normal)])
        batch.close()
    for other in films[1:]:
        assert all((a == b).all() for a, b in zip(films[0], other))
    assert float(films[0][0].sum()) > 0 and float(films[0][4].sum()) > 0


@pytest.mark.parametrize("res,spp", [((512, 384), 8), ((512, 385), 8)])
def test_replay_of_large_frames_equals_the_full_relaunch(gpu, res, spp):
    """The queued replay on both sides of 3 x 2^19 paths (strided below and at it, one shared counter a level
    above), from a record and tracing its rays again, against one launch per bounce over all paths: the same
    path records and gradients. The gradients are float64 sums of up to 1e7 terms of one sign (the target is
    black) in another order: 1e7 x 2^-53 = 1.1e-9 of the largest, times four for the terms of the other sign."""
    import torch
    from gonzales_amd.camera import Film, PerspectiveCamera, pbrt_transform
    from gonzales_amd.diff import DiffRenderer

    bh, gz, _, _ = scenes.inverse_rendering_scene(subdivisions=3, n_params=8)
    bh.upload_to_gpu()
    cam = PerspectiveCamera(pbrt_transform([1, 0, 0, 0, 0, 1, 0, 0, 0, 0, -1, 0, 0, -1, 6.8, 1]), 19.5, Film(*res), spp, 0)
    assert cam.path_count == res[0] * res[1] * spp
    opt = MisOptions(max_depth=3, zsobol_seed=cam.c.zsSeed, log2_spp=cam.c.zsLog2Spp, base4_digits=cam.c.zsBase4Digits)
    r = DiffRenderer(bh, cam, gz, opt)
    out = []
    for launch, record in (((0, 256, 1, 256, 0), False), ((3, 256, 1, 64, 0), True), ((3, 256, 1, 64, 2), True),
                           ((1, 128, 1, 256, 0), False)):
        r.integrator.set_launch(*launch)
        img = r.render()
        assert (r.recorded_levels > 0) == record
        ga, gr = r.backward(2 * img)
        out.append((ga, gr, r.d_paths.clone()))
    for ga, gr, paths in out[1:]:
        assert torch.equal(paths, out[0][2])
        for x, y in ((ga, out[0][0]), (gr, out[0][1])):
            assert float(y.abs().max()) > 0
            assert float((x - y).abs().max()) <= 5e-9 * float(y.abs().max())
    bh.free()


def test_diff_renderers_of_two_sizes_on_one_handle(gpu):
    """Each renderer runs under its own launch whatever others of the same hierarchy are made between, and the
    handle's launch stays the default: a large frame records every level, a small one up to its drain level,
    with the images and gradients of renderers of their own hierarchies. A launch set on the handle holds for both."""
    import torch
    from gonzales_amd.camera import Film, PerspectiveCamera, pbrt_transform
    from gonzales_amd.diff import DiffRenderer

    def make(bh, gz, res, spp):
        cam = PerspectiveCamera(pbrt_transform([1, 0, 0, 0, 0, 1, 0, 0, 0, 0, -1, 0, 0, -1, 6.8, 1]), 19.5, Film(*res), spp, 0)
        opt = MisOptions(max_depth=3, zsobol_seed=cam.c.zsSeed, log2_spp=cam.c.zsLog2Spp, base4_digits=cam.c.zsBase4Digits)
        return DiffRenderer(bh, cam, gz, opt)

    def step(r):
        img = r.render()
        return (img, *r.backward(2 * img), r.recorded_levels)

    def scene():
        bh, gz, _, _ = scenes.inverse_rendering_scene(subdivisions=3, n_params=8)
        bh.upload_to_gpu()
        return bh, gz

    sizes = (((512, 257), 8), ((64, 48), 4), ((512, 200), 8))
    bh, gz = scene()
    shared = [make(bh, gz, *size) for size in sizes]
    got = [step(r) for r in shared]
    assert [g[3] for g in got] == [4, 2, 3]
    assert shared[0].integrator.launch_by_size()
    for size, g in zip(sizes, got):
        bh2, gz2 = scene()
        img, ga, gr, levels = step(make(bh2, gz2, *size))
        assert torch.equal(img, g[0]) and levels == g[3]
        for x, y in ((ga, g[1]), (gr, g[2])):
            assert float((x - y).abs().max()) <= 5e-9 * float(y.abs().max())
        bh2.free()
    shared[0].integrator.set_launch(3, 256, 1, 64, 1)
    assert [step(r)[3] for r in shared] == [1, 1, 1]
    shared[0].integrator.reset_launch()
    assert [step(r)[3] for r in shared] == [4, 2, 3]
    bh.free()
