"""The default launches by size and the way back to them: set(get()) of a handle that none was set for changes
nothing, the defaults marked as the choice by size put a handle (a batch) back under the rules, the same
values unmarked are a launch like any other."""
import ctypes

import numpy as np
import pytest

from gonzales_amd import abi, scenes
from gonzales_amd.accelerator import BoundingHierarchy
from helpers import assert_isect_equal, random_rays, random_soup_hierarchy

pytestmark = pytest.mark.gpu

N = 1 << 18  # binned by an explicit default configuration, traced in the given order by the rule


def _binned(bh, rays, tmax):
    """Whether a batch makes the handle keep binning storage (a stream of its own: nothing is kept yet)."""
    import torch

    d = torch.from_numpy(rays.view(np.uint8).reshape(-1)).cuda()
    t = torch.from_numpy(tmax).cuda()
    out = torch.empty(len(tmax) * 16, dtype=torch.uint8, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    before = bh.info().deviceBytes
    bh.closest_device(d, t, out, stream=s)
    s.synchronize()
    return bh.info().deviceBytes - before > 16 * N


def test_trace_config_set_get_and_back(gpu):
    lib = abi.load()
    bh = random_soup_hierarchy(500, 3, scale=0.1)
    bh.upload_to_gpu()
    rays, tmax = random_rays(N, 4)
    c = bh.trace_config()
    assert c.reserved == abi.GZ_LAUNCH_BY_SIZE
    assert not _binned(bh, rays, tmax)
    abi.check(lib.gz_gpu_set_trace_config(bh.handle, ctypes.byref(c)))  # set(get())
    assert bh.trace_config().reserved == abi.GZ_LAUNCH_BY_SIZE and not _binned(bh, rays, tmax)
    bh.set_trace_config()  # the same values, set
    assert bh.trace_config().reserved == 0 and _binned(bh, rays, tmax)
    c = bh.trace_config()
    abi.check(lib.gz_gpu_set_trace_config(bh.handle, ctypes.byref(c)))
    assert _binned(bh, rays, tmax)
    bh.set_trace_config(by_size=1)
    assert bh.trace_config().reserved == abi.GZ_LAUNCH_BY_SIZE and not _binned(bh, rays, tmax)
    bh.set_trace_config(record_times=1, by_size=1)  # timed, still by size
    assert bh.trace_config().recordTimes == 1 and not _binned(bh, rays, tmax)
    assert bh.trace_config().reserved == abi.GZ_LAUNCH_BY_SIZE
    c = bh.trace_config()
    c.refillLanes = 16  # read, changed, set: as given
    abi.check(lib.gz_gpu_set_trace_config(bh.handle, ctypes.byref(c)))
    assert bh.trace_config().reserved == 0 and bh.trace_config().refillLanes == 16 and _binned(bh, rays, tmax)
    bh.free()


def _cornell(mixed):
    from gonzales_amd.camera import cornell_camera
    from gonzales_amd.integrator import MisOptions, VolumePathIntegrator, conductor_material, diffuse_material

    bh, _ = scenes.cornell_hierarchy()
    bh = BoundingHierarchy(bh.scene, bh.prim_ids, bh.nodes)
    bh.upload_to_gpu()
    cam = cornell_camera(res=256, spp=4, seed=3)
    opt = MisOptions(max_depth=4, zsobol_seed=cam.c.zsSeed, log2_spp=cam.c.zsLog2Spp, base4_digits=cam.c.zsBase4Digits)
    mats = None
    if mixed:
        kinds = [diffuse_material((0.5, 0.4, 0.3)), conductor_material(roughness=0.3)]
        mats = abi.concat([kinds[k % 2] for k in range(len(bh.scene.materials))], abi.GZ_MATERIAL)
    return VolumePathIntegrator(bh, opt, materials=mats), cam


@pytest.mark.parametrize("mixed,default", [(False, (1, 256, 1, 256, 3)), (True, (3, 256, 1, 64, 3))])
def test_mis_launch_set_get_and_back(gpu, mixed, default):
    import torch

    lib = abi.load()
    integ, cam = _cornell(mixed)
    start = torch.empty(N * abi.GZ_PATH.itemsize, dtype=torch.uint8, device="cuda")
    cam.paths_device(start, 0, N)
    work = start.clone()
    integ.trace(work)
    ref = work.clone()

    def whole():
        """Whether a trace keeps no queue storage; its records are the first trace's."""
        integ.release_queues()
        work.copy_(start)
        torch.cuda.synchronize()
        free, _ = torch.cuda.mem_get_info()
        integ.trace(work)
        torch.cuda.synchronize()
        kept = free - torch.cuda.mem_get_info()[0]
        assert torch.equal(work, ref)
        return kept == 0

    c = integ._launch()
    assert integ.launch_by_size() and integ.launch() == default and whole()
    abi.check(lib.gz_gpu_set_mis_launch(integ.bh.handle, ctypes.byref(c)))  # set(get())
    assert integ.launch_by_size() and whole()
    integ.set_launch(*default)  # the same values, set
    assert not integ.launch_by_size() and integ.launch() == default and not whole()
    c = integ._launch()
    abi.check(lib.gz_gpu_set_mis_launch(integ.bh.handle, ctypes.byref(c)))
    assert not integ.launch_by_size() and not whole()
    integ.reset_launch()
    assert integ.launch_by_size() and integ.launch() == default and whole()
    c = integ._launch()
    c.chunk = 128  # read, changed, set: as given
    abi.check(lib.gz_gpu_set_mis_launch(integ.bh.handle, ctypes.byref(c)))
    assert not integ.launch_by_size() and integ.launch()[3] == 128 and not whole()
    c.reserved[0] = 2
    assert lib.gz_gpu_set_mis_launch(integ.bh.handle, ctypes.byref(c)) == abi.GZ_E_INVALID
    integ.bh.free()


def test_batch_launch_back_to_the_default(gpu):
    from gonzales_amd.batch import BatchEntry, SceneBatch
    from gonzales_amd.camera import DeviceFilm

    entries = [BatchEntry(i, c, DeviceFilm(c)) for i, c in (_cornell(False), _cornell(True))]
    batch = SceneBatch(entries)
    films = []
    for launch in (None, (256, 1, 64, 3, 3), (256, 1, 256, 3, 1, 1), (256, 1, 256, 3, 1), (256, 1, 64, 3, 3, 1),
                   (256, 1, 128, 3, 1, 1)):
        if launch:
            batch.set_launch(*launch)
        batch.clear_films()
        batch.render()
        batch.check()
        films.append([t.clone() for e in entries for t in (e.film.light, e.film.weight, e.film.albedo, e.film.normal)])
    for other in films[1:]:
        assert all((a == b).all() for a, b in zip(films[0], other))
    c = abi.GzMisLaunch(1, 256, 1, 256, 3, (2, 0, 0))
    assert abi.load().gz_batch_set_launch(batch.handle, ctypes.byref(c)) == abi.GZ_E_INVALID
    batch.close()


def test_noalloc_under_the_set_default_configuration(gpu):
    """gz_gpu_traverse_batch_noalloc with the default configuration set for every batch (persistent lanes by
    XCD also for small ones)."""
    bh = random_soup_hierarchy(50_000, 21)
    bh.upload_to_gpu()
    bh.set_trace_config()
    for n, seed in ((200_000, 22), (333, 23)):
        rays, t = random_rays(n, seed)
        out = np.zeros(n, abi.INTERSECTION)
        abi.check(abi.load().gz_gpu_traverse_batch_noalloc(bh.handle, abi.ptr(rays), abi.ptr(t), n, abi.ptr(out)))
        assert_isect_equal(out, bh.intersect_batch_gpu(rays, t))
    bh.free()


def test_tuners_apply_what_they_choose(gpu, tmp_path, monkeypatch):
    """The tuners leave the handle at the choice by size where they choose the default, read that back from a
    cache, and set any other choice. (The choice is given: timings are not this test's matter.)"""
    import torch
    from gonzales_amd import autotune as at

    integ, cam = _cornell(False)
    n = 30_000
    start = torch.empty(n * abi.GZ_PATH.itemsize, dtype=torch.uint8, device="cuda")
    cam.paths_device(start, 0, n)
    bh = random_soup_hierarchy(2000, 3, scale=0.05)
    bh.upload_to_gpu()
    rays, tmax = random_rays(5000, 4)
    d = torch.from_numpy(rays.view(np.uint8).reshape(-1)).cuda()
    t = torch.from_numpy(tmax).cuda()
    integ.set_launch(3, 256, 1, 64, 1)
    bh.set_trace_config(3, 8, 32)
    for k, by_size in ((0, True), (1, False), (0, True)):
        monkeypatch.setattr(at, "fastest", lambda timings: list(timings)[k])
        best, timings = at.autotune_mis(integ, start, n, reps=1)
        assert set(timings) == set(at.MIS_CANDIDATES) and best == at.MIS_CANDIDATES[k]
        assert integ.launch_by_size() == by_size and (by_size or integ.launch() == (3, 256, 1, 64, 0))
        cache = tmp_path / f"tuned{k}.json"
        cache.unlink(missing_ok=True)
        best, timings = at.autotune(bh, d, t, reps=1, cache=cache)
        assert set(timings) == set(at.CANDIDATES) and best == at.CANDIDATES[k]
        assert (bh.trace_config().reserved == abi.GZ_LAUNCH_BY_SIZE) == by_size
        bh.set_trace_config(1, 8, 32)
        again, none = at.autotune(bh, d, t, cache=cache)
        assert again == best and none == {}
        assert (bh.trace_config().reserved == abi.GZ_LAUNCH_BY_SIZE) == by_size
    integ.bh.free()
    bh.free()
