"""Tiles of Z-Sobol samples on both sides of the grouped kernel's rule (samples per pixel a power of two,
indexes below 2^32), bit-exact against the oracle: every group width, odd and even sample bits, the wrap
of the last dimensions, both layouts, partial last waves."""
import ctypes

import numpy as np
import pytest

import oracle
from gonzales_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spp,res,x0,y0,w,h,start", [
    (1, 512, 3, 5, 37, 11, 0), (2, 512, 0, 0, 33, 3, 0), (4, 640, 100, 40, 17, 9, 1), (8, 1920, 1900, 1000, 13, 7, 0),
    (16, 1920, 7, 3, 19, 5, 0), (32, 1920, 0, 9, 11, 3, 1020), (64, 64, 60, 60, 4, 4, 1022), (512, 512, 1, 1, 3, 2, 0),
    (12, 512, 5, 6, 9, 7, 0), (3, 512, 0, 0, 9, 7, 0),             # not a power of two: the general kernel
    (4, 1 << 16, (1 << 15) - 3, 0, 3, 2, 0), (4, 1 << 16, (1 << 15) - 2, 0, 3, 2, 0),  # the line of the 32-bit index
    (16, 64, 500, 700, 5, 3, 0)])                                  # pixels beyond the digits of the resolution
@pytest.mark.parametrize("layout", [0, 1])
def test_tiles_match_the_oracle(gpu, spp, res, x0, y0, w, h, start, layout):
    import torch

    lib = abi.load()
    p = abi.GzZSobolParams()
    abi.check(lib.gz_zsobol_params(spp, res, res, 77, ctypes.byref(p)))
    pat = np.array([2, 1, 3, 2], np.int8)
    n = w * h * spp
    out = torch.full((n * 8 + 64,), -1.0, dtype=torch.float32, device="cuda")
    abi.check(lib.gz_zsobol_tile_device(ctypes.byref(p), x0, y0, w, h, spp, start, pat.ctypes.data, len(pat),
                                        abi.ptr(out), layout, abi.stream_ptr()))
    torch.cuda.synchronize()
    assert bool((out[n * 8:] == -1.0).all())
    o = out[:n * 8].cpu().numpy()
    got = o.reshape(n, 8) if layout == 0 else o.reshape(8, n).T
    pix = np.repeat(np.arange(w * h), spp)
    ref = oracle.zsobol_batch(spp, res, res, 77, x0 + pix % w, y0 + pix // w, np.tile(np.arange(spp), w * h), pat, start)
    assert np.array_equal(np.ascontiguousarray(got).view(np.uint32), ref.view(np.uint32))
