"""The corners of a raw selection against a NumPy scan: rows shorter than a
32-sample mask, of one mask and ragged ones, selections that are sparse,
clustered, full and empty, one and more groups of tiles, and a capacity that
ends inside a wave."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _volume(dim, how, rng):
    n = dim[0] * dim[1] * dim[2]
    if how == "sparse":
        return (rng.random(n) < 0.01).astype(np.uint8) * 9
    if how == "half":
        return (rng.random(n) < 0.5).astype(np.uint8) * 9
    if how == "full":
        return np.full(n, 9, np.uint8)
    if how == "none":
        return np.zeros(n, np.uint8)
    # runs of 1 to 3000 samples
    v = np.zeros(n, np.uint8)
    at = 0
    while at < n:
        run = int(rng.integers(1, 3000))
        v[at:at + run] = 9 * int(rng.integers(0, 2))
        at += run
    return v


@pytest.mark.parametrize("dim", [(1, 1, 1), (5, 7, 1), (9, 1, 3), (40, 30, 31),
                                 (17, 20, 32), (3, 3, 8193), (60, 61, 63),
                                 (1, 300001, 29)])
@pytest.mark.parametrize("how", ["sparse", "half", "full", "none", "runs"])
def test_raw_corners(gpu, dim, how):
    import torch
    from voxvision_amd import _lib, voxtrees as VT
    rng = np.random.default_rng(dim[2] + len(how))
    v = _volume(dim, how, rng)
    at = np.flatnonzero(v > 4)
    scale = np.array([0.5, 1.25, 3.0], np.float32)
    want = np.stack(np.unravel_index(at, dim), 1).astype(np.float32) * scale
    dev = torch.from_numpy(v).cuda()
    got = VT.raw_select(dev, dim, 1, threshold=4, voxel=tuple(scale))
    assert np.array_equal(got.cpu().numpy(), want)
    # a shorter output: nothing is written behind it
    m = max(1, len(at) * 2 // 3)
    L = _lib.load()
    d = (C.c_uint * 3)(*dim)
    vs = (C.c_float * 3)(*[float(x) for x in scale])
    out = torch.full((m + 4, 3), -1.0, device="cuda")
    cnt = torch.empty(1, dtype=torch.int64, device="cuda")
    _lib.check(L.voxg_raw_select(dev.data_ptr(), d, 1, 5, 256, vs,
                                 out.data_ptr(), m, cnt.data_ptr(), None))
    torch.cuda.synchronize()
    assert int(cnt.item()) == len(at)
    k = min(m, len(at))
    assert np.array_equal(out[:k].cpu().numpy(), want[:k])
    assert bool((out[k:] == -1.0).all())
