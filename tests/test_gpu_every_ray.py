"""Every entry of a ray call's outputs is written, whatever the hand-out of
the rays: the arrays hold marks that no ray has (an id of -2, a point at
12345) before the call, for numbers of rays at the edges of the hand-out's
rules and for other grids, through the calls that take rows, one array per
coordinate, and a batch of trees."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
MISS = 0xFFFFFFFF


@pytest.fixture(scope="module")
def scene(oracle):
    from voxvision_amd import scenes, voxtrees as VT
    dots = scenes.volume_to_dots(scenes.blobs64(3))
    o, d = scenes.random_rays(4093, *scenes.bbox_of(dots), seed=17)
    vox, hit = oracle.Tree(dots).rays(o, d)
    assert 0 < int((vox == MISS).sum()) < len(vox)
    hit[:, vox == MISS] = np.nan
    return (VT.make_tree(dots), torch.from_numpy(o).cuda(),
            torch.from_numpy(d).cuda(),
            torch.from_numpy(vox.astype(np.int64)).cuda(),
            torch.from_numpy(hit).cuda())


def _check(scene, n, how):
    from voxvision_amd import _lib, batch
    L = _lib.load()
    G, o, d, vox, hit = scene
    i = torch.arange(n, device="cuda") % len(o)
    o, d, vox, hit = o[i], d[i], vox[i], hit[:, i]
    st = torch.cuda.current_stream().cuda_stream
    word = torch.int64 if how == "rows" else torch.int32
    v = torch.full((n,), -2, dtype=word, device="cuda")
    leaf = torch.full((n,), -2, dtype=word, device="cuda")
    h = torch.full((3, n), 12345.0, device="cuda")
    if how == "rows":
        _lib.check(L.voxg_ray_batch_rows(
            G.handle, n, o.data_ptr(), d.data_ptr(), v.data_ptr(),
            leaf.data_ptr(), *[x.data_ptr() for x in h], 1, st))
    else:
        so, sd = batch.soa(o), batch.soa(d)
        if how == "columns":
            _lib.check(L.voxg_ray_batch(
                G.handle, n, *[x.data_ptr() for x in so + sd], v.data_ptr(),
                leaf.data_ptr(), *[x.data_ptr() for x in h], st))
        else:
            k = n // 3
            B = batch.Batch([(G, 0, k), (G, k, n - k)] if k else [(G, 0, n)])
            B.ray(so, sd, v, leaf=leaf, hit=h)
    assert not bool((v == -2).any()) and not bool((leaf == -2).any())
    assert torch.equal(v.to(torch.int64) & MISS, vox)
    miss = vox == MISS
    assert torch.equal((leaf.to(torch.int64) & MISS) == MISS, miss)
    if how != "rows":  # a miss leaves the point as it was
        assert bool((h[:, miss] == 12345.0).all())
        hit = torch.where(miss, h, hit)
    assert torch.equal(h.view(torch.int32), hit.contiguous().view(torch.int32))


@pytest.mark.parametrize("how", ["rows", "columns", "batch"])
@pytest.mark.parametrize("n", [1, 3, 2047, 2049, 131071, 131073, 524288,
                               524289, 8 * 1048576 + 5])
def test_every_entry(gpu, scene, n, how):
    _check(scene, n, how)


@pytest.mark.parametrize("how", ["rows", "columns", "batch"])
@pytest.mark.parametrize("waves,block", [(1, 64), (1, 256), (3, 192),
                                         (64, 128)])
def test_other_grids(gpu, scene, waves, block, how):
    from voxvision_amd import voxtrees as VT
    with VT.saved_launch_configs():
        VT.set_launch_config("batch" if how == "batch" else "rays",
                             waves_per_cu=waves, block=block)
        for n in (5, 40000, 300001):
            _check(scene, n, how)
