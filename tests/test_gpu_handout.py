"""Work hand-out of the traversal launches: equal first shares, spread over
fewer lanes per wave in small launches, then pools from the per-XCD
counters.  Ray counts at the edges of those rules (one lane per wave and
its end, 64 lanes per wave, every wave's share and one unit more, several
pools) trace every ray once; so do ray batches under small grids, and
renders whose queued units lie on either side of the halved grid."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
MISS = 0xFFFFFFFF


def _scene(oracle):
    from voxvision_amd import scenes, voxtrees as VT
    dots = scenes.volume_to_dots(scenes.blobs64(3))
    bmin, bmax = scenes.bbox_of(dots)
    o, d = scenes.random_rays(4093, bmin, bmax, seed=17)
    vox, hit = oracle.Tree(dots).rays(o, d)
    return VT.make_tree(dots), o, d, vox, hit


def _check(G, o, d, vox, hit, n):
    """n rays, the base rays over and over (4093: no two neighbours of a
    wave or a pool repeat)."""
    from voxvision_amd import voxtrees as VT
    idx = np.arange(n) % len(o)
    i = torch.from_numpy(idx).cuda()
    og, dg = torch.from_numpy(o).cuda()[i], torch.from_numpy(d).cuda()[i]
    v, h = VT.ray_tree_intersection(G, og, dg)
    want = torch.from_numpy(vox.astype(np.int64)).cuda()[i]
    assert torch.equal(v, want)
    m = want != MISS
    wh = torch.from_numpy(hit).cuda()[:, i]
    assert torch.equal(h[:, m].view(torch.int32), wh[:, m].view(torch.int32))


@pytest.mark.parametrize("n", [1, 3, 2047, 2049, 131071, 131073, 524288,
                               524289, 8 * 1048576 + 5])
def test_every_ray_is_traced_once(gpu, oracle, n):
    _check(*_scene(oracle), n)


@pytest.mark.parametrize("waves,block", [(1, 64), (1, 256), (3, 192),
                                         (64, 128)])
def test_other_grids(gpu, oracle, waves, block):
    from voxvision_amd import voxtrees as VT
    s = _scene(oracle)
    with VT.saved_launch_configs():
        VT.set_launch_config("rays", waves_per_cu=waves, block=block)
        for n in (5, 40000, 300001):
            _check(*s, n)


@pytest.mark.parametrize("W,H,frames", [(16, 4, 1), (160, 120, 1),
                                        (1920, 1080, 1), (1920, 1080, 5)])
@pytest.mark.parametrize("quality", [0, 2, 6])
def test_renders_of_every_size(gpu, oracle, W, H, frames, quality):
    """The same frames one by one through whole-block units equal them
    together through the coherent one-pixel units, whatever the grid."""
    from voxvision_amd import scenes, voxrnd, voxtrees as VT
    dots = scenes.volume_to_dots(scenes.blobs64(3))
    G = VT.make_tree(dots)
    cams = scenes.orbit_cameras((32, 32, 32), 80.0, frames, W, H)
    out = voxrnd.render(G, cams, W, H, quality=quality, want_colors=False)
    v = out["voxel"].cpu().numpy()
    h = out["hit"].cpu().numpy()
    with VT.saved_launch_configs():
        for k in ("render", "render_best"):
            VT.set_launch_config(k, render_cull=0, split_best=0,
                                 waves_per_cu=5)
        ref = voxrnd.render(G, cams, W, H, quality=quality,
                            want_colors=False)
    assert np.array_equal(v, ref["voxel"].cpu().numpy())
    assert np.array_equal(h.view(np.uint32),
                          ref["hit"].cpu().numpy().view(np.uint32))
