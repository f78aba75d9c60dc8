"""Ball queries at the sizes where their kernel can go wrong: one query, the
edges of a workgroup's tile at its smallest and largest, queries that the
grid answers and queries that it does not, centres outside the box, a hollow
shell whose pending nodes overflow a group's stack, a tree of one leaf, and
bodies; answers equal the oracle's."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _scene(kind):
    from voxvision_amd import scenes
    if kind == "blobs":
        return scenes.volume_to_dots(scenes.blobs64(2))
    if kind == "shell":
        return scenes.volume_to_dots(scenes.shell_volume(150, 0.02))
    return np.array([[3, 4, 5], [4, 4, 5], [9, 4, 5]], np.float32)


def _balls(dots, n, seed):
    """Centres in the box and around it, radii from a voxel to the box."""
    rng = np.random.default_rng(seed)
    lo, hi = dots.min(0) - 3.0, dots.max(0) + 4.0
    c = rng.uniform(lo, hi, (n, 3)).astype(np.float32)
    r = np.exp(rng.uniform(np.log(0.3), np.log(0.5 * (hi - lo).max()),
                           n)).astype(np.float32)
    # balls around the middle that just miss or just reach the voxels
    mid = ((lo + hi) / 2).astype(np.float32)
    k = n // 3
    c[:k] = mid + rng.normal(0, 0.5, (k, 3)).astype(np.float32)
    near = np.sqrt((np.maximum(np.maximum(dots - mid, mid - dots - 1), 0)
                    ** 2).sum(1).min())
    r[:k] = near + rng.normal(0, 0.3, k).astype(np.float32)
    return c, r


@pytest.mark.parametrize("kind", ["blobs", "shell", "leaf"])
def test_balls_of_every_kind(gpu, oracle, kind):
    from voxvision_amd import voxtrees as VT
    dots = _scene(kind)
    c, r = _balls(dots, 5000, 5)
    want = oracle.Tree(dots).balls(c, r)
    got = VT.tree_ball_collidep(VT.make_tree(dots), c, r).cpu().numpy()
    assert np.array_equal(got, want)
    assert 0 < want.sum() < len(want)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 131071, 1048575, 1048577,
                               1100000])
def test_tiles_of_every_size(gpu, oracle, n):
    from voxvision_amd import voxtrees as VT
    dots = _scene("blobs")
    c, r = _balls(dots, 4093, 9)
    want = torch.from_numpy(oracle.Tree(dots).balls(c, r)).cuda()
    i = torch.arange(n, device="cuda") % len(c)
    got = VT.tree_ball_collidep(VT.make_tree(dots), torch.from_numpy(c).cuda()[i],
                                torch.from_numpy(r).cuda()[i])
    assert torch.equal(got, want[i])


@pytest.mark.parametrize("n", [1, 65, 70001])
def test_bodies(gpu, oracle, n):
    from voxvision_amd import voxrnd, voxtrees as VT
    dots = _scene("blobs")
    c, r = _balls(dots, n, 21)
    last = c + np.float32(1.0)
    still = np.arange(n) % 5 == 3
    last[still] = c[still]
    G = VT.make_tree(dots)
    pos = [torch.from_numpy(np.ascontiguousarray(c[:, k])).cuda() for k in range(3)]
    lst = [torch.from_numpy(np.ascontiguousarray(last[:, k])).cuda()
           for k in range(3)]
    hit = voxrnd.cd_collide(G, pos, lst, torch.from_numpy(r).cuda())
    want = oracle.Tree(dots).balls(c, r).astype(bool) & ~still
    assert np.array_equal(hit.cpu().numpy().astype(bool), want)
    p = np.stack([t.cpu().numpy() for t in pos], 1)
    q = np.stack([t.cpu().numpy() for t in lst], 1)
    assert np.array_equal(p, np.where(want[:, None], last, c))
    assert np.array_equal(q, np.where(want[:, None], last, c))
