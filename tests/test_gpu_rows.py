"""Rays and balls stored as rows against the calls that take one array per
coordinate: numbers around a lane's run of rays and a workgroup's tile, rows
at a 4-byte offset, strided and 64-bit inputs, missed rays with and without
hit_init, a hit_init that shares the rays' memory, and another stream.
Results are equal bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _tree():
    from voxvision_amd import scenes, voxtrees as VT
    return VT.make_tree(scenes.volume_to_dots(scenes.blobs64(3)))


def _rays(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    o = torch.rand((n, 3), device="cuda", generator=g) * 96 - 16
    return o, torch.randn((n, 3), device="cuda", generator=g)


def _columns(tree, o, d, nan):
    from voxvision_amd import _lib
    L = _lib.load()
    n = o.shape[0]
    oc, dc = o.t().contiguous(), d.t().contiguous()
    vox, leaf = (torch.empty(n, dtype=torch.int32, device="cuda")
                 for _ in range(2))
    hit = torch.full((3, n), nan, device="cuda")
    _lib.check(L.voxg_ray_batch(
        tree.handle, n, *[x.data_ptr() for x in oc],
        *[x.data_ptr() for x in dc], vox.data_ptr(), leaf.data_ptr(),
        *[x.data_ptr() for x in hit],
        torch.cuda.current_stream().cuda_stream))
    return (vox.to(torch.int64) & 0xFFFFFFFF, hit,
            leaf.to(torch.int64) & 0xFFFFFFFF)


def _same(a, b):
    return all(torch.equal(x.view(torch.int32), y.view(torch.int32))
               for x, y in zip(a, b))


@pytest.mark.parametrize("n", [1, 7, 8, 9, 65, 4097, 300001])
def test_rays_in_rows(gpu, n):
    from voxvision_amd import voxtrees as VT
    tree = _tree()
    o, d = _rays(n, n)
    want = _columns(tree, o, d, float("nan"))
    if n > 100:
        missed = want[0] == 0xFFFFFFFF
        assert bool(missed.any()) and not bool(missed.all())
    assert _same(VT.ray_tree_intersection(tree, o, d, want_leaf=True), want)
    assert _same(VT.ray_tree_intersection(tree, o, d), want[:2])
    # rows that start 4 bytes into an allocation, every other column's rows
    at = torch.empty(3 * n + 1, device="cuda")[1:].view(n, 3).copy_(o)
    wide = torch.empty((n, 6), dtype=torch.float64, device="cuda")
    wide[:, ::2] = d.double()
    assert _same(VT.ray_tree_intersection(tree, at, wide[:, ::2]), want[:2])
    assert _same(VT.ray_tree_intersection(tree, o.cpu().numpy(), d.cpu()),
                 want[:2])
    init = torch.full((3, n), -7.0, device="cuda")
    got = VT.ray_tree_intersection(tree, o, d, hit_init=init)
    assert got[1] is init and _same(got, _columns(tree, o, d, -7.0)[:2])
    both = torch.empty((2 * n, 3), device="cuda")
    both[:n] = o
    shared = both[:n].view(3, n)
    fill = shared.clone()
    got = VT.ray_tree_intersection(tree, both[:n], d, hit_init=shared)
    assert torch.equal(got[0], want[0])
    assert torch.equal(shared, torch.where(want[0] == 0xFFFFFFFF, fill,
                                           want[1]))
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        got = VT.ray_tree_intersection(tree, o, d)
    side.synchronize()
    assert _same(got, want[:2])


@pytest.mark.parametrize("n", [1, 64, 65, 70001])
def test_balls_in_rows(gpu, n):
    from voxvision_amd import _lib, voxtrees as VT
    tree = _tree()
    c, _ = _rays(n, 7 * n)
    r = torch.rand(n, device="cuda") * 6
    cc = c.t().contiguous()
    want = torch.empty(n, dtype=torch.uint8, device="cuda")
    _lib.check(_lib.load().voxg_ball_batch(
        tree.handle, n, *[x.data_ptr() for x in cc], r.data_ptr(),
        want.data_ptr(), torch.cuda.current_stream().cuda_stream))
    assert torch.equal(VT.tree_ball_collidep(tree, c, r), want)
    at = torch.empty(3 * n + 1, device="cuda")[1:].view(n, 3).copy_(c)
    assert torch.equal(VT.tree_ball_collidep(tree, at, r.double()), want)


def test_too_few_rows(gpu):
    from voxvision_amd import voxtrees as VT
    tree = _tree()
    o, d = _rays(9, 1)
    with pytest.raises(ValueError):
        VT.ray_tree_intersection(tree, o, d[:8])
    with pytest.raises(ValueError):
        VT.tree_ball_collidep(tree, o, torch.ones(8))
