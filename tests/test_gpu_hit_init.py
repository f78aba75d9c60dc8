"""hit_init in the forms a caller may hold it: three arrays of their own, a
longer array per coordinate, and memory that overlaps the rays without being
the same storage."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _scene(n):
    from voxvision_amd import scenes, voxtrees as VT
    tree = VT.make_tree(scenes.volume_to_dots(scenes.blobs64(3)))
    g = torch.Generator(device="cuda").manual_seed(n)
    o = torch.rand((n, 3), device="cuda", generator=g) * 96 - 16
    d = torch.randn((n, 3), device="cuda", generator=g)
    vox, hit = VT.ray_tree_intersection(tree, o, d)
    return VT, tree, o, d, vox, hit


@pytest.mark.parametrize("form", [list, tuple])
@pytest.mark.parametrize("n,extra", [(1, 0), (5000, 0), (5000, 7)])
def test_three_arrays(gpu, form, n, extra):
    VT, tree, o, d, vox, hit = _scene(n)
    init = form(torch.full((n + extra,), -7.0, device="cuda")
                for _ in range(3))
    v, h = VT.ray_tree_intersection(tree, o, d, hit_init=init)
    assert h is init and torch.equal(v, vox)
    for k in range(3):
        assert torch.equal(h[k][:n], torch.where(vox == 0xFFFFFFFF, -7.0,
                                                 hit[k]))
        assert bool((h[k][n:] == -7.0).all())


@pytest.mark.parametrize("at", [0, 1, 5000, 10000])
def test_overlap_of_another_storage(gpu, at):
    n = 5000
    VT, tree, o, d, vox, hit = _scene(n)
    mem = torch.empty(6 * n, device="cuda")
    mem[:3 * n] = o.reshape(-1)
    # a tensor of its own over the same memory, from `at` floats on
    init = torch.from_dlpack(mem[at:at + 3 * n]).view(3, n)
    assert init.untyped_storage().data_ptr() == mem.data_ptr() + 4 * at
    fill = init.clone()
    v, h = VT.ray_tree_intersection(tree, mem[:3 * n].view(n, 3), d,
                                    hit_init=init)
    assert torch.equal(v, vox)
    want = torch.where(vox == 0xFFFFFFFF, fill, hit)
    assert torch.equal(h.view(torch.int32), want.view(torch.int32))
