"""Ray, ball, count and selection calls with `stream` naming another stream than the current
one: the inputs are written on the current stream behind queued work and
overwritten right after the call, the call's temporaries are dropped and
their memory asked for again while the other stream is still busy, and the
stream may be any object with a `cuda_stream`.  Results equal those of the
same call on the current stream."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu


def _scene(n):
    from voxvision_amd import scenes, voxtrees as VT
    tree = VT.make_tree(scenes.volume_to_dots(scenes.blobs64(3)))
    g = torch.Generator(device="cuda").manual_seed(n)
    o = torch.rand((n, 3), device="cuda", generator=g) * 96 - 16
    d = torch.randn((n, 3), device="cuda", generator=g)
    r = torch.rand(n, device="cuda", generator=g) * 6
    return VT, tree, o, d, r


def _busy(big):
    for _ in range(30):  # about 3 ms on this card
        big.add_(1.0)


def _same(a, b):
    return all(torch.equal(x.view(torch.int32), y.view(torch.int32))
               for x, y in zip(a, b))


@pytest.mark.parametrize("n", [1, 4096, 300001])
@pytest.mark.parametrize("busy", ["current", "other"])
@pytest.mark.parametrize("plain", [False, True])
def test_another_stream(gpu, n, busy, plain):
    VT, tree, o, d, r = _scene(n)
    rays = VT.ray_tree_intersection(tree, o, d, want_leaf=True)
    init = torch.full((3, n), -7.0, device="cuda")
    kept = VT.ray_tree_intersection(tree, o, d, hit_init=init.clone())
    balls = VT.tree_ball_collidep(tree, o, r)
    # the calls of a stream allocate its workspace the first time
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        VT.ray_tree_intersection(tree, o, d)
        VT.tree_ball_collidep(tree, o, r)
    big = torch.zeros(1 << 26, device="cuda")
    big2 = torch.zeros(1 << 26, device="cuda")
    ins = [torch.full_like(x, float("nan")) for x in (o, d, r)]
    torch.cuda.synchronize()
    st = types.SimpleNamespace(cuda_stream=side.cuda_stream) if plain else side
    if busy == "current":
        _busy(big)
    else:
        with torch.cuda.stream(side):
            _busy(big2)
    for x, y in zip(ins, (o, d, r)):
        x.copy_(y)
    init = torch.full((3, n), -7.0, device="cuda")
    a = VT.ray_tree_intersection(tree, ins[0], ins[1], want_leaf=True,
                                 stream=st)
    b = VT.ray_tree_intersection(tree, ins[0], ins[1], hit_init=init,
                                 stream=st)
    c = VT.tree_ball_collidep(tree, ins[0], ins[2], stream=st)
    for x in ins:
        x.fill_(float("nan"))
    again = [torch.full(x.shape, float("nan"), device="cuda")
             for x in ins for _ in range(4)]
    side.synchronize()
    assert _same(a, rays)
    assert _same(b, kept)
    assert torch.equal(c, balls)
    del again


@pytest.mark.parametrize("busy", ["current", "other"])
def test_counts_and_selection_on_another_stream(gpu, busy):
    VT, tree, o, d, r = _scene(5000)
    dim = (96, 80, 64)
    raw = (torch.arange(96 * 80 * 64, device="cuda") * 37 % 251).to(torch.uint8)
    want = (VT.ray_counts(tree, o, d), VT.ball_counts(tree, o, r),
            VT.raw_select(raw, dim, 1, threshold=200))
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        VT.ray_counts(tree, o, d)
        VT.raw_select(raw, dim, 1, threshold=200)
    big = torch.zeros(1 << 26, device="cuda")
    ins = [torch.full_like(x, float("nan")) for x in (o, d, r)]
    src = torch.zeros_like(raw)
    torch.cuda.synchronize()
    for k in range(3):
        if busy == "current":
            _busy(big)
        else:
            with torch.cuda.stream(side):
                _busy(big)
        if k == 0:
            ins[0].copy_(o)
            ins[1].copy_(d)
            got = VT.ray_counts(tree, ins[0], ins[1], stream=side)
        elif k == 1:
            ins[2].copy_(r)
            got = VT.ball_counts(tree, ins[0], ins[2], stream=side)
        else:
            src.copy_(raw)
            got = VT.raw_select(src, dim, 1, threshold=200, stream=side)
            again = [torch.full_like(got, -1.0) for _ in range(4)]
            side.synchronize()
            assert torch.equal(got, want[k])
            del again
        if k < 2:
            assert got == want[k]
        torch.cuda.synchronize()
