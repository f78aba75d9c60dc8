"""FAST and ADAPTIVE renders on either side of the size where the replay
takes 16 lanes per block: a call of several frames is a large one, its frames
one by one are small ones (or the largest small one); cameras near, far,
inside and beside the scene.  Outputs are equal bit for bit."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _render(G, cams, W, H, quality, texture, lights):
    from voxvision_amd import voxrnd
    out = voxrnd.render(G, cams, W, H, quality=quality, texture=texture,
                        lights=lights)
    return [out["squares"].view(len(cams), -1), out["voxel"].view(len(cams), -1),
            out["hit"].view(torch.int32).view(3, len(cams), -1).transpose(0, 1)]


@pytest.mark.parametrize("W,H,scene", [(640, 480, "blobs"), (640, 480, "ct"),
                                       (1024, 1024, "ct")])
@pytest.mark.parametrize("lit", [False, True])
def test_small_and_large_calls(gpu, W, H, scene, lit):
    from voxvision_amd import lights, scenes, voxrnd, voxtrees as VT
    n = 64 if scene == "blobs" else 100
    occ = scenes.blobs64(2) if scene == "blobs" else scenes.ct_volume(n, 3)
    G = VT.make_tree(scenes.volume_to_dots(occ))
    mid = (n / 2.0,) * 3
    cams = []
    for k, far in enumerate((1.5, 0.7, 0.2, 4.0)):
        cams += scenes.orbit_cameras(mid, far * n * math.sqrt(3.0), 1, W, H,
                                     phase=0.7 * k)
    side = scenes.orbit_cameras((n, 0.0, n), 0.5 * n, 1, W, H, phase=2.0)
    cams[3:] = side + cams[3:]
    g = torch.Generator(device="cuda").manual_seed(3)
    tex = torch.randint(64, 256, (32, 32, 32), dtype=torch.uint8,
                        device="cuda", generator=g)
    L = None
    if lit:
        L = lights.Lights()
        L.set_ambient((0.2, 0.3, 0.4))
        for k in range(9):
            L.insert((n * (k % 3) / 2.0, n * (k // 3) / 2.0, mid[2]), n * 0.4,
                     (0.1 * k, 0.5, 1.0 - 0.1 * k))
    assert len(cams) * W * H // 16 > 1 << 16 >= W * H // 16
    for quality in (1, 2):
        large = _render(G, voxrnd.cameras_tensor(cams), W, H, quality, tex, L)
        hits = (large[1] != -1).sum(1)
        assert bool((hits[:3] > 0).all())
        for k, cam in enumerate(cams):
            small = _render(G, voxrnd.cameras_tensor([cam]), W, H, quality,
                            tex, L)
            for a, b in zip(small, large):
                assert torch.equal(a[0], b[k]), (quality, k)
    best = _render(G, voxrnd.cameras_tensor(cams), W, H, 0, tex, L)
    # the replay's leaf tries change some pixels
    assert not torch.equal(best[1], large[1])
