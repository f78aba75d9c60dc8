"""Which trees take the division-free tests (voxvision_amd/csrc/raymath.h and
tree_build.h): tree_build.cpp compiled for the host with g++ says so for built
and for uploaded trees with coordinates on either side of 2^60, a voxel size
beyond it, infinities, NaN and an inverted box, in top levels, in subtrees and
in leaves.  On the GPU, trees on either side answer rays, balls, bodies and
renders as the oracle does."""
import os
import subprocess

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include "tree_build.h"
#include <math.h>
#include <stdio.h>
using namespace voxg;

static int bad;
static std::vector<float> grid(float scale, float x) {
    std::vector<float> p;
    for (int i = 0; i < 40; i++)
        for (int j = 0; j < 40; j++)
            for (int k = 0; k < 40; k++)
                if ((i * 7 + j * 5 + k * 3) % 11 == 0)
                    for (int c : {i, j, k}) p.push_back(scale * (float)c);
    p[3 * (p.size() / 6)] += x;
    return p;
}
static void built(const char *what, const std::vector<float> &p, float v, bool want) {
    HostTree h;
    std::string err;
    const float V[3] = {v, v, v};
    if (build_tree(p.data(), p.size() / 3, 3, V, h, err) || plain(h) != want) {
        printf("built %s: plain %d\n", what, (int)plain(h));
        bad++;
    }
}
// the last regular leaf and the node above it
static void find(struct vox_node *at, struct vox_node *&leaf, struct vox_node *&above) {
    for (struct vox_node *c : at->data.inner.children) {
        if (!c) continue;
        if (!(c->flags & VOX_LEAF_MASK)) find(c, leaf, above);
        else if (!(c->flags & VOX_DENSE_LEAF)) {
            leaf = c;
            above = at;
        }
    }
}
static void uploaded(const char *what, int at, float value, bool want) {
    // a reference-layout tree of the grid with one number changed: `at` says
    // where (0 the root's box, 1 a deep node's box, 2 a dot, 3 a centre)
    std::vector<float> p = grid(1.0f, 0.0f);
    const float V[3] = {1, 1, 1};
    std::string err;
    struct vox_node *root = nullptr;
    if (build_reference(p.data(), p.size() / 3, 3, V, &root, err)) { bad++; return; }
    struct vox_node *n = nullptr, *inner = nullptr;
    find(root, n, inner);
    if (!n || inner == root) { bad++; return; }
    float *w = at == 0 ? &root->bounding_box.max[1]
             : at == 1 ? &n->bounding_box.min[2]
             : at == 2 ? &n->data.dots[0][0] : &inner->data.inner.center[2];
    const float was = *w;
    *w = value;
    HostTree h;
    if (flatten_reference(root, V, h, err) || plain(h) != want) {
        printf("uploaded %s: plain %d\n", what, (int)plain(h));
        bad++;
    }
    *w = was;
    destroy_reference(root);
}
int main(void) {
    const float t60 = 0x1p60f, over = nextafterf(0x1p60f, INFINITY);
    built("unit", grid(1.0f, 0.0f), 1.0f, true);
    built("2^54", grid(0x1p54f, 0.0f), 0x1p54f, true);
    built("2^55 cells of 40", grid(0x1p55f, 0.0f), 0x1p55f, false);
    built("2^100", grid(0x1p100f, 0.0f), 0x1p100f, false);
    built("one dot at -2^60", grid(1.0f, -t60), 1.0f, true);
    built("one dot below it", grid(1.0f, -over), 1.0f, false);
    built("an infinite dot", grid(1.0f, INFINITY), 1.0f, false);
    built("a large voxel", grid(1.0f, 0.0f), over, false);
    for (int at = 0; at < 4; at++) {
        const bool low = at == 1;  // a lower corner may not exceed the upper
        uploaded("2^60", at, low ? -t60 : t60, true);
        uploaded("beyond", at, low ? -over : over, false);
        uploaded("infinite", at, -INFINITY, false);
        uploaded("nan", at, NAN, false);
    }
    uploaded("inverted", 1, 1e6f, false);
    HostTree h;
    std::string err;
    const float V[3] = {1, 1, 1};
    bad += build_tree(nullptr, 0, 3, V, h, err) != 0;
    printf("bad %d\n", bad);
    return bad != 0;
}
"""


def test_which_trees_are_plain(tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(CHECK)
    csrc = os.path.join(ROOT, "voxvision_amd", "csrc")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-pthread",
                        "-ffp-contract=off", "-I", csrc, str(src),
                        os.path.join(csrc, "tree_build.cpp"), "-o", str(exe)],
                       capture_output=True, text=True)
    if r.returncode:
        pytest.fail(r.stderr)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("voxel", [2.0 ** 53, 2.0 ** 56, 2.0 ** 62])
def test_large_trees_on_the_gpu(gpu, oracle, voxel):
    """64 cells an axis: coordinates to 2^59, 2^62 and 2^68 (there squared
    distances overflow)."""
    from voxvision_amd import scenes, voxrnd, voxtrees as VT
    from voxvision_amd.camera import set_window_size
    rng = np.random.default_rng(60)
    V = (voxel,) * 3
    dots = scenes.volume_to_dots(scenes.blobs64(3))[:, :3] * np.float32(voxel)
    T, G = oracle.Tree(dots, V), VT.make_tree(dots, V)
    assert G.hash() == T.hash()
    n = 20000
    o, d = scenes.random_rays(n, np.zeros(3), np.full(3, 64.0), seed=8)
    o = (o * voxel).astype(np.float32)
    vo, ho = T.rays(o, d)
    vg, hg = VT.ray_tree_intersection(G, o, d)
    hits = vo != oracle.MISS
    assert np.array_equal(vg.cpu().numpy().astype(np.uint32), vo)
    assert np.array_equal(hg.cpu().numpy()[:, hits].view(np.uint32),
                          ho[:, hits].view(np.uint32))
    assert 0 < hits.sum() < n
    c = (rng.uniform(-2, 66, (n, 3)) * voxel).astype(np.float32)
    r = (rng.uniform(0.2, 6, n) * voxel).astype(np.float32)
    want = T.balls(c, r)
    for _ in range(2):
        assert np.array_equal(VT.tree_ball_collidep(G, c, r).cpu().numpy(), want)
        G.prepare_balls()
    pos = [torch.from_numpy(np.ascontiguousarray(c[:, k])).cuda() for k in range(3)]
    last = [x + np.float32(8 * voxel) for x in pos]
    hit = voxrnd.cd_collide(G, pos, last, torch.from_numpy(r).cuda())
    assert np.array_equal(hit.cpu().numpy(), want)
    if voxel > 2.0 ** 60:
        return
    W, H = 64, 48
    cam = dict(scenes.orbit_cameras((32, 32, 32), 90.0, 1, W, H)[0])
    cam["position"] = [float(x) * voxel for x in cam["position"]]
    cam["mul"], cam["xsub"], cam["ysub"] = set_window_size(cam["fov"], W, H)
    for q in (oracle.QUALITY_BEST, oracle.QUALITY_ADAPTIVE):
        out = voxrnd.render(G, [cam], W, H, quality=q, want_colors=False)
        _, v, h, _ = T.render(cam, W, H, q)
        m = v != oracle.MISS
        assert np.array_equal(out["voxel"].cpu().numpy().view(np.uint32), v)
        assert np.array_equal(out["hit"].cpu().numpy()[:, m].view(np.uint32),
                              h[:, m].view(np.uint32))
        assert 0 < m.sum() < m.size
