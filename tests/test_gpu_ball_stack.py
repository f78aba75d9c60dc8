"""Ball queries whose pending inner nodes outgrow a group's stack: trees in the
reference's layout, a chain of nodes with seven siblings each that the ball
touches and that hold nothing near it.  The group's steps are followed on the
host, so that the stack is known to overflow, at the fewest levels that do it
and at more, or to hold at one level less; answers equal the oracle's."""
import ctypes as C
import os
import re

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LEAF = 1


class _Node(C.Structure):
    """struct vox_node (include/voxgpu.h)."""
    _fields_ = [("min", C.c_float * 4), ("max", C.c_float * 4),
                ("flags", C.c_uint), ("dots_num", C.c_uint),
                ("align", C.c_uint * 2), ("center", C.c_float * 4),
                ("children", C.c_void_p * 8)]


class _Chain:
    def __init__(self, levels):
        self.mem = np.zeros((16 * levels + 64) * 128 + 16, np.uint8)
        self.dots = np.zeros(64 * (8 * levels + 16) + 16, np.uint8)
        self.at = -(-self.mem.ctypes.data // 16) * 16
        self.dot_at = -(-self.dots.ctypes.data // 16) * 16
        self.nodes = []
        # the last node of the chain: a voxel 8 away from the middle
        end = self.inner([self.leaf([(40, 32, 32), (41, 33, 33)]),
                          self.leaf([(1, 1, 1), (2, 2, 2)])])
        for k in range(levels):
            corner = [(1 + 61 * (k >> j & 1)) for j in range(3)]
            end = self.inner([self.inner([self.leaf(
                [corner, [x + 1 for x in corner]])]) for _ in range(7)] + [end])
        self.root = end

    def _new(self):
        nd = _Node.from_address(self.at + 128 * len(self.nodes))
        self.nodes.append(nd)
        return nd

    def leaf(self, voxels):
        nd = self._new()
        v = np.array(voxels, np.float32)
        nd.min[:3], nd.max[:3] = v.min(0).tolist(), (v.max(0) + 1).tolist()
        nd.flags, nd.dots_num = LEAF, len(voxels)
        out = np.ctypeslib.as_array((C.c_float * (4 * len(v))).from_address(
            self.dot_at)).reshape(-1, 4)
        out[:, :3] = v
        C.c_void_p.from_address(C.addressof(nd) + 48).value = self.dot_at
        self.dot_at += out.nbytes
        return nd

    def inner(self, children):
        nd = self._new()
        nd.min[:3], nd.max[:3], nd.center[:3] = [0] * 3, [64] * 3, [32] * 3
        for k, c in enumerate(children):
            nd.children[k] = C.addressof(c)
        return nd

    def pending(self, c, r):
        """The most entries that a group asks its stack for."""
        def touches(nd):
            lo, hi = np.array(nd.min[:3]), np.array(nd.max[:3])
            return ((np.clip(c, lo, hi) - c) ** 2).sum() < r * r
        stack, most = [self.root], 0
        while stack:
            nd = stack.pop()
            near = [k for k in (_Node.from_address(p) for p in nd.children if p)
                    if touches(k)]
            add = [k for k in near if not k.flags]
            most = max(most, len(stack) + len(add))
            stack += add
        return most


def _stack_size():
    src = open(os.path.join(ROOT, "voxvision_amd", "csrc", "voxgpu.hip")).read()
    return int(re.search(r"kBallStack = (\d+);", src).group(1))


@pytest.mark.parametrize("more", [-1, 0, 1, 8])
def test_stack(gpu, oracle, more):
    from voxvision_amd import voxrnd, voxtrees as VT
    size = _stack_size()
    fewest = 1
    while _Chain(fewest).pending(np.full(3, 32.0), 5.0) <= size:
        fewest += 1
    chain = _Chain(fewest + more)
    ask = chain.pending(np.full(3, 32.0), 5.0)
    assert (ask > size) == (more >= 0)
    rng = np.random.default_rng(more + 2)
    n = 3000
    c = np.full((n, 3), 32.0, np.float32)
    r = rng.choice(np.float32([5.0, 7.9, 8.1, 20.0, 70.0]), n)
    c[n // 2:] += rng.normal(0, 4, (n - n // 2, 3)).astype(np.float32)
    ptr = C.addressof(chain.root)
    L = oracle.lib()
    oracle.set_voxel()
    want = np.zeros(n, np.uint8)
    col = [np.ascontiguousarray(c[:, k]) for k in range(3)] + [r]
    L.orc_ball_batch(ptr, n, *[oracle._fp(x) for x in col],
                     want.ctypes.data_as(C.POINTER(C.c_uint8)), 0,
                     C.byref(oracle._Counters()))
    assert 0 < want.sum() < n
    G = VT.Tree.upload(ptr)
    for _ in range(2):
        got = VT.tree_ball_collidep(G, c, r).cpu().numpy()
        assert np.array_equal(got, want)
        pos = [torch.from_numpy(x.copy()).cuda() for x in col[:3]]
        last = [x + 1.0 for x in pos]
        hit = voxrnd.cd_collide(G, pos, last, torch.from_numpy(r).cuda())
        assert np.array_equal(hit.cpu().numpy(), want)
        G.prepare_balls()
