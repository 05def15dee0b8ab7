"""Draw sizes around the kernels' wave (64) and block (256) boundaries, frame by
frame against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle_lib as O
import retrofire_amd as rf
from retrofire_amd import batch as RB
from test_gpu_parity import random_soup

pytestmark = pytest.mark.gpu


def check_frame(w, h, draws, ctx, octx):
    """One batched frame of (kind, n) random draws equals the oracle's."""
    rng = np.random.default_rng([w, h] + [n for _, n in draws])
    fb = RB.DeviceFramebuf(w, h, 0, True)
    ocol = np.zeros((h, w, 4), np.uint8)
    ocol[...] = (0, 0, 0, 255)
    odep = np.zeros((h, w), np.float32)
    ost = np.zeros(8, np.uint64)
    tex = rng.integers(0, 256, size=(16, 16, 4), dtype=np.uint8)
    dtex = RB.Texture(tex)
    shaders = {0: rf.shader.Flat((9, 200, 77, 255)), 1: rf.shader.Gouraud(), 3: rf.shader.TexRepeatPot(tex)}
    meshes, mds = [], []
    for kind, n in draws:
        pos, attr, tris, mvp, vp = random_soup(rng, n, w, h, kind)
        meshes.append(RB.Mesh(pos, tris, attr))
        mds.append(RB.mesh_draw(meshes[-1], shaders[kind], mvp, vp, texture=dtex if kind == 3 else None))
        err, _ = O.render(kind, tris, pos, attr, mvp, vp, ocol, depth=odep, flat=(9, 200, 77, 255),
                          tex=tex if kind == 3 else None, ctx=octx, stats=ost)
        assert err == 0
    b = RB.Batch([(fb, ctx, mds)], tile_w=32)
    for _ in range(2):
        b.run()
        s = b.wait()[0]
        gcol, gdep = fb.read()
        assert np.array_equal(gcol, ocol)
        assert np.array_equal(gdep.view(np.uint32), odep.view(np.uint32))
        assert [s.calls, s.prims_i, s.prims_o, s.verts_i, s.verts_o, s.frags_i, s.frags_o] == [int(x) for x in ost[:7]]
    b.free()
    fb.free()
    dtex.free()
    for m in meshes:
        m.free()


@pytest.mark.parametrize("sizes", [(1,), (63, 1), (64, 65), (255, 2, 1), (256,), (257, 130, 3), (1, 1, 1, 1, 600)])
def test_sorted_draws_of_every_size(sizes):
    """Depth-sorted draws that end inside a wave, at its end and at a block's
    end, several in one block: each call's clip fans sort among themselves."""
    kinds = [1, 0, 3, 1, 3]
    check_frame(150, 90, [(kinds[i], n) for i, n in enumerate(sizes)],
                rf.Context(clear=True, depth_test=None, face_cull=None, depth_sort="back_to_front"), (0, 0, 1, 1, 2))
