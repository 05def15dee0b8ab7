"""Draw sizes around the kernels' wave (64) and block (256) boundaries, frame by
frame against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle_lib as O
import retrofire_amd as rf
from retrofire_amd import batch as RB
from retrofire_amd import mat as M
from test_gpu_parity import random_soup

pytestmark = pytest.mark.gpu


def small_soup(rng, n, w, h, kind):
    """Triangles a few pixels wide, slivers among them, at random depths: most
    are hidden once some layers are drawn."""
    pos, attr, tris, mvp, vp = random_soup(rng, n, w, h, kind)
    pos = pos.reshape(n, 3, 3)
    size = rng.choice([0.0, 0.02, 0.1, 0.3], n).astype(np.float32)
    pos[:, 1:] = pos[:, :1] + (pos[:, 1:] - pos[:, :1]) * size[:, None, None]
    thin = rng.random(n) < 0.2
    pos[thin, 2] = pos[thin, 0] + (pos[thin, 1] - pos[thin, 0]) * np.float32(0.999)
    return pos.reshape(-1, 3), attr, tris, mvp, vp


def check_frame(w, h, draws, ctx, octx, soup=random_soup, tile_w=32):
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
        pos, attr, tris, mvp, vp = soup(rng, n, w, h, kind)
        meshes.append(RB.Mesh(pos, tris, attr))
        mds.append(RB.mesh_draw(meshes[-1], shaders[kind], mvp, vp, texture=dtex if kind == 3 else None))
        err, _ = O.render(kind, tris, pos, attr, mvp, vp, ocol, depth=odep, flat=(9, 200, 77, 255),
                          tex=tex if kind == 3 else None, ctx=octx, stats=ost)
        assert err == 0
    b = RB.Batch([(fb, ctx, mds)], tile_w=tile_w)
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


@pytest.mark.parametrize("tw,th", [(16, 16), (32, 32), (64, 32), (32, 64), (64, 64)])
@pytest.mark.parametrize("w,h", [(64, 64), (101, 67)])
def test_hidden_small_triangles(w, h, tw, th):
    """Thousands of small triangles a tile, most of them behind others: the
    tiles pass over those (whole and partial tiles, clipped triangles and
    large ones among them), and every counter still is the oracle's."""
    dev = rf.default_device()
    dev.set_tile_height(th)
    try:
        check_frame(w, h, [(1, 4000), (3, 3000), (0, 2000)], rf.Context(clear=True, face_cull=None), (1, 0, 1, 1, 0),
                    small_soup, tw)
    finally:
        dev.set_tile_height(0)


@pytest.mark.parametrize("dt,dw", [("less", False), ("greater", True), ("equal", True), (None, True)])
def test_small_triangles_under_other_tests(dt, dw):
    """As above where nothing may be passed over, or depth never changes."""
    check_frame(64, 48, [(3, 3000), (1, 3000)], rf.Context(clear=True, face_cull=None, depth_test=dt, depth_write=dw),
                ({None: 0, "less": 1, "equal": 2, "greater": 3}[dt], 0, 1, int(dw), 0), small_soup)


@pytest.mark.parametrize("n", [61, 62, 63, 130, 300])
def test_tiles_of_many_draws(n):
    """More draws meet in one tile than its colour sources can name at a time."""
    kinds = [3, 1, 3, 0]
    check_frame(40, 40, [(kinds[i % 4], 1 + i % 3) for i in range(n)], rf.Context(clear=True, face_cull=None),
                (1, 0, 1, 1, 0))


@pytest.mark.parametrize("runs", [63, 64, 65, 1023, 1024, 1025, 4096, 4097])
def test_run_lists_of_every_length(runs):
    """One tile of a 16 x 16 frame with about 64 triangles in each of `runs`
    groups: lists are ordered in registers, by a wave, by a block and in global
    memory, and a small triangle in front decides nothing about the others."""
    w = h = 16
    rng = np.random.default_rng(runs)
    n = 64 * runs
    # every triangle meets the frame, so every group has its run in the tile
    pos = rng.uniform([-0.9, -0.9, 0.0], [0.9, 0.9, 4.0], size=(n, 1, 3)).astype(np.float32)
    pos = (pos + rng.uniform(-0.3, 0.3, size=(n, 3, 3)).astype(np.float32)).reshape(-1, 3)
    tris = np.arange(3 * n, dtype=np.uint32).reshape(n, 3)
    attr = rng.uniform(0, 1, size=(3 * n, 3)).astype(np.float32)
    mvp = M.then(M.translate3(0, 0, 2.0), M.perspective(1.2, np.float32(1.0), 0.1, 8.0))
    vp = M.viewport(0, h, w, 0)
    ocol, odep, ost = np.zeros((h, w, 4), np.uint8), np.zeros((h, w), np.float32), np.zeros(8, np.uint64)
    ocol[...] = (0, 0, 0, 255)
    err, _ = O.render(1, tris, pos, attr, mvp, vp, ocol, depth=odep, ctx=(1, 0, 1, 1, 0), stats=ost)
    assert err == 0
    fb, m = RB.DeviceFramebuf(w, h, 0, True), RB.Mesh(pos, tris, attr)
    b = RB.Batch([(fb, rf.Context(clear=True, face_cull=None), [RB.mesh_draw(m, rf.shader.Gouraud(), mvp, vp)])],
                 tile_w=16)
    for _ in range(2):
        b.run()
        s = b.wait()[0]
        gcol, gdep = fb.read()
        assert np.array_equal(gcol, ocol)
        assert np.array_equal(gdep.view(np.uint32), odep.view(np.uint32))
        assert [s.prims_o, s.frags_i, s.frags_o] == [int(ost[2]), int(ost[5]), int(ost[6])]
    b.free()
    fb.free()
    m.free()


@pytest.mark.parametrize("frames", [1, 255, 256, 257, 600])
def test_tile_counts_around_the_scan_kernels(frames):
    """64 x 64 frames of 16 tiles each, 4,096 tiles being what one block scans:
    empty frames, dense ones (whose tiles are heavy) and ordinary ones."""
    rng = np.random.default_rng(frames)
    w = h = 64
    soups = [small_soup(rng, n, w, h, 1) for n in (3, 40, 1500)]
    meshes = [RB.Mesh(p, t, a) for p, a, t, _, _ in soups]
    want = []
    for pos, attr, tris, mvp, vp in soups:
        ocol, odep, ost = np.zeros((h, w, 4), np.uint8), np.zeros((h, w), np.float32), np.zeros(8, np.uint64)
        ocol[...] = (0, 0, 0, 255)
        err, _ = O.render(1, tris, pos, attr, mvp, vp, ocol, depth=odep, ctx=(1, 0, 1, 1, 0), stats=ost)
        assert err == 0
        want.append((ocol, odep, int(ost[5]), int(ost[6])))
    dev = rf.default_device()
    dev.set_tile_height(16)
    try:
        which = [None if i % 7 == 3 else 2 if i % 11 == 0 else i % 2 for i in range(frames)]
        fbs = [RB.DeviceFramebuf(w, h, 0, True) for _ in range(frames)]
        ctx = rf.Context(clear=True, face_cull=None)
        b = RB.Batch([(fbs[i], ctx, [] if k is None else [RB.mesh_draw(meshes[k], rf.shader.Gouraud(), *soups[k][3:])])
                      for i, k in enumerate(which)], tile_w=16)
        b.run()
        for fb, k, s in zip(fbs, which, b.wait()):
            gcol, gdep = fb.read()
            if k is None:
                assert (gcol == (0, 0, 0, 255)).all() and (gdep == 0).all() and s.frags_i == 0
            else:
                assert np.array_equal(gcol, want[k][0])
                assert np.array_equal(gdep.view(np.uint32), want[k][1].view(np.uint32))
                assert (s.frags_i, s.frags_o) == want[k][2:]
        b.free()
    finally:
        dev.set_tile_height(0)
        for x in fbs + meshes:
            x.free()


@pytest.mark.parametrize("w,h", [(1, 1), (3, 700), (255, 257), (512, 512), (513, 511), (1031, 997)])
@pytest.mark.parametrize("fmt", [rf.PIX_RGBA8, rf.PIX_RGB8, rf.PIX_RGB565])
@pytest.mark.parametrize("pad,clear,depth", [(0, True, True), (0, False, True), (7, False, True), (7, True, False)])
def test_plain_calls_into_targets_of_every_size(w, h, fmt, pad, clear, depth):
    """rf_render's staged copies: packed targets and views, cleared and drawn
    over, smaller than one part of the read-back and of several; the parent's
    bytes around a view stay as they are."""
    rng = np.random.default_rng([w, h, fmt, pad])
    shape = (h + pad, w + pad) + ({0: (4,), 1: (3,)}.get(fmt, ()))
    col = rng.integers(0, 250, size=shape).astype(np.uint16 if fmt == rf.PIX_RGB565 else np.uint8)
    dep = rng.uniform(0.0, 0.2, size=(h + pad, w + pad)).astype(np.float32)
    gcol, gdep = col.copy(), dep.copy()
    cut = (slice(pad // 2, pad // 2 + h), slice(pad // 2, pad // 2 + w))
    ocol, odep = np.ascontiguousarray(col[cut]), np.ascontiguousarray(dep[cut])
    if clear:
        ocol[...] = 0 if fmt == rf.PIX_RGB565 else np.array([0, 0, 0, 255][:ocol.shape[2]], np.uint8)
        odep[...] = 0.0
    pos, attr, tris, mvp, vp = random_soup(rng, 40, w, h, 1)
    ost = np.zeros(8, np.uint64)
    err, _ = O.render(1, tris, pos, attr, mvp, vp, ocol, depth=odep if depth else None, fmt=fmt, ctx=(1, 0, 1, 1, 0),
                      stats=ost)
    assert err == 0
    ctx = rf.Context(clear=clear, face_cull=None)
    target = rf.Framebuf(gcol[cut], gdep[cut], fmt) if depth else rf.Colorbuf(gcol[cut], fmt)
    rf.render(tris, (pos, attr), rf.shader.Gouraud(), mvp, vp, target, ctx)
    assert np.array_equal(gcol[cut], ocol)
    assert [ctx.stats.prims_o, ctx.stats.frags_i, ctx.stats.frags_o] == [int(ost[2]), int(ost[5]), int(ost[6])]
    if depth:
        assert np.array_equal(gdep[cut].view(np.uint32), odep.view(np.uint32))
    gcol[cut], gdep[cut] = col[cut], dep[cut]
    assert np.array_equal(gcol, col) and np.array_equal(gdep, dep)


@pytest.mark.parametrize("counts", [(1, 2), (63, 1, 64), (65, 130), (300, 5)])
def test_culled_draws_of_several_frames_in_a_wave(counts):
    """Frames of `counts` draws, half of them hidden whole by their bounding
    boxes: the hidden calls, primitives and vertices are each frame's own."""
    rng = np.random.default_rng(counts)
    pos = rng.uniform(-0.2, 0.2, size=(30, 3)).astype(np.float32)
    tris = np.arange(30, dtype=np.uint32).reshape(10, 3)
    m = RB.Mesh(pos, tris)
    vp, proj = M.viewport(0, 48, 64, 0), M.perspective(1.2, np.float32(64 / 48), 0.1, 8.0)
    frames, want = [], []
    for n in counts:
        draws, ocol, ost = [], np.zeros((48, 64, 4), np.uint8), np.zeros(8, np.uint64)
        ocol[...] = (0, 0, 0, 255)
        hidden = 0
        for k in range(n):
            x = 40.0 if rng.random() < 0.5 else float(rng.uniform(-0.5, 0.5))
            mvp = M.then(M.translate3(x, 0.0, 2.0), proj)
            draws.append(RB.mesh_draw(m, rf.shader.Flat((k % 256, 9, 200, 255)), mvp, vp, cull=True))
            if O.bbox_visibility(O.bbox_of(pos), mvp) == O.HIDDEN:
                hidden += 1
                continue
            err, _ = O.render(0, tris, pos, None, mvp, vp, ocol, flat=(k % 256, 9, 200, 255), ctx=(0, 0, 1, 1, 0),
                              stats=ost)
            assert err == 0
        frames.append((RB.DeviceFramebuf(64, 48, 0, False), rf.Context(clear=True, face_cull=None), draws))
        want.append((ocol, [n, n - hidden] + [int(x) for x in ost[:7]]))
    b = RB.Batch(frames, tile_w=32)
    for _ in range(2):
        b.run()
        for s, (fb, _, _), (ocol, counts_) in zip(b.wait(), frames, want):
            assert np.array_equal(fb.read()[0], ocol)
            assert [s.objs_i, s.objs_o, s.calls, s.prims_i, s.prims_o, s.verts_i, s.verts_o, s.frags_i,
                    s.frags_o] == counts_
    b.free()
    m.free()
    for fb, _, _ in frames:
        fb.free()


@pytest.mark.parametrize("n", [1, 31, 32, 33, 63, 64, 65, 130])
@pytest.mark.parametrize("draws", [1, 3])
def test_groups_of_many_tiles(n, draws):
    """One group of 64 triangles (and, with more draws, several and the end of
    one) meets n tiles of a row: what k_setup keeps of its runs, what k_bin walks
    again, and lists of exactly 64."""
    check_frame(16 * n, 16, [(1, 64), (3, 64), (0, 40)][:draws], rf.Context(clear=True, face_cull=None), (1, 0, 1, 1, 0),
                random_soup, 16)


@pytest.mark.parametrize("n,per", [(2, 3), (64, 17), (3000, 3), (9000, 21)])
def test_many_depth_sorted_draws(n, per):
    """So many sorted render() calls that draw, depth and index still fit one
    sort key, or (9,000 calls of 21 triangles) do not: each sorts its own."""
    rng = np.random.default_rng(n)
    w = h = 24
    kinds = [small_soup(rng, per, w, h, 1) for _ in range(min(n, 50))]
    meshes = [RB.Mesh(p, t, a) for p, a, t, _, _ in kinds]
    fb = RB.DeviceFramebuf(w, h, 0, False)
    ocol, ost = np.zeros((h, w, 4), np.uint8), np.zeros(8, np.uint64)
    ocol[...] = (0, 0, 0, 255)
    draws = []
    for k in range(n):
        pos, attr, tris, mvp, vp = kinds[k % len(kinds)]
        draws.append(RB.mesh_draw(meshes[k % len(kinds)], rf.shader.Gouraud(), mvp, vp))
        err, _ = O.render(1, tris, pos, attr, mvp, vp, ocol, ctx=(0, 0, 1, 1, 2), stats=ost)
        assert err == 0
    ctx = rf.Context(clear=True, face_cull=None, depth_test=None, depth_sort="back_to_front")
    b = RB.Batch([(fb, ctx, draws)], tile_w=16)
    for _ in range(2):
        b.run()
        s = b.wait()[0]
        assert np.array_equal(fb.read()[0], ocol)
        assert [s.calls, s.prims_i, s.prims_o, s.verts_i, s.verts_o, s.frags_i, s.frags_o] == [int(x) for x in ost[:7]]
    b.free()
    fb.free()
    for m in meshes:
        m.free()


def coherent_soup(rng, n, w, h, kind):
    """Small triangles whose 64 of a group lie together, the groups at depths of
    their own; every fifth group has one triangle through the near plane or one
    as large as the frame among them."""
    pos, attr, tris, _, vp = random_soup(rng, n, w, h, kind)
    g = -(-n // 64)
    mid = np.repeat(rng.uniform([-0.8, -0.8, 0.0], [0.8, 0.8, 5.0], size=(g, 3)), 64, axis=0)[:n, None]
    pos = mid + rng.uniform(-1, 1, size=(n, 3, 3)) * [0.15, 0.15, 0.02]
    odd = np.arange(7, n, 320)
    pos[odd[0::2], 2, 2] = -3.0
    pos[odd[1::2]] = mid[odd[1::2]] + rng.uniform(-1, 1, size=(len(odd[1::2]), 3, 3)) * [3.0, 3.0, 0.5]
    mvp = M.then(M.translate3(0, 0, 2.0), M.perspective(1.2, np.float32(w / h), 0.1, 8.0))
    return pos.reshape(-1, 3).astype(np.float32), attr, tris, mvp, vp


@pytest.mark.parametrize("w,h,tw", [(16, 16, 16), (37, 29, 32)])
@pytest.mark.parametrize("groups", [64, 65, 128, 129, 300])
def test_whole_groups_behind(groups, w, h, tw):
    """Run lists around multiples of 64, most of whose groups are hidden as a whole."""
    check_frame(w, h, [(1, 64 * groups - 5), (3, 130)], rf.Context(clear=True, face_cull=None), (1, 0, 1, 1, 0),
                coherent_soup, tw)


@pytest.mark.parametrize("w,h", [(128, 128), (144, 128), (1024, 16), (1040, 16), (16, 1040)])
@pytest.mark.parametrize("sizes", [(64,), (200,), (33, 31, 70)])
def test_groups_over_a_block_of_tiles(w, h, sizes):
    """Groups whose triangles span 64 tiles (of 16 x 16) and more, of one draw
    and of several."""
    dev = rf.default_device()
    dev.set_tile_height(16)
    try:
        check_frame(w, h, [(1, n) for n in sizes], rf.Context(clear=True, face_cull=None), (1, 0, 1, 1, 0), tile_w=16)
    finally:
        dev.set_tile_height(0)
