"""Dense frames drawn over depth that the caller's target holds, infinities and
NaN among it: what the tiles pass over as hidden must still count, and must
still report a span outside the target, as the oracle does."""
import numpy as np
import pytest

import oracle_lib as O
import retrofire_amd as rf
from retrofire_amd import mat as M
from test_gpu_sizes import coherent_soup

pytestmark = pytest.mark.gpu

RF_E_BOUNDS = -2


def kept_depth(rng, w, h, fill):
    """Depth as a caller may leave it. `random` lies where the soup's does."""
    dep = rng.uniform(0.0, 0.4, size=(h, w)).astype(np.float32)
    if fill == "halves":  # one half of each kind, side by side in a tile
        dep[:, : w // 2] = np.inf
        dep[h // 2:, w // 2:] = np.nan
    elif fill == "spots":
        dep[rng.random((h, w)) < 0.3] = np.inf
        dep[rng.random((h, w)) < 0.3] = np.nan
    elif fill != "random":
        dep[...] = {"inf": np.inf, "nan": np.nan, "-inf": -np.inf}[fill]
    return dep


@pytest.mark.parametrize("groups", [65, 200])
@pytest.mark.parametrize("w,h", [(16, 16), (37, 29), (64, 40)])
@pytest.mark.parametrize("fill", ["inf", "nan", "-inf", "halves", "spots", "random"])
def test_dense_frames_over_kept_depth(fill, w, h, groups):
    """Clipped and frame-high triangles, whose depth bound is not known, among
    small ones: no pixel passes where the depth is +inf or NaN, but fragments
    count."""
    rng = np.random.default_rng([w, h, groups])
    pos, attr, tris, mvp, vp = coherent_soup(rng, 64 * groups * (2 if w > 32 else 1), w, h, 1)
    ocol = rng.integers(0, 256, size=(h, w, 4), dtype=np.uint8)
    odep = kept_depth(rng, w, h, fill)
    gcol, gdep = ocol.copy(), odep.copy()
    err, ost = O.render(1, tris, pos, attr, mvp, vp, ocol, depth=odep, ctx=(1, 0, 1, 1, 0))
    assert err == 0
    ctx = rf.Context(clear=False, face_cull=None)
    rf.render(tris, (pos, attr), rf.shader.Gouraud(), mvp, vp, rf.Framebuf(gcol, gdep), ctx)
    s = ctx.stats
    assert [s.prims_o, s.verts_o, s.frags_i, s.frags_o] == [int(ost[k]) for k in (2, 4, 5, 6)]
    assert np.array_equal(gcol, ocol)
    assert np.array_equal(gdep.view(np.uint32), odep.view(np.uint32))


def test_depth_cleared_to_infinity():
    """depth_clear = 0 clears to 1 / 0."""
    w, h = 37, 29
    pos, attr, tris, mvp, vp = coherent_soup(np.random.default_rng(8), 64 * 130, w, h, 1)
    ocol, odep = np.zeros((h, w, 4), np.uint8), np.full((h, w), np.inf, np.float32)
    ocol[...] = (0, 0, 0, 255)
    err, ost = O.render(1, tris, pos, attr, mvp, vp, ocol, depth=odep, ctx=(1, 0, 1, 1, 0))
    assert err == 0
    gcol, gdep = np.empty_like(ocol), np.empty_like(odep)
    ctx = rf.Context(clear=True, face_cull=None, depth_clear=0.0)
    rf.render(tris, (pos, attr), rf.shader.Gouraud(), mvp, vp, rf.Framebuf(gcol, gdep), ctx)
    assert [ctx.stats.frags_i, ctx.stats.frags_o] == [int(ost[5]), int(ost[6])]
    assert np.array_equal(gcol, ocol) and np.array_equal(gdep, odep)


def crowded(rng, w, h, last):
    """10,240 triangles a few pixels wide inside a w x h target, at depths of
    their own, the last one at the screen positions `last`. The viewport is that
    of a larger target, so that nothing is clipped at this one's edges."""
    n, big = 64 * 160, 64
    px = rng.uniform([1.5, 1.5], [w - 1.5, h - 1.5], size=(n, 1, 2)) + rng.uniform(-1.0, 1.0, size=(n, 3, 2))
    px[n - 1] = last
    cw = rng.uniform(1.0, 5.0, size=(n, 1, 1)) * rng.uniform(0.99, 1.01, size=(n, 3, 1))  # clip w; depth is 1 / w
    xy = np.stack([px[..., 0] / big - 1, 1 - px[..., 1] / big], -1)
    pos = np.concatenate([xy * cw, cw], -1).astype(np.float32).reshape(-1, 3)
    tris = np.arange(3 * n, dtype=np.uint32).reshape(n, 3)
    attr = rng.uniform(0, 1, size=(3 * n, 3)).astype(np.float32)
    mvp = np.array([[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 0, 0], [0, 0, 1, 0]], np.float32)
    return pos, attr, tris, mvp, M.viewport(0, 2 * big, 2 * big, 0)


W, H = 32, 48
LAST = {"inside": [(8, 20), (16, 20), (10, 26)],
        "tall": [(8, 2), (W + 9, 30), (10, 46)],
        "small right": [(W - 4, 20), (W + 5, 23), (W - 3, 26)],
        "small bottom": [(8, H - 4), (16, H - 3), (10, H + 4)],
        "sliver right": [(W - 1, 20.2), (W + 3, 20.8), (W + 0.4, 21.2)]}


@pytest.mark.parametrize("where", LAST)
@pytest.mark.parametrize("fill", ["random", "inf"])
def test_spans_outside_the_target_among_many_small_triangles(where, fill):
    """One triangle of a dense frame reaches past the target's edge, visible or
    behind everything: an error, as in the oracle."""
    rng = np.random.default_rng(5)
    pos, attr, tris, mvp, vp = crowded(rng, W, H, LAST[where])
    ocol, odep = np.zeros((H, W, 4), np.uint8), kept_depth(rng, W, H, fill)
    gcol, gdep = ocol.copy(), odep.copy()
    err, ost = O.render(1, tris, pos, attr, mvp, vp, ocol, depth=odep, ctx=(1, 0, 1, 1, 0))
    assert (err == 0) == (where == "inside")
    ctx = rf.Context(clear=False, face_cull=None)

    def call():
        rf.render(tris, (pos, attr), rf.shader.Gouraud(), mvp, vp, rf.Framebuf(gcol, gdep), ctx)

    if where == "inside":
        call()
        assert [ctx.stats.frags_i, ctx.stats.frags_o] == [int(ost[5]), int(ost[6])]
        assert np.array_equal(gcol, ocol) and np.array_equal(gdep, odep)
    else:
        with pytest.raises(rf.RenderError) as e:
            call()
        assert e.value.status == RF_E_BOUNDS
