"""rf_render into targets beyond the sizes at which its copies change their way:
the caller's bytes are the oracle's, the bytes around a view stay as they are, and
no such call takes the runtime's row-by-row copies (ten times as long)."""
import time

import numpy as np
import pytest

import oracle_lib as O
import retrofire_amd as rf
from retrofire_amd import mat as M
from test_gpu_parity import random_soup

pytestmark = pytest.mark.gpu


def triangles(rng, w, h, n=30):
    """Triangles of about 200 pixels, anywhere on a w x h target, at depths of
    their own."""
    px = rng.uniform([0, 0], [w, h], size=(n, 1, 2)) + rng.uniform(-100, 100, size=(n, 3, 2))
    px = np.clip(px, 1, [w - 1, h - 1])
    cw = rng.uniform(1.0, 5.0, size=(n, 3, 1))  # clip w; depth is 1 / w
    xy = np.stack([px[..., 0] / (w / 2) - 1, 1 - px[..., 1] / (h / 2)], -1)
    pos = np.concatenate([xy * cw, cw], -1).astype(np.float32).reshape(-1, 3)
    mvp = np.array([[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 0, 0], [0, 0, 1, 0]], np.float32)
    return np.arange(3 * n).reshape(n, 3), pos, rng.uniform(0, 1, size=(3 * n, 3)).astype(np.float32), mvp, \
        M.viewport(0, h, w, 0)


def parent(w, h, item, fill):
    """A w x h view, and what lies around it, if `fill` columns do."""
    a = np.full((h + 2, w + fill) if item == 1 else (h + 2, w + fill, item), 0.1 if item == 1 else 77,
                np.float32 if item == 1 else np.uint8)
    return a, a[1:h + 1, fill // 2:fill // 2 + w]


def seconds(draw, col, dep, clear):
    """The quickest of three calls."""
    tris, pos, attr, mvp, vp = draw
    best = 1e9
    for _ in range(3):
        t = time.perf_counter()
        rf.render(tris, (pos, attr), rf.shader.Gouraud(), mvp, vp, rf.Framebuf(col, dep),
                  rf.Context(clear=clear, face_cull=None))
        best = min(best, time.perf_counter() - t)
    return best


# (width, height, columns around the colour view, around the depth view, cleared)
CASES = {"kept, 131 MiB, rows of no 16 bytes": (4099, 4200, 0, 0, False),
         "kept view, 131 MiB": (4099, 4200, 5, 3, False),
         "view of 281 MiB": (16001, 2300, 6, 2, True),
         "colour view of 281 MiB, kept": (16001, 2300, 6, 0, False),
         "depth view of 281 MiB, kept": (16001, 2300, 0, 2, False)}


@pytest.mark.parametrize("case", CASES)
def test_large_targets(case):
    w, h, cfill, dfill, clear = CASES[case]
    draw = triangles(np.random.default_rng(w), w, h)
    tris, pos, attr, mvp, vp = draw
    cpar, col = parent(w, h, 4, cfill)
    dpar, dep = parent(w, h, 1, dfill)
    ctx = rf.Context(clear=clear, face_cull=None)
    rf.render(tris, (pos, attr), rf.shader.Gouraud(), mvp, vp, rf.Framebuf(col, dep), ctx)
    ocol, odep = np.full((h, w, 4), 77, np.uint8), np.full((h, w), 0.1, np.float32)
    if clear:
        ocol[...] = (0, 0, 0, 255)
        odep[...] = 0.0
    err, ost = O.render(1, tris, pos, attr, mvp, vp, ocol, depth=odep, ctx=(1, 0, 1, 1, 0))
    assert err == 0
    assert np.array_equal(col, ocol) and np.array_equal(dep, odep)
    assert [ctx.stats.frags_i, ctx.stats.frags_o] == [int(ost[5]), int(ost[6])] and ctx.stats.frags_o > 10000
    del ocol, odep
    col[...], dep[...] = 77, 0.1
    assert (cpar == 77).all() and (dpar == np.float32(0.1)).all()
    # the same call with fewer rows, on the near side of the line
    h2 = h * 9 // 10
    near = seconds(triangles(np.random.default_rng(w), w, h2), parent(w, h2, 4, cfill)[1], parent(w, h2, 1, dfill)[1],
                   clear)
    took = seconds(draw, col, dep, clear)
    print(f"{case}: {1e3 * took:.1f} ms, with {h2} of {h} rows {1e3 * near:.1f} ms")
    assert took < 3.0 * near


@pytest.mark.parametrize("pad", [0, 6])
def test_kept_target_of_a_call_that_is_run_again(pad):
    """A device's first call of 47 groups of triangles that each cover most of 352
    tiles: far more runs than it has room for (47 * 4 + 352 + 1,024), and more clip
    fans than 1,024, so the call is run again, over the caller's own target."""
    w, h = 700, 501
    rng = np.random.default_rng(pad)
    pos, attr, tris, mvp, vp = random_soup(rng, 3000, w, h, 1)
    cpar, col = parent(w, h, 4, pad)
    dpar, dep = parent(w, h, 1, pad)
    col[...] = rng.integers(0, 256, size=col.shape)
    dep[...] = rng.uniform(0.0, 0.6, size=dep.shape)
    ocol, odep = col.copy(), dep.copy()
    err, ost = O.render(1, tris, pos, attr, mvp, vp, ocol, depth=odep, ctx=(1, 0, 1, 1, 0))
    assert err == 0
    ctx = rf.Context(clear=False, face_cull=None)
    dev = rf.Device()
    try:
        rf.render(tris, (pos, attr), rf.shader.Gouraud(), mvp, vp, rf.Framebuf(col, dep), ctx, device=dev)
    finally:
        dev.close()
    assert np.array_equal(col, ocol)
    assert np.array_equal(dep.view(np.uint32), odep.view(np.uint32))
    assert [ctx.stats.frags_i, ctx.stats.frags_o] == [int(ost[5]), int(ost[6])]
    col[...], dep[...] = 77, 0.1
    assert (cpar == 77).all() and (dpar == np.float32(0.1)).all()
