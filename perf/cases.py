"""The render path's measured workloads, through the package's public calls.

A case is one of three ways a program draws:

  plain   `render()` with host buffers: upload, draw, read back, one call a frame;
  batch   resident meshes and targets, frames planned once and replayed (`Batch.run`);
  serve   a burst of requests submitted to a `Server` and polled until all are back.

Scenes (seeded, the shapes of retrofire_amd.scenes and of the benchmark):

  quad     a textured quad (the golden image test's scene)
  sphere   a Gouraud UV-sphere, 64 x 32
  crates   n textured unit cubes on a 100 x 100 field, first-person camera inside it
  objects  the same crates as n draws with whole-object culling
  spheres  n icospheres of 320 triangles in the unit ball, orbiting camera
  mix      crates and spheres in one frame, 10-100 % of each, resolutions uneven
  wire     n crates filled flat with their edges drawn over them (debug view)
  sorted   n icospheres back to front into a colour-only target (painter's order)
"""
from __future__ import annotations

import functools

import numpy as np
import torch

import retrofire_amd as rf
from retrofire_amd import batch as RB
from retrofire_amd import mat as M
from retrofire_amd import scenes as S

F = np.float32
NEAR = 0.1
SAMPLERS = ("repeat", "clamp", "once")
ITEM = {0: ("<i4", 4), 1: ("|u1", 3), 2: ("<i4", 4), 3: ("<i4", 4), 4: ("<i4", 4), 5: ("<i4", 4), 6: ("<i2", 2),
        7: ("<i2", 2)}


# ------------------------------------------------------------------ cases

def case(path, scene, n, w, h, frames=1, fmt=0, depth=True, sampler="repeat", uneven=False, pitched=False, **kw):
    return dict(path=path, scene=scene, n=n, w=w, h=h, frames=frames, fmt=fmt, depth=depth, sampler=sampler,
                uneven=uneven, pitched=pitched, **kw)


def listed():
    return [
        # the smallest call there is: two triangles, where a call's fixed cost is everything
        case("plain", "quad", 1, 256, 256, sampler="clamp", name="plain_quad_256"),
        # a program that moves one ordinary model to the GPU call by call
        case("plain", "sphere", 1, 640, 480, name="plain_sphere_640"),
        # a full-HD scene call by call: the copies of a frame count beside its drawing
        case("plain", "crates", 1000, 1920, 1080, name="plain_crates_1080"),
        # drawing into part of a pitched surface of odd size (a window system's buffer), over what is there
        case("plain", "crates", 200, 1003, 667, fmt=3, sampler="clamp", pitched=True, name="plain_pitched_1003"),
        # the smallest resident frame: latency of a launch (thumbnails, previews)
        case("batch", "crates", 125, 256, 256, name="batch_crates_256"),
        # the headline: full-HD textured frames in one launch
        case("batch", "crates", 1000, 1920, 1080, frames=32, name="batch_crates_1080"),
        # many small triangles: 3.2M a frame
        case("batch", "spheres", 10000, 1920, 1080, frames=8, name="batch_spheres_1080"),
        # uneven frames of both scenes at once (a render farm's or a data generator's launch); the largest
        case("batch", "mix", 10000, 0, 0, frames=32, uneven=True, name="batch_mix_uneven"),
        # a scene of separate objects, each its own draw with its own matrix, culled whole
        case("batch", "objects", 1000, 1920, 1080, frames=4, name="batch_objects_1080"),
        # painter's order without a depth buffer: the depth sort
        case("batch", "sorted", 500, 1280, 720, frames=4, depth=False, name="batch_sorted_720"),
        # debug view in 16-bit colour at an odd size: lines, flat fills, partial tiles
        case("batch", "wire", 500, 853, 479, frames=8, fmt=7, name="batch_wire_853"),
        # a burst of requests of mixed meshes and sizes to the serving loop
        case("serve", "mix", 500, 0, 0, frames=24, uneven=True, name="serve_burst_24"),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    path = rng.choice(["plain", "batch", "batch", "batch", "serve"])
    if path == "serve":
        return case("serve", "mix", _log(rng, 40, 700), 0, 0, frames=rng.randint(3, 24), uneven=True)
    w, h = _log(rng, 100, 2048), _log(rng, 80, 2048)
    fmt = rng.choice([0, 0, 0, 1, 2, 3, 4, 5, 6, 7])
    sampler = rng.choice(SAMPLERS)
    if path == "plain":
        scene = rng.choice(["quad", "sphere", "crates", "spheres"])
        n = {"quad": 1, "sphere": 1, "crates": _log(rng, 20, 1500), "spheres": _log(rng, 10, 1000)}[scene]
        return case("plain", scene, n, w, h, fmt=fmt, depth=rng.random() < 0.8, sampler=sampler,
                    pitched=rng.random() < 0.3)
    scene = rng.choice(["crates", "crates", "spheres", "spheres", "mix", "objects", "sorted", "wire"])
    frames = _log(rng, 1, 32)
    n = {"crates": (20, 2000), "spheres": (50, 10000), "mix": (100, 5000), "objects": (30, 1000), "sorted": (20, 700),
         "wire": (20, 1000)}[scene]
    n = _log(rng, *n)
    if scene in ("objects", "sorted"):
        frames = min(frames, 8)
    if scene == "spheres":
        frames = max(1, min(frames, 80000 // n))
    uneven = scene == "mix"
    return case("batch", scene, n, 0 if uneven else w, 0 if uneven else h, frames=frames,
                fmt=0 if uneven else fmt, depth=scene != "sorted" and (uneven or rng.random() < 0.85),
                sampler=sampler, uneven=uneven)


# ------------------------------------------------------------------ inputs

def texture(rng, n=256):
    y, x = np.mgrid[0:n, 0:n]
    base = np.where(((x // 32) ^ (y // 32)) & 1, 0xC0, 0x30).astype(np.uint8)
    tex = base[..., None] ^ rng.integers(0, 64, (n, n, 4)).astype(np.uint8)
    tex[..., 3] = 255
    return np.ascontiguousarray(tex)


def inset(uv, sampler):
    # SamplerOnce takes coordinates inside the texture only (an atlas cell's)
    return (F(0.05) + uv * F(0.9)).astype(F) if sampler == "once" else uv


def crate_models(rng, n):
    a = rng.uniform(0.0, 2.0 * np.pi, n)
    m = np.zeros((n, 4, 4), F)
    m[:, 0, 0], m[:, 0, 2], m[:, 2, 0], m[:, 2, 2] = np.cos(a), np.sin(a), -np.sin(a), np.cos(a)
    m[:, 1, 1] = m[:, 3, 3] = 1.0
    m[:, 0, 3], m[:, 2, 3] = rng.uniform(-50.0, 50.0, n), rng.uniform(-50.0, 50.0, n)
    return m


def crates(rng, n):
    cpos, cuv, ctri = S.cube(1.0)
    m = crate_models(rng, n)
    pos = (np.einsum("nij,vj->nvi", m[:, :3, :3], cpos) + m[:, None, :3, 3]).astype(F).reshape(-1, 3)
    tris = (ctri[None] + 24 * np.arange(n, dtype=np.uint32)[:, None, None]).reshape(-1, 3).astype(np.uint32)
    return pos, np.tile(cuv, (n, 1)), tris


@functools.lru_cache(maxsize=None)
def _ico():
    return S.icosphere(0.05, 2)


@functools.lru_cache(maxsize=None)
def _lathe():
    return S.lathe_sphere(64, 32, 1.0)


def spheres(rng, n):
    ipos, itri = _ico()
    c = rng.uniform(-1.0, 1.0, (4 * n + 64, 3))
    c = c[(c * c).sum(1) <= 1.0][:n]
    n, nv = len(c), len(ipos)
    pos = (ipos[None] + c[:, None].astype(F)).astype(F).reshape(-1, 3)
    attr = np.repeat(rng.uniform(0.0, 1.0, (n, 3)).astype(F), nv, axis=0)
    tris = (itri[None] + nv * np.arange(n, dtype=np.uint32)[:, None, None]).reshape(-1, 3).astype(np.uint32)
    return pos, attr, tris


def edges_of(tris):
    e = np.sort(np.concatenate([tris[:, [0, 1]], tris[:, [1, 2]], tris[:, [2, 0]]]), axis=1)
    return np.unique(e, axis=0).astype(np.uint32)


def sizes(c):
    if not c["uneven"]:
        return [(c["w"], c["h"])] * c["frames"]
    # each resolution about equally often, in the same mixed order for every seed
    k = np.random.default_rng(c["frames"]).permutation(np.arange(c["frames"]) % len(S.RESOLUTIONS))
    return [S.RESOLUTIONS[i] for i in k]


def model(c, seed):
    """The case's inputs on the host, from its numbers and the seed alone: meshes [(kind, pos, attr, prims)],
    the texture, and the frames: (w, h, viewport, [(mesh, mvp, first, count)])."""
    rng = np.random.default_rng([seed, c["n"], c["frames"], c["w"], c["h"]])
    sc = c["scene"]
    tex = texture(rng)
    frames = []
    if sc == "quad":
        pos = np.array([[-1, -1, 0], [-1, 1, 0], [1, -1, 0], [1, 1, 0]], F) + rng.uniform(-0.2, 0.2, (4, 3)).astype(F)
        uv = inset(np.array([[0, 0], [0, 1], [1, 0], [1, 1]], F), c["sampler"])
        meshes = [("tex", pos, uv, np.array([[0, 1, 2], [3, 2, 1]], np.uint32))]
        for w, h in sizes(c):
            mvp = M.then(M.translate3(0.0, 0.0, 2.5), M.perspective(F(1.0), F(w) / F(h), NEAR, 100.0))
            frames.append((w, h, M.viewport(0, h, w, 0), [(0, mvp, 0, 2)]))
    elif sc == "sphere":
        pos, tris = _lathe()
        meshes = [("rgb", pos, rng.uniform(0.0, 1.0, (len(pos), 3)).astype(F), tris)]
        for w, h in sizes(c):
            proj = M.perspective(F(1.7320508), F(w) / F(h), NEAR, 100.0)
            view = M.then(M.rotate_y(rng.random()), M.translate3(0.0, 0.0, 3.0))
            frames.append((w, h, M.viewport(0, 0, w, h), [(0, M.then(view, proj), 0, len(tris))]))
    elif sc in ("crates", "wire"):
        pos, uv, tris = crates(rng, c["n"])
        if sc == "crates":
            meshes = [("tex", pos, inset(uv, c["sampler"]), tris)]
        else:
            meshes = [("flat", pos, None, tris), ("line", pos, None, edges_of(tris))]
        for w, h in sizes(c):
            mvp = S.crates_mvp(w, h, rng.random())
            frames.append((w, h, M.viewport(0, h, w, 0), [(i, mvp, 0, len(m[3])) for i, m in enumerate(meshes)]))
    elif sc == "objects":
        cpos, cuv, ctri = S.cube(1.0)
        meshes = [("tex", cpos, inset(cuv, c["sampler"]), ctri)]
        models = crate_models(rng, c["n"])
        for w, h in sizes(c):
            mvps = np.matmul(S.crates_mvp(w, h, rng.random()), models).astype(F)
            frames.append((w, h, M.viewport(0, h, w, 0), [(0, m, 0, 12) for m in mvps]))
    elif sc in ("spheres", "sorted"):
        meshes = [("rgb", *spheres(rng, c["n"]))]
        for w, h in sizes(c):
            frames.append((w, h, M.viewport(0, h, w, 0),
                           [(0, S.spheres_mvp(w, h, rng.random()), 0, len(meshes[0][3]))]))
    else:  # mix: n spheres and a tenth as many crates
        nc = max(10, c["n"] // 10 if c["path"] == "batch" else c["n"])
        cp, cu, ct = crates(rng, nc)
        meshes = [("tex", cp, inset(cu, c["sampler"]), ct), ("rgb", *spheres(rng, c["n"]))]
        part = rng.permutation((np.arange(c["frames"]) + rng.random()) / c["frames"])  # 10-100 %, spread evenly
        for i, (w, h) in enumerate(sizes(c)):
            k = 0.1 + 0.9 * part[i]
            both = [(0, S.crates_mvp(w, h, rng.random()), 0, 12 * max(1, int(k * nc))),
                    (1, S.spheres_mvp(w, h, rng.random()), 0, 320 * max(1, int(k * len(meshes[1][3]) // 320)))]
            if c["path"] == "serve":
                both = both[i % 2:i % 2 + 1]  # a request names one mesh
            frames.append((w, h, M.viewport(0, h, w, 0), both))
    return meshes, tex, frames


def shader(kind, tex, sampler):
    if kind == "tex":
        return {"repeat": rf.shader.TexRepeatPot, "clamp": rf.shader.TexClamp, "once": rf.shader.TexOnce}[sampler](tex)
    if kind == "rgb":
        return rf.shader.Gouraud()
    return rf.shader.Flat((255, 255, 255, 255) if kind == "line" else (60, 90, 160, 255))


def host_target(c, rng, w, h):
    """Colour and depth arrays, or views into larger ones; what a frame before has left in them."""
    pad = 29 if c["pitched"] else 0
    if c["fmt"] < 2:
        col = rng.integers(0, 256, (h + pad, w + pad, 4 if c["fmt"] == 0 else 3), dtype=np.uint8)
    else:
        t = np.uint32 if c["fmt"] < 6 else np.uint16
        col = rng.integers(0, np.iinfo(t).max, (h + pad, w + pad), dtype=t)
    dep = np.zeros((h + pad, w + pad), F) if c["depth"] else None
    a, b = pad // 2, pad // 2
    col = col[a:a + h, b:b + w]
    dep = dep[a:a + h, b:b + w] if dep is not None else None
    return rf.Framebuf(col, dep, c["fmt"]) if dep is not None else rf.Colorbuf(col, c["fmt"])


# ------------------------------------------------------------------ state

class Resident:
    """A resident target with its memory as torch tensors."""

    def __init__(self, w, h, fmt, depth):
        self.fb = RB.DeviceFramebuf(w, h, fmt, depth)

    def tensors(self):
        t = rf._ffi.RfTarget()
        rf.check(rf._ffi.lib().rf_framebuf_target(self.fb.h, rf._ffi.C.byref(t)))
        w, h = t.width, t.height
        kind, size = ITEM[self.fb.fmt]
        shape = (h, w, 3) if self.fb.fmt == 1 else (h, w)
        out = [torch.as_tensor(_Memory(self, t.color, kind, shape), device="cuda")]
        if self.fb.with_depth:
            ptr = rf._ffi.C.cast(t.depth, rf._ffi.C.c_void_p).value
            out.append(torch.as_tensor(_Memory(self, ptr, "<f4", (h, w)), device="cuda"))
        return out

    def __del__(self):
        self.fb.free()


class _Memory:
    def __init__(self, owner, ptr, kind, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, typestr=kind, data=(ptr, False), version=2)


class State:
    def __init__(self):
        self.batch = self.server = None
        self.held = []  # meshes and textures

    def __del__(self):
        if self.server is not None:
            self.server.close()
        if self.batch is not None:
            self.batch.free()
        for x in self.held:
            x.free()


def context(c):
    # edges and colour-only frames as the debug view and the painter's order use them
    if c["scene"] == "sorted":
        return rf.Context(clear=True, depth_sort="back_to_front", depth_test=None)
    return rf.Context(clear=not c["pitched"], face_cull=None if c["scene"] == "quad" else "back")


def prepare(case, seed):
    meshes, tex, frames = model(case, seed)
    st = State()
    st.case = case
    if case["path"] == "plain":
        w, h, vp, draws = frames[0]
        kind, pos, attr, prims = meshes[0]
        st.target = host_target(case, np.random.default_rng(seed), w, h)
        st.first = (st.target.color.copy(), None if st.target.depth is None else st.target.depth.copy())
        st.args = (prims, pos if attr is None else (pos, attr), shader(kind, tex, case["sampler"]), draws[0][1], vp)
        return st
    shd = [shader(m[0], tex, case["sampler"]) for m in meshes]
    res = [RB.Mesh(m[1], m[3], m[2]) for m in meshes]
    texr = RB.Texture(tex)
    st.held = res + [texr]

    def mesh_draws(draws):
        return [RB.mesh_draw(res[i], shd[i], mvp, vp, first_tri=first, n_tris=count,
                             texture=texr if meshes[i][0] == "tex" else None, cull=case["scene"] == "objects")
                for i, mvp, first, count in draws]

    if case["path"] == "serve":
        st.server = RB.Server(budget_bytes=1 << 30, max_batch=32, n_streams=6)
        st.requests = []
        for w, h, vp, draws in frames:
            st.requests.append((mesh_draws(draws), w, h))
        st.buffers = [np.empty(max(w * h for _, w, h in st.requests) * 4, np.uint8) for _ in st.requests]
        return st
    st.targets, spec = [], []
    for w, h, vp, draws in frames:
        t = Resident(w, h, case["fmt"], case["depth"])
        st.targets.append(t)
        spec.append((t.fb, context(case), mesh_draws(draws)))
    st.batch = RB.Batch(spec)
    st.out = [x for t in st.targets for x in t.tensors()]
    return st


def run(state):
    c = state.case
    if c["path"] == "plain":
        ctx = context(c)
        if not ctx.clear:  # the surface's own content first: the picture it is drawn over
            state.target.color[...] = state.first[0]
            if state.target.depth is not None:
                state.target.depth[...] = state.first[1]
        rf.render(*state.args, state.target, ctx)
        s = ctx.stats
        out = {"color": state.target.color, "stats": [s.prims_o, s.verts_o, s.frags_i, s.frags_o]}
        if state.target.depth is not None:
            out["depth"] = state.target.depth
        return out
    if c["path"] == "serve":
        for i, (draws, w, h) in enumerate(state.requests):
            state.server.submit(i, draws, w, h)
        done, left, out = [], list(state.buffers), [None] * len(state.requests)
        while len(done) < len(state.requests):
            got = state.server.poll(len(left), timeout_ms=1000, buffers=left)
            for r, b in zip(got, left):
                rf.check(r.status)
                out[r.id] = b[:r.width * r.height * 4]
            left = left[len(got):]
            done += got
        return out
    state.batch.run()
    if c["frames"] > 1:
        return state.out
    # a frame loop of single frames reads its statistics too
    s = state.batch.wait()[0]
    return state.out + [s.prims_o, s.verts_o, s.frags_i, s.frags_o]


# ------------------------------------------------------------------ what a pass cannot do without

def work(case):
    """Each mesh and texture read once, each target pixel written once (and read where it is drawn over); the
    vertex transforms, the triangles' planes and the pixels' interpolation."""
    meshes, tex, frames = model(case, 0)
    read = sum(m[1].nbytes + (0 if m[2] is None else m[2].nbytes) + m[3].nbytes for m in meshes)
    read += tex.nbytes if any(m[0] == "tex" for m in meshes) else 0
    px = sum(w * h for w, h, _, _ in frames)
    bpp = ITEM[case["fmt"]][1] + (4 if case["depth"] and case["path"] != "serve" else 0)
    verts = sum(len(meshes[i][1]) for f in frames for i, _, _, _ in f[3])
    prims = sum(k for f in frames for _, _, _, k in f[3])
    return {"bytes": float(read + px * bpp * (2 if case["pitched"] else 1)),
            "flops": float(28 * verts + 60 * prims + 8 * px)}


# ------------------------------------------------------------------ depth in 64 bits

def depth64(meshes, w, h, vp, draws):
    """1 / w of the nearest surface at every pixel centre, 0 where there is none, by homogeneous edge
    functions in 64 bits (no clipping: a pixel's barycentric coordinates over w decide)."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    buf = torch.zeros(h * w + 1, dtype=torch.float64, device=dev)  # the last one takes what is outside

    def t64(a):
        return torch.from_numpy(np.ascontiguousarray(a, np.float64)).to(dev)

    v = t64(vp)
    for i, mvp, first, count in draws:
        pos = t64(meshes[i][1])
        c = torch.cat([pos, torch.ones_like(pos[:, :1])], 1) @ t64(mvp).T
        hom = torch.stack([v[0, 0] * c[:, 0] + v[0, 3] * c[:, 3], v[1, 1] * c[:, 1] + v[1, 3] * c[:, 3], c[:, 3]], 1)
        tri = hom[torch.from_numpy(meshes[i][3][first:first + count].astype(np.int64)).to(dev)]  # n, corner, (x, y, w)
        tri = tri[(tri[:, :, 2] > NEAR).any(1)]
        a, b, d = tri[:, 0], tri[:, 1], tri[:, 2]
        e = torch.stack([torch.linalg.cross(b, d), torch.linalg.cross(d, a), torch.linalg.cross(a, b)], 1)
        det = (a * e[:, 0]).sum(1)
        tri, e, det = tri[det != 0], e[det != 0], det[det != 0]
        e = e / det[:, None, None]
        whole = (tri[:, :, 2] > NEAR).all(1)
        p = tri[:, :, :2] / tri[:, :, 2:]
        lo = torch.where(whole[:, None], p.amin(1), torch.zeros_like(p[:, 0])).floor()
        hi = torch.where(whole[:, None], p.amax(1), torch.tensor([float(w), float(h)], device=dev,
                                                                 dtype=torch.float64)).ceil()
        lim = torch.tensor([float(w), float(h)], device=dev, dtype=torch.float64)
        lo, hi = lo.clamp(min=0), torch.minimum(hi, lim)
        keep = (hi > lo).all(1)
        e, lo, hi = e[keep], lo[keep], hi[keep]
        size = (hi - lo).amax(1)
        k = 4
        while k < 2 * max(w, h):
            mine = (size <= k) & (size > (k // 2 if k > 4 else 0))
            ee, ll = e[mine], lo[mine].long()
            off = torch.arange(k, device=dev)
            step = max(1, (1 << 23) // (k * k))
            for at in range(0, len(ee), step):
                x = ll[at:at + step, 0, None, None] + off[None, None, :]
                y = ll[at:at + step, 1, None, None] + off[None, :, None]
                q = ee[at:at + step, :, :, None, None]
                bary = q[:, :, 0] * (x + 0.5)[:, None] + q[:, :, 1] * (y + 0.5)[:, None] + q[:, :, 2]
                z = bary.sum(1)
                ok = (bary >= 0).all(1) & (z <= 1.0 / NEAR) & (x < w) & (y < h)
                buf.scatter_reduce_(0, torch.where(ok, y * w + x, h * w).reshape(-1), z.reshape(-1), "amax")
            k *= 2
    return buf[:-1].view(h, w).cpu()


def exact(case, seed):
    """The depth buffers in 64 bits (of the first two frames); colours and counts are whole numbers, and a
    line's depth is its first end's, which has no such value."""
    if not case["depth"] or case["scene"] == "wire" or case["path"] == "serve":
        return None
    meshes, _, frames = model(case, seed)
    if case["path"] == "plain":
        w, h, vp, draws = frames[0]
        return {"color": None, "stats": [None] * 4, "depth": depth64(meshes, w, h, vp, draws)}
    out = []
    for i, (w, h, vp, draws) in enumerate(frames):
        out += [None, depth64(meshes, w, h, vp, draws) if i < 2 else None]
    return out + ([None] * 4 if case["frames"] == 1 else [])
