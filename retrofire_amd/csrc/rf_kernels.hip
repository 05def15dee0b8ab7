// HIP kernels of the render path for gfx950 (CDNA4, wave64).
//
//   k_setup    one wave per group of 64 consecutive triangles: primitive
//              assembly (prim.rs:17-19), the built-in vertex shader at each
//              corner (ProjMat3::apply, mat.rs:965-969), outcodes
//              (clip.rs:303-309), frustum clipping (clip.rs:350-400),
//              to_screen, face culling (render.rs:185-196), the tile rectangle
//              of each triangle, and the per-tile count of bin runs.
//   k_scan     exclusive scan of the run counts, the lists of tiles.
//   k_bin      two groups a wave: writes one run (group, 64-bit mask)
//              per distinct tile the group touches.
//   k_binsort  sorts the long run lists by group, which
//              restores primitive submission order inside the tile.
//   k_raster   one wave per tile (persistent): the tile's depth and colour
//              sources live in LDS; a lane walks a triangle's edges, then
//              lanes take its row spans in submission order and apply
//              pixels under ordered (row, 8-column) cell claims (tri_fill/scan
//              raster.rs:185-302, ScanlineIter::next raster.rs:84-113,
//              rasterize_fb target.rs:163-198); the tile is written to HBM
//              once.
//
// The file is compiled three times: as the pipeline (every kernel but k_raster,
// and the launchers), and with RF_RASTER_TU defined as k_raster alone, for
// launches without (0) and with (1) edges, under the max-ilp scheduler. That
// scheduling shortens k_raster's dependent chains (1.145 -> 1.131 ms per 64
// crates1080 frames) and would lengthen k_setup's (0.092 -> 0.096 ms), so it
// applies to k_raster only.
//
// Exactness: the serial recurrences of the reference (edge stepping per row,
// varying stepping per pixel) are reproduced as serial sums; no closed forms.
#include <hip/hip_runtime.h>

#include <cstddef>
#include <type_traits>

#include "rf_ff.hpp"
#include "rf_math.hpp"
#include "rf_types.hpp"
#include "rf_internal.hpp"

namespace rf {

constexpr int WAVE = 64;
typedef uint32_t rf_u32x4 __attribute__((ext_vector_type(4)));
constexpr int BIN_MARGIN = 2;  // pixels around a triangle's bounding box, besides the drift bound
// Rows above the target (y < 0) that a triangle may fold onto row 0; more is
// RF_E_VIEWPORT (the row counter y0 + k, a float in the reference, stays
// exact below 2^22).
constexpr int32_t FOLD_ROWS_MAX = 1 << 22;
// Tuning constants (overridable at build time for sweeps).
#ifndef RF_FF_MIN
#define RF_FF_MIN 12
#endif
constexpr int FF_MIN = RF_FF_MIN;  // step counts above this use the exact fast-forward

// ---------------------------------------------------------------------------
// wave helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

// Cross-lane steps through DPP (row shifts, mirrors and row broadcasts: VALU
// operations, no LDS round trip). Every caller runs with all 64 lanes active.
template <int CTRL, int ROW_MASK = 0xF, int BANK_MASK = 0xF>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t old, uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, ROW_MASK, BANK_MASK, false);
}
constexpr int DPP_QUAD_1032 = 0xB1, DPP_QUAD_2301 = 0x4E, DPP_ROW_MIRROR = 0x140, DPP_ROW_HALF_MIRROR = 0x141,
              DPP_ROW_SHR1 = 0x111, DPP_ROW_SHR2 = 0x112, DPP_ROW_SHR3 = 0x113, DPP_ROW_SHR4 = 0x114,
              DPP_ROW_SHR8 = 0x118, DPP_ROW_BCAST15 = 0x142, DPP_ROW_BCAST31 = 0x143;

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t v) {
    v = min(v, dpp_u32<DPP_QUAD_1032>(v, v));
    v = min(v, dpp_u32<DPP_QUAD_2301>(v, v));
    v = min(v, dpp_u32<DPP_ROW_HALF_MIRROR>(v, v));
    v = min(v, dpp_u32<DPP_ROW_MIRROR>(v, v));
    v = min(v, dpp_u32<DPP_ROW_BCAST15, 0xA>(v, v));
    v = min(v, dpp_u32<DPP_ROW_BCAST31, 0xC>(v, v));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// The least of each 16-bit half.
__device__ __forceinline__ uint32_t min_u16x2(uint32_t a, uint32_t b) {
    using u16x2 = uint16_t __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t wave_min_u16x2(uint32_t v) {
    v = min_u16x2(v, dpp_u32<DPP_QUAD_1032>(v, v));
    v = min_u16x2(v, dpp_u32<DPP_QUAD_2301>(v, v));
    v = min_u16x2(v, dpp_u32<DPP_ROW_HALF_MIRROR>(v, v));
    v = min_u16x2(v, dpp_u32<DPP_ROW_MIRROR>(v, v));
    v = min_u16x2(v, dpp_u32<DPP_ROW_BCAST15, 0xA>(v, v));
    v = min_u16x2(v, dpp_u32<DPP_ROW_BCAST31, 0xC>(v, v));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// Inclusive scan with operator op over the lanes; `id` is op's identity.
template <class Op>
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v, uint32_t id, Op op) {
    uint32_t x = op(v, dpp_u32<DPP_ROW_SHR1>(id, v));
    x = op(x, dpp_u32<DPP_ROW_SHR2>(id, v));
    x = op(x, dpp_u32<DPP_ROW_SHR3>(id, v));
    x = op(x, dpp_u32<DPP_ROW_SHR4, 0xF, 0xE>(id, x));
    x = op(x, dpp_u32<DPP_ROW_SHR8, 0xF, 0xC>(id, x));
    x = op(x, dpp_u32<DPP_ROW_BCAST15, 0xA>(id, x));
    x = op(x, dpp_u32<DPP_ROW_BCAST31, 0xC>(id, x));
    return x;
}
__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
    return v;
}
// Exclusive prefix sum over the wave.
__device__ __forceinline__ uint32_t wave_excl_scan(uint32_t v, uint32_t* total) {
    const uint32_t x = wave_incl_scan(v, 0u, [](uint32_t a, uint32_t b) { return a + b; });
    *total = (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
    return x - v;
}

// Rust's saturating float-to-integer casts (`as i32`, `as u32`, `as u8`) in
// one instruction each: V_CVT_I32_F32 and V_CVT_U32_F32 truncate toward
// zero, saturate out-of-range values (infinities included) and convert NaN to
// 0, which is exactly the `as` semantics; a C cast would leave those cases
// undefined.
__device__ __forceinline__ int32_t cvt_i32(float x) {
    int32_t r;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}
__device__ __forceinline__ uint32_t cvt_u32(float x) {
    uint32_t r;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}
__device__ __forceinline__ uint32_t cvt_u8(float x) {
    const uint32_t r = cvt_u32(x);
    return r < 255u ? r : 255u;
}

__device__ __forceinline__ uint32_t find_draw_tri(const DrawDesc* d, uint32_t n, uint64_t g) {
    uint32_t lo = 0, hi = n;  // last draw with tri_base <= g
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (d[mid].tri_base <= g) lo = mid; else hi = mid;
    }
    return lo;
}
// The same searches from a hint: the last draw with base <= a key at or
// before this one (draw bases never decrease); usually one load.
__device__ __forceinline__ uint32_t draw_of_tri(const DrawDesc* d, uint32_t n, uint32_t hint, uint64_t g) {
    uint32_t k = hint;
    while (k + 1 < n && d[k + 1].tri_base <= g) ++k;
    return k;
}
// ---------------------------------------------------------------------------
// k_setup helpers: clipping in registers
// ---------------------------------------------------------------------------
struct CV {
    float p[4];
    float a[3];
    uint32_t oc;
};

__device__ __forceinline__ void cv_make(CV& o, const float* p, const float* a) {
    for (int k = 0; k < 4; ++k) o.p[k] = p[k];
    for (int k = 0; k < 3; ++k) o.a[k] = a[k];
    o.oc = outcode(p[0], p[1], p[2], p[3]);
}

// vertex(mvp.apply(&v.pos), v.attrib) of the built-in vertex shader: the
// clip position of a draw's vertex i (ProjMat3::apply, mat.rs:965-969, to_hom
// w = 1) and its attributes. Shaded at each corner that names the vertex:
// the same operations on the same inputs give the same bits, and a triangle's
// corners cost less than writing every vertex of the mesh to HBM (56 bytes
// each) and reading it back: 8 frames of 3.2M triangles took 0.36 ms in a
// vertex kernel and 1.22 in k_setup, and took 1.25 in k_setup alone (1.19 now,
// the small triangles' walk included); 32 mixed frames whose draws use a part of
// their mesh 1.27 + 2.67, then 2.80 (2.31).
__device__ __forceinline__ void shade_pos(const float* m, const float* pos, uint32_t i, float* p) {
    const float x = pos[3ull * i], y = pos[3ull * i + 1], z = pos[3ull * i + 2];
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] = dot4(m + 4 * r, x, y, z, 1.0f);
}
__device__ __forceinline__ void fetch_attr(uint32_t kind, const float* attr, uint32_t stride, uint32_t i, float* a) {
    const int na = kind_attrs(kind);
    const float* src = attr + (uint64_t)stride * i;
    a[0] = a[1] = a[2] = 0.0f;
    if (na >= 2) {
        a[0] = src[0];
        a[1] = src[1];
    }
    if (na == 3) a[2] = src[2];
}
__device__ __forceinline__ void shade_vertex(const DrawDesc* D, uint32_t i, CV& o) {
    shade_pos(D->mvp, D->pos, i, o.p);
    fetch_attr(D->kind, D->attr, D->attr_stride, i, o.a);
    o.oc = outcode(o.p[0], o.p[1], o.p[2], o.p[3]);
}

// Screen vertex of a clip vertex (to_screen, prim.rs:62-88).
__device__ __forceinline__ void to_screen(const CV& c, const float* vp, bool persp, float* s) {
    const float w = c.p[3];
    const float nx = c.p[0] / w, ny = c.p[1] / w, nz = 1.0f / w;
    s[0] = dot4(vp + 0, nx, ny, nz, 1.0f);
    s[1] = dot4(vp + 4, nx, ny, nz, 1.0f);
    s[2] = dot4(vp + 8, nx, ny, nz, 1.0f);
    s[3] = persp ? c.a[0] / w : c.a[0];
    s[4] = persp ? c.a[1] / w : c.a[1];
    s[5] = persp ? c.a[2] / w : c.a[2];
}

// Tri::winding() == Cw (geom/prim.rs:288-295).
__device__ __forceinline__ bool backface(const float* s0, const float* s1, const float* s2) {
    const float ux = s1[0] - s0[0], uy = s1[1] - s0[1];
    const float vx = s2[0] - s0[0], vy = s2[1] - s0[1];
    float z = 0.0f;
    z = z + (-uy) * vx;
    z = z + ux * vy;
    return z < 0.0f;
}
__device__ __forceinline__ bool culled(int32_t fc, bool bf) {
    return (fc == FC_BACK && bf) || (fc == FC_FRONT && !bf);
}

// Sutherland-Hodgman over the six planes (clip.rs:167-193, 283-301).
// `poly` holds n vertices on entry; returns the output count (0..CLIP_MAX), or
// -1 if a plane would produce more than CLIP_MAX vertices (a convex polygon
// gains at most one vertex per plane, 3 + 6 = 9; more only arises from a
// numerically non-convex polygon and is reported instead of stored).
constexpr int CLIP_MAX = 9;
__device__ int clip_polygon(CV* poly, int n, CV* tmp) {
    CV* in = poly;
    CV* out = tmp;
    for (int p = 0; p < 6; ++p) {
        const uint32_t bit = 1u << p;
        // a plane that every vertex is inside of keeps them all and cuts no
        // edge (no distance is > 0, so no product of two is < 0): most
        // polygons meet one plane of the six
        uint32_t any = 0;
        for (int k = 0; k < n; ++k) any |= in[k].oc;
        if ((any & bit) == 0) continue;
        int m = 0;
        for (int k = 0; k < n; ++k) {
            const CV& v0 = in[k];
            const CV& v1 = in[k + 1 < n ? k + 1 : 0];
            if ((bit & v0.oc) == 0) {
                if (m == CLIP_MAX) return -1;
                out[m++] = v0;
            }
            const float d0 = plane_dist(p, v0.p[0], v0.p[1], v0.p[2], v0.p[3]);
            const float d1 = plane_dist(p, v1.p[0], v1.p[1], v1.p[2], v1.p[3]);
            if (d0 * d1 < 0.0f) {
                if (m == CLIP_MAX) return -1;
                const float t = -d0 / (d1 - d0);
                float q[4], a[3];
                for (int c = 0; c < 4; ++c) q[c] = v0.p[c] + (v1.p[c] - v0.p[c]) * t;
                for (int c = 0; c < 3; ++c) a[c] = v0.a[c] + (v1.a[c] - v0.a[c]) * t;
                cv_make(out[m++], q, a);
            }
        }
        n = m;
        if (n == 0) break;
        CV* s = in; in = out; out = s;
    }
    if (n > 0 && in != poly)
        for (int k = 0; k < n; ++k) poly[k] = in[k];
    return n;
}

__device__ __forceinline__ void write_scr(ScrTri* dst, const float* s0, const float* s1,
                                          const float* s2, uint32_t draw, uint32_t kind) {
    float* d = &dst->v[0][0];
    for (int c = 0; c < 6; ++c) d[c] = s0[c];
    for (int c = 0; c < 6; ++c) d[6 + c] = s1[c];
    for (int c = 0; c < 6; ++c) d[12 + c] = s2[c];
    dst->draw = draw;
    dst->kind = kind;
}

// Screen-space extent of a primitive's vertices. fminf / fmaxf skip NaN
// operands, so the extent is that of the vertices' numbers; `nan` records a
// NaN x or y, `inf` an infinite one.
struct RectAcc {
    float xmin, xmax, ymin, ymax;
    bool nan, inf;
    __device__ void init() {
        xmin = ymin = __builtin_inff();
        xmax = ymax = -__builtin_inff();
        nan = inf = false;
    }
    __device__ void add(const float* s) {
        nan = nan || s[0] != s[0] || s[1] != s[1];
        inf = inf || __builtin_isinf(s[0]) || __builtin_isinf(s[1]);
        xmin = fminf(xmin, s[0]);
        xmax = fmaxf(xmax, s[0]);
        ymin = fminf(ymin, s[1]);
        ymax = fmaxf(ymax, s[1]);
    }
};

// Pixel rectangle that holds a triangle's pixels. Rows are exact: tri_fill covers rows
// floor(top_y + 0.5) .. floor(bot_y + 0.5) (scan, raster.rs:286-300). Columns
// are the vertex x range widened by a margin that bounds how far the serially
// stepped edges drift from the exact edges (the rasterizer checks every span
// stays inside):
//   - each row step x + dl rounds by at most half an ulp of the values it
//     passes, so n steps drift by at most n * ulp(X) / 2, X bounding |x|;
//   - dl itself, (x1 - x0) * (1 / (y1 - y0)), is off by a few ulps relative,
//     which over the edge's rows adds at most |x1 - x0| * 2^-22.
// margin_px = BIN_MARGIN + round(D), with D = rows * ulp(X) +
// (xmax - xmin) * 2^-20 (twice and four times those bounds), tolerates a
// drift of D + 1 pixel beyond the rounding of the span ends (round_up_to_half)
// that BIN_MARGIN alone covers. Ordinary content keeps the base margin
// (1080p: X < 2048, a few hundred rows, D < 0.5); a 16k-row edge at
// x = 16,000 gets 18 pixels.
__device__ __forceinline__ int32_t bin_margin(const RectAcc& r, float rows) {
    const float xmin = __builtin_isfinite(r.xmin) ? r.xmin : 0.0f, xmax = __builtin_isfinite(r.xmax) ? r.xmax : 0.0f;
    const float X = fmaxf(fabsf(xmin), fabsf(xmax)) + 1.0f;
    const float ulp = u2f((f2u(X) & 0x7F800000u) - (23u << 23));  // ulp of X (X >= 1)
    const float D = rows * ulp + (xmax - xmin) * 0x1p-20f;
    return BIN_MARGIN + (int32_t)floorf(D + 0.5f);
}
//
// A triangle with a NaN vertex (the screen position of a w = 0 clip vertex,
// 0/0) draws no pixel, but its rows whose left edge is NaN are spans
// `0..x1` (`x0 as usize` of NaN is 0, raster.rs:104-107) that count in
// frags.i: its columns start at 0.
__device__ __forceinline__ bool pixel_rect(const RectAcc& r, uint32_t width, uint32_t height, uint32_t* out) {
    const float r0 = floorf(r.ymin + 0.5f), r1 = floorf(r.ymax + 0.5f);
    if (!(r1 > r0)) return false;
    const float xmin = r.nan ? 0.0f : r.xmin, xmax = r.xmax >= xmin ? r.xmax : xmin;
    const int32_t margin = bin_margin(r, r1 - r0);
    // saturating 32-bit steps: past 2^31 the rectangle is only larger
    // rows above the target fold onto row 0 (`self.y as usize`, raster.rs:106)
    const int32_t row0 = max(cvt_i32(r0), 0), row1 = min(max(cvt_i32(r1) - 1, 0), (int32_t)height - 1);
    const int32_t c0 = max(__builtin_elementwise_sub_sat(cvt_i32(floorf(xmin)), margin), 0);
    const int32_t c1 = min(__builtin_elementwise_add_sat(cvt_i32(floorf(xmax)), margin), (int32_t)width - 1);
    if (row1 < row0 || c1 < c0) return false;
    out[0] = (uint32_t)c0 | ((uint32_t)row0 << 16);
    out[1] = (uint32_t)c1 | ((uint32_t)row1 << 16);
    return true;
}

// The tiles (of 1 << twl columns x 1 << thl rows) a pixel rectangle meets:
// one corner's tile column | tile row << 16.
__device__ __forceinline__ uint32_t rect_tile(uint32_t corner, uint32_t twl, uint32_t thl) {
    return ((corner & 0xFFFFu) >> twl) | ((corner >> 16 >> thl) << 16);
}

// Visit, over the whole wave, each distinct tile in the union of the lanes'
// rectangles, in increasing tile order: lane k collects the k-th tile and the
// mask of the lanes whose rectangles contain it, and `flush(n, tile, mask,
// first)` runs on the whole wave for every 64 of them and for the rest. Each
// lane walks its own rectangle in row-major (= increasing id) order; the wave
// minimum of the lanes' next tiles is processed next, so a lane whose rectangle
// contains that tile always has it as its next one. Returns their number.
template <class Fn>
__device__ __forceinline__ uint32_t for_each_tile(bool valid, uint32_t r0, uint32_t r1, uint32_t base, uint32_t ntx,
                                                  Fn&& flush) {
    const uint32_t tx0 = r0 & 0xFFFF, tx1 = r1 & 0xFFFF, ty1 = r1 >> 16;
    uint32_t cx = tx0, next = valid ? base + (r0 >> 16) * ntx + tx0 : 0xFFFFFFFFu;
    const uint32_t last = base + ty1 * ntx + tx1, row = ntx - (tx1 - tx0);
    uint32_t my_tile = 0, k = 0, done = 0;
    unsigned long long my_mask = 0;
    for (;;) {
        const uint32_t t = wave_min_u32(next);
        if (t == 0xFFFFFFFFu) break;
        const bool mine = next == t;
        const unsigned long long m = __ballot(mine);
        if (lane_id() == k) {
            my_tile = t;
            my_mask = m;
        }
        if (++k == (uint32_t)WAVE) {
            flush(k, my_tile, my_mask, done == 0);
            done += k;
            k = 0;
        }
        if (mine) {
            const bool wrap = cx == tx1;
            next = next == last ? 0xFFFFFFFFu : next + (wrap ? row : 1u);
            cx = wrap ? tx0 : cx + 1;
        }
    }
    if (k) flush(k, my_tile, my_mask, done == 0);
    return done + k;
}

// One Edge<usize> primitive (prim.rs:41-60): assembly, edge clipping
// (clip.rs:311-348), to_screen, face culling (an edge is never a backface,
// render.rs:72-75, so only FaceCull::Front drops it, ctx.rs:95-101), and the
// set-up of raster::line (raster.rs:122-177). Returns the primitives kept (0
// or 1). The ScrTri holds in v[0] the line's first end after the swaps (its z
// and varyings are every fragment's) and in v[1] its pixel walk: first
// column (wide) or row (tall), pixel count, the stepped coordinate's start
// and step, and the wide flag. The binning rectangle is the exact pixel
// rectangle; a pixel outside the target is the reference's out-of-bounds
// panic (target.rs:173-174).
__device__ uint32_t edge_setup(const BatchDesc& B, const DrawDesc* D, const FrameDesc& F, uint32_t di, uint64_t g,
                               uint64_t t, uint32_t* rect, bool& has_rect) {
    const uint32_t i0 = D->tris[2 * t], i1 = D->tris[2 * t + 1];
    if (i0 >= D->n_verts || i1 >= D->n_verts) {
        atomicOr(B.err, ERRB_INDEX);
        return 0;
    }
    CV ea, eb;
    shade_vertex(D, i0, ea);
    shade_vertex(D, i1, eb);
    if (ea.oc & eb.oc) return 0;  // both ends outside one plane
    const bool persp = kind_persp(D->kind);
    float a[6], b[6];
    if ((ea.oc | eb.oc) != 0) {
        for (int p = 0; p < 6; ++p) {
            const uint32_t bit = 1u << p;
            const bool a_in = (bit & ea.oc) == 0, b_in = (bit & eb.oc) == 0;
            if (!a_in && !b_in) return 0;
            // ClipPlane::intersect (clip.rs:121-145)
            const float d0 = plane_dist(p, ea.p[0], ea.p[1], ea.p[2], ea.p[3]);
            const float d1 = plane_dist(p, eb.p[0], eb.p[1], eb.p[2], eb.p[3]);
            if (d0 * d1 < 0.0f) {
                const float tt = -d0 / (d1 - d0);
                float q[4], qa[3];
                for (int c = 0; c < 4; ++c) q[c] = ea.p[c] + (eb.p[c] - ea.p[c]) * tt;
                for (int c = 0; c < 3; ++c) qa[c] = ea.a[c] + (eb.a[c] - ea.a[c]) * tt;
                CV v;
                cv_make(v, q, qa);
                if (a_in) eb = v;
                else if (b_in) ea = v;
            }
        }
    }
    to_screen(ea, D->vp, persp, a);
    to_screen(eb, D->vp, persp, b);
    if (F.face_cull == FC_FRONT) return 0;
    if (!(__builtin_isfinite(a[0]) && __builtin_isfinite(a[1]) && __builtin_isfinite(b[0]) &&
          __builtin_isfinite(b[1]))) {
        atomicOr(B.err, ERRB_NONFINITE);
        return 0;
    }
    // raster::line: top end first; a wide line then runs left to right
    float v0[6], v1[6];
    const bool sw = a[1] > b[1];
    for (int c = 0; c < 6; ++c) {
        v0[c] = sw ? b[c] : a[c];
        v1[c] = sw ? a[c] : b[c];
    }
    const float dx = v1[0] - v0[0], dy = v1[1] - v0[1];
    const bool wide = fabsf(dx) > dy;
    if (wide && dx < 0.0f)
        for (int c = 0; c < 6; ++c) {
            const float tmp = v0[c];
            v0[c] = v1[c];
            v1[c] = tmp;
        }
    // wide: columns (x0 as usize)..(x1 as usize), y stepped by dy/dx from its
    // value at the rounded x0; tall: rows likewise, x stepped by dx/dy
    const int ax = wide ? 0 : 1;  // the axis walked pixel by pixel
    const float r0 = round_up_to_half(v0[ax]), r1 = round_up_to_half(v1[ax]);
    const float step = wide ? dy / dx : dx / dy;
    const float base = v0[1 - ax] + step * (r0 - v0[ax]);
    const uint64_t S64 = as_usize(r0), E64 = as_usize(r1);
    const uint64_t n64 = E64 > S64 ? E64 - S64 : 0;
    float* d = &B.scr[g].v[0][0];
    for (int c = 0; c < 6; ++c) d[c] = v0[c];
    B.scr[g].draw = di;
    B.scr[g].kind = D->kind | KIND_LINE;
    if (n64 == 0) {
        d[6] = u2f(0);
        d[7] = u2f(0);
        return 1;  // counted, draws nothing
    }
    const uint64_t lim_walk = wide ? F.width : F.height, lim_step = wide ? F.height : F.width;
    if (E64 > lim_walk) {
        atomicOr(B.err, ERRB_BOUNDS);
        return 1;
    }
    const uint32_t S = (uint32_t)S64, n = (uint32_t)n64;
    const float last = n > 1 ? ff_add(base, step, n - 1) : base;
    // the stepped coordinate is monotone along the walk, so its pixels lie
    // between those of the first and last steps
    const uint64_t e0 = as_usize(base), e1 = as_usize(last);
    const uint64_t lo = e0 < e1 ? e0 : e1, hi = e0 < e1 ? e1 : e0;
    if (hi >= lim_step) {
        atomicOr(B.err, ERRB_BOUNDS);
        return 1;
    }
    d[6] = u2f(S);
    d[7] = u2f(n);
    d[8] = base;
    d[9] = step;
    d[10] = u2f(wide ? 1u : 0u);
    d[11] = 0.0f;
    const uint32_t w0 = S, w1 = S + n - 1, t0 = (uint32_t)lo, t1 = (uint32_t)hi;
    rect[0] = wide ? (w0 | t0 << 16) : (t0 | w0 << 16);
    rect[1] = wide ? (w1 | t1 << 16) : (t1 | w1 << 16);
    has_rect = true;
    return 1;
}

struct Trap {
    float y0i;             // first row (floor(y0 + 0.5))
    uint32_t n;            // row count
    float lx, lz, la[3];   // left state at the first row
    float dlx, dlz, dla[3];
    float rx, drx;         // right x at the first row, step
    float dvz, dva[3];     // d(varyings)/dx
};
struct Slot {
    Trap t[2];
    int32_t ylo, yhi;      // rows covered (absolute)
};

// scan (raster.rs:248-302) for one trapezoid; y components are not needed by
// any output and are left out.
__device__ __forceinline__ void scan_setup(Trap& T, float y0, float y1, const float* l0,
                                           const float* l1, const float* r0, const float* r1,
                                           int na) {
    // l*/r* layout: x, y, z, a0, a1, a2
    const float recip_dy = 1.0f / (y1 - y0);
    float dl[6], dr[6];
    for (int c = 0; c < 6; ++c) {
        dl[c] = (l1[c] - l0[c]) * recip_dy;
        dr[c] = (r1[c] - r0[c]) * recip_dy;
    }
    float l0s[6], r0s[6];
    for (int c = 0; c < 6; ++c) {
        l0s[c] = l0[c] + dl[c];
        r0s[c] = r0[c] + dr[c];
    }
    const float dx = r0s[0] - l0s[0];
    const float rdx = 1.0f / dx;
    T.dvz = (r0s[2] - l0s[2]) * rdx;
    for (int c = 0; c < 3; ++c) T.dva[c] = (c < na) ? (r0s[3 + c] - l0s[3 + c]) * rdx : 0.0f;
    const float y0r = round_up_to_half(y0);
    const float y1r = round_up_to_half(y1);
    const float tweak = y0r - y0;
    // l0.lerp(&l0.step(&dl_dy), y_tweak) == l0 + ((l0 + dl) - l0) * tweak
    T.lx = l0[0] + (l0s[0] - l0[0]) * tweak;
    T.lz = l0[2] + (l0s[2] - l0[2]) * tweak;
    for (int c = 0; c < 3; ++c) T.la[c] = (c < na) ? l0[3 + c] + (l0s[3 + c] - l0[3 + c]) * tweak : 0.0f;
    T.dlx = dl[0];
    T.dlz = dl[2];
    for (int c = 0; c < 3; ++c) T.dla[c] = (c < na) ? dl[3 + c] : 0.0f;
    T.rx = r0[0] + dr[0] * tweak;
    T.drx = dr[0];
    T.n = as_u32(y1r - y0r);
    T.y0i = y0r - 0.5f;
}

// tri_fill (raster.rs:185-224) setup for one screen triangle (vertices as
// x, y, z, a0, a1, a2; sorted in registers).
__device__ __forceinline__ void swap6(float* a, float* b) {
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const float t = a[k];
        a[k] = b[k];
        b[k] = t;
    }
}
// The total_cmp order key of a screen y. A NaN y (0/0, the screen position
// of a w = 0 clip vertex) is keyed as x86-64's default NaN, which has its
// sign bit set and so sorts before -inf: that is the NaN the reference's
// arithmetic produces there (the GPU's own NaN has no defined sign).
__device__ __forceinline__ int32_t y_key(float y) { return total_key(y == y ? y : u2f(0xFFC00000u)); }

__device__ __forceinline__ void tri_setup(Slot& S, float (&va)[6], float (&vb)[6], float (&vc)[6], int na) {
    // stable sort by total_cmp of y (slice::sort_by is stable)
    if (y_key(vb[1]) < y_key(va[1])) swap6(va, vb);
    if (y_key(vc[1]) < y_key(vb[1])) swap6(vb, vc);
    if (y_key(vb[1]) < y_key(va[1])) swap6(va, vb);
    const float* top = va;
    const float* mid0 = vb;
    const float* bot = vc;
    const float top_y = top[1], mid_y = mid0[1], bot_y = bot[1];
    const float tt = (mid_y - top_y) / (bot_y - top_y);
    float mid1[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) mid1[k] = top[k] + (bot[k] - top[k]) * tt;
    const bool l_is_mid0 = mid0[0] < mid1[0];
    float left[6], right[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        left[k] = l_is_mid0 ? mid0[k] : mid1[k];
        right[k] = l_is_mid0 ? mid1[k] : mid0[k];
    }
    scan_setup(S.t[0], top_y, mid_y, top, left, top, right, na);
    scan_setup(S.t[1], mid_y, bot_y, left, bot, right, bot, na);
    int32_t lo = 0x7FFFFFFF, hi = -0x7FFFFFFF;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (S.t[h].n == 0) continue;
        const int32_t y0 = (int32_t)S.t[h].y0i;
        const int32_t y1 = y0 + (int32_t)S.t[h].n;
        lo = y0 < lo ? y0 : lo;
        hi = y1 > hi ? y1 : hi;
    }
    S.ylo = lo;
    S.yhi = hi;
}

// ---------------------------------------------------------------------------
// Small triangles: what the rasterizer needs to pass over one without
// walking it
// ---------------------------------------------------------------------------
// A scene of many small triangles is mostly hidden: of 8 icospheres1080
// frames' 285M fragments 43M pass the depth test. The rasterizer skips a
// triangle of a tile whose every fragment must fail (see k_raster), but the
// fragments still count in frags.i, and rows outside the target still are an
// error. So k_setup walks the rows of each triangle of up to SMALL_ROWS rows
// here, once: x only, the same serial sums as the rasterizer's, and an upper
// bound of its fragments' z. Larger triangles are counted where they are
// drawn.
//
// A triangle without any fragment (no pixel centre in it) is not binned at all:
// one 125 x 181 frame of 519 icospheres 0.60 -> 0.24 ms in the rasterizer.
//
// The walk costs a small launch 4 to 8 us (one 256 x 256 frame of 20 crates:
// k_setup 8.8 -> 14.2 us), so it is made where tiles have more triangles than
// this on average: at 0, 8 and 32, crates and lines lose 5, 1 and 0 us, and 4
// frames of 160,000 depth-sorted triangles gain 8 in all three.
#ifndef RF_SMALL_TRIS
#define RF_SMALL_TRIS 32
#endif
constexpr uint32_t SMALL_ROWS = 32;
struct SmallTri {
    uint32_t frags;  // frags.i of the whole triangle
    float zmax;      // no fragment's z is above this
    uint32_t err;
};
// The triangle's corners are finite and at or below row 0; cols: the columns
// of its tiles, first | end << 16. False (nothing counted) if it is too tall
// or the bound is not finite.
__device__ __forceinline__ bool small_tri(const float* v0, const float* v1, const float* v2, uint32_t width,
                                          uint32_t height, uint32_t cols, SmallTri& o) {
    float va[6], vb[6], vc[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        va[c] = v0[c];
        vb[c] = v1[c];
        vc[c] = v2[c];
    }
    Slot S;
    tri_setup(S, va, vb, vc, 0);
    o.frags = o.err = 0;
    o.zmax = -__builtin_inff();
    const uint32_t n0 = S.t[0].n, n1 = S.t[1].n;
    if (n0 > SMALL_ROWS || n1 > SMALL_ROWS || n0 + n1 > SMALL_ROWS) return false;
    // Both halves in one loop, so that a wave takes as many steps as its
    // tallest triangle has rows (8 icosphere frames: 1.53 -> 1.49 ms). Span ends as cvt_u32(x + 0.5): what
    // cvt_u32(round_up_to_half(x)) is below 2^23, and above it both are past
    // any target. Ends outside the target or the tiles' columns are met again
    // below.
    float wh[2] = {0.0f, 0.0f};
    bool out = (n0 != 0 && (uint32_t)(int32_t)S.t[0].y0i + n0 > height) ||
               (n1 != 0 && (uint32_t)(int32_t)S.t[1].y0i + n1 > height);
    {
        float lx = S.t[0].lx, rx = S.t[0].rx, dlx = S.t[0].dlx, drx = S.t[0].drx, w = 0.0f;
        uint32_t lo = 0xFFFFFFFFu, hi = 0;
        for (uint32_t k = 0; k < n0 + n1; ++k) {
            if (k == n0) {
                lx = S.t[1].lx;
                rx = S.t[1].rx;
                dlx = S.t[1].dlx;
                drx = S.t[1].drx;
                wh[0] = w;
                w = 0.0f;
            }
            w = fmaxf(w, rx - lx);
            const uint32_t xs = cvt_u32(lx + 0.5f), xe = max(cvt_u32(rx + 0.5f), xs);
            lo = min(lo, xs);
            hi = max(hi, xe);
            o.frags += xe - xs;
            lx = lx + dlx;
            rx = rx + drx;
        }
        wh[0] = n1 == 0 ? w : wh[0];
        wh[1] = w;
        out = out || hi > width || (n0 + n1 != 0 && (lo < (cols & 0xFFFFu) || hi > (cols >> 16)));
    }
    if (out) {
        o.frags = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const Trap& T = S.t[h];
            float lx = T.lx, rx = T.rx;
            uint32_t y = (uint32_t)(int32_t)T.y0i;
            for (uint32_t k = 0; k < T.n; ++k, ++y) {
                const uint32_t xs = cvt_u32(round_up_to_half(lx));
                uint32_t xe = cvt_u32(round_up_to_half(rx));
                xe = xe < xs ? xs : xe;
                if (xe > width || y >= height) {
                    o.err |= ERRB_BOUNDS;
                } else {
                    if (xe > xs && (xs < (cols & 0xFFFFu) || xe > (cols >> 16))) o.err |= ERRB_MARGIN;
                    o.frags += xe - xs;
                }
                lx = lx + T.dlx;
                rx = rx + T.drx;
            }
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const Trap& T = S.t[h];
        if (T.n == 0) continue;
        // z starts at the left edge (lz + k dlz) and goes on by dvz a pixel,
        // at most w + 1 pixels: a bound of the exact values, and of the
        // rounding of rows + w + 8 operations on values up to m (each half an
        // ulp, 2^-24 relative; taken four times)
        const float n = (float)T.n, w = wh[h], m = fabsf(T.lz) + n * fabsf(T.dlz) + (w + 2.0f) * fabsf(T.dvz);
        const float z = fmaxf(T.lz, T.lz + n * T.dlz) + (w + 2.0f) * fmaxf(T.dvz, 0.0f) + (n + w + 8.0f) * 0x1p-22f * m;
        o.zmax = z > o.zmax || z != z ? z : o.zmax;
        if (z != z) return false;
    }
    return o.zmax < __builtin_inff();
}

// ---------------------------------------------------------------------------
// k_setup
// ---------------------------------------------------------------------------
#ifndef RF_RASTER_TU
// The corners of triangle (i0, i1, i2) of draw D: clip positions, outcodes,
// and screen positions of a triangle that needs no clipping (prim.rs:62-88).
// Called with D wave-uniform (the matrices come through scalar loads) or not.
__device__ __forceinline__ void corners(const float* mvp, const float* v, const float* pos, const uint32_t* ix,
                                        float (&p)[3][4], uint32_t (&oc)[3], float (&s)[3][3]) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        shade_pos(mvp, pos, ix[k], p[k]);
        oc[k] = outcode(p[k][0], p[k][1], p[k][2], p[k][3]);
    }
    if ((oc[0] | oc[1] | oc[2]) == 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float w = p[k][3];
            const float nx = p[k][0] / w, ny = p[k][1] / w, nz = 1.0f / w;
            s[k][0] = dot4(v + 0, nx, ny, nz, 1.0f);
            s[k][1] = dot4(v + 4, nx, ny, nz, 1.0f);
            s[k][2] = dot4(v + 8, nx, ny, nz, 1.0f);
        }
    }
}

// What k_setup reads of a triangle's draw and frame.
//
// k_setup of a dense batch is bound by VALU issue and by what it waits for: 8
// frames of 3.2M icosphere triangles issued 1,770 VALU and 62 memory
// instructions a wave (1.49 ms), more than half of the latter for the draw's
// and frame's fields, lane by lane. With those read by the wave, 32-bit rectangles, the
// tiles of a group asked in turn and six waves a SIMD (80 VGPRs; 83 and five
// without the bound, and at seven it spills: 1.34 and 1.36 ms) it takes 1.19
// ms instead of 1.53, and 2.31 instead of 2.88 for 32 mixed frames.
struct DrawIn {
    const float *pos, *attr;
    const uint32_t* tris;
    uint64_t tri_base;
    uint32_t n_verts, kind, attr_stride, prim, pre, frame, width, height, tile_base, ntx;
    int32_t face_cull;
    __device__ __forceinline__ void read(const BatchDesc& B, uint32_t di) {
        const DrawDesc& D = B.draws[di];
        const FrameDesc& F = B.frames[D.frame];
        pos = D.pos;
        attr = D.attr;
        tris = D.tris;
        tri_base = D.tri_base;
        n_verts = D.n_verts;
        kind = D.kind;
        attr_stride = D.attr_stride;
        prim = D.prim;
        pre = D.pre;
        frame = D.frame;
        width = F.width;
        height = F.height;
        tile_base = F.tile_base;
        ntx = F.ntx;
        face_cull = F.face_cull;
    }
};

__global__ __launch_bounds__(256, 6) void k_setup(BatchDesc B) {
    const uint32_t lane = lane_id();
    const uint32_t group = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (group >= B.n_groups) return;  // whole wave exits together
    const uint64_t g = (uint64_t)group * WAVE + lane;
    bool valid = g < B.n_tris;
    uint32_t nf = 0, extra_base = 0;
    uint32_t rect[2] = {0, 0};
    bool has_rect = false;
    uint32_t frags = 0;
    float zmax = __builtin_nanf("");  // not known
    bool empty = false;  // a small triangle without a fragment: nothing to bin
    bool hr = false;     // rect is the triangle's already
    const uint32_t twl = (uint32_t)__builtin_ctz(B.tile_w), thl = (uint32_t)__builtin_ctz(B.tile_h);
    uint32_t frame = 0xFFFFFFFFu;
    const uint32_t d0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)B.group_draw[group]);
    const uint32_t di = valid ? draw_of_tri(B.draws, B.n_draws, d0, g) : d0;
    const bool uniform = __ballot(di != d0) == 0ull;
    // The draw and its frame: of the whole wave in scalar loads (before any
    // store), or each lane's own.
    DrawIn I;
    if (uniform) I.read(B, d0);
    else I.read(B, di);
    frame = valid ? I.frame : frame;
    if (valid) {
        const DrawDesc* D = &B.draws[di];
        const FrameDesc& F = B.frames[frame];
        const uint64_t t = g - I.tri_base;
        if (B.any_cull && !B.draw_vis[di]) {
            // the caller skips a hidden object before render() (crates.rs:118-122)
        } else if (I.prim == PRIM_EDGE) {
            nf = edge_setup(B, D, F, di, g, t, rect, has_rect);
        } else if (!I.pre && (I.tris[3 * t] >= I.n_verts || I.tris[3 * t + 1] >= I.n_verts ||
                               I.tris[3 * t + 2] >= I.n_verts)) {
            atomicOr(B.err, ERRB_INDEX);
        } else {
            uint32_t ix[3] = {(uint32_t)(3 * t), (uint32_t)(3 * t + 1), (uint32_t)(3 * t + 2)};
            if (!I.pre)
#pragma unroll
                for (int k = 0; k < 3; ++k) ix[k] = I.tris[3 * t + k];
            float p[3][4], sp[3][3];
            uint32_t oc[3] = {0, 0, 0};
            if (!I.pre) {
                if (uniform) corners(B.draws[d0].mvp, B.draws[d0].vp, I.pos, ix, p, oc, sp);
                else corners(D->mvp, D->vp, I.pos, ix, p, oc, sp);
            }
            const uint32_t all_out = oc[0] & oc[1] & oc[2], any_out = oc[0] | oc[1] | oc[2];
            RectAcc ra;
            ra.init();
            if (all_out != 0) {
                // Hidden
            } else if (any_out == 0) {
                // Visible
                float v[3][6];
                if (I.pre) {  // a depth-sorted clip fan's screen vertices
#pragma unroll
                    for (int k = 0; k < 3; ++k)
#pragma unroll
                        for (int c = 0; c < 6; ++c) v[k][c] = B.sv[6 * (D->vert_base + ix[k]) + c];
                } else {
#pragma unroll
                    for (int k = 0; k < 3; ++k)
#pragma unroll
                        for (int c = 0; c < 3; ++c) v[k][c] = sp[k][c];
                }
                if (!culled(I.face_cull, backface(v[0], v[1], v[2]))) {
                    if (!I.pre) {
#pragma unroll
                        for (int k = 0; k < 3; ++k) fetch_attr(I.kind, I.attr, I.attr_stride, ix[k], &v[k][3]);
                        if (kind_persp(I.kind)) {
#pragma unroll
                            for (int k = 0; k < 3; ++k)
#pragma unroll
                                for (int c = 3; c < 6; ++c) v[k][c] = v[k][c] / p[k][3];
                        }
                    }
                    ra.add(v[0]);
                    ra.add(v[1]);
                    ra.add(v[2]);
                    nf = 1;
                    uint32_t kind = I.kind;
                    if (B.small_tris && !ra.nan && !ra.inf && ra.ymin >= 0.0f && ra.ymax - ra.ymin <= (float)SMALL_ROWS &&
                        (hr = pixel_rect(ra, I.width, I.height, rect))) {
                        const uint32_t cols = ((rect[0] & 0xFFFFu) >> twl << twl) |
                                              ((((rect[1] & 0xFFFFu) >> twl) + 1) << twl << 16);
                        SmallTri st;
                        if (small_tri(v[0], v[1], v[2], I.width, I.height, cols, st)) {
                            kind |= KIND_COUNTED;
                            frags = st.frags;
                            zmax = st.zmax;
                            empty = st.frags == 0 && st.err == 0;
                            if (st.err) atomicOr(B.err, st.err);
                        }
                    }
                    write_scr(&B.scr[g], v[0], v[1], v[2], di, kind);
                }
            } else {
                // Clipped
                CV poly[CLIP_MAX], tmp[CLIP_MAX];
                for (int k = 0; k < 3; ++k) {
                    for (int c = 0; c < 4; ++c) poly[k].p[c] = p[k][c];
                    fetch_attr(I.kind, I.attr, I.attr_stride, ix[k], poly[k].a);
                    poly[k].oc = oc[k];
                }
                const int n = clip_polygon(poly, 3, tmp);
                if (n < 0) atomicOr(B.err, ERRB_CLIP);
                if (n >= 3) {
                    const bool persp = kind_persp(I.kind);
                    // screen vertices in registers, two passes over the fan
                    // (recomputed, same bits), rather than a per-lane array
                    // in scratch memory
                    float s0v[6], sa[6], sb[6];
                    to_screen(poly[0], D->vp, persp, s0v);
                    // fan [p, e0, e1] over rest.windows(2) (clip.rs:373-396)
                    uint32_t keep = 0, cnt = 0;
                    to_screen(poly[1], D->vp, persp, sa);
                    for (int k = 1; k + 1 < n; ++k) {
                        to_screen(poly[k + 1], D->vp, persp, sb);
                        if (!culled(I.face_cull, backface(s0v, sa, sb))) {
                            keep |= 1u << k;
                            ++cnt;
                        }
                        for (int c = 0; c < 6; ++c) sa[c] = sb[c];
                    }
                    if (cnt > 1) {
                        extra_base = atomicAdd(B.extra_count, cnt - 1);
                        if (extra_base + cnt - 1 > B.extra_cap) {
                            atomicOr(B.err, ERRB_EXTRA);
                            cnt = 0;
                        }
                    }
                    uint32_t j = 0;
                    to_screen(poly[1], D->vp, persp, sa);
                    for (int k = 1; k + 1 < n && j < cnt; ++k) {
                        to_screen(poly[k + 1], D->vp, persp, sb);
                        if (keep & (1u << k)) {
                            ScrTri* dst = (j == 0) ? &B.scr[g] : &B.extra[extra_base + j - 1];
                            write_scr(dst, s0v, sa, sb, di, I.kind);
                            ra.add(s0v);
                            ra.add(sa);
                            ra.add(sb);
                            ++j;
                        }
                        for (int c = 0; c < 6; ++c) sa[c] = sb[c];
                    }
                    nf = cnt;
                }
            }
            if (nf > 0) {
                if (ra.inf) {
                    // an infinite screen coordinate: the reference walks up
                    // to 2^32 scanlines for it; reported instead
                    atomicOr(B.err, ERRB_NONFINITE);
                    nf = 0;
                } else if (ra.ymin < -(float)FOLD_ROWS_MAX) {
                    // rows above the target fold onto row 0 through the
                    // saturating `self.y as usize` (raster.rs:106), each a
                    // span of its own; beyond this many the float row
                    // counter of the reference loses its halves
                    atomicOr(B.err, ERRB_NEGY);
                    nf = 0;
                } else {
                    // rows at or below the last one panic in the reference
                    // (target.rs:173-174); so does a span starting past the right edge
                    const float rr0 = floorf(ra.ymin + 0.5f), rr1 = floorf(ra.ymax + 0.5f);
                    if (rr1 > rr0 && (rr1 > (float)I.height || floorf(ra.xmin) > (float)I.width + 1.0f))
                        atomicOr(B.err, ERRB_BOUNDS);
                    has_rect = !empty && (hr || pixel_rect(ra, I.width, I.height, rect));
                }
            }
        }
    }
    if (valid) {
        B.hdr[g] = nf | (extra_base << 3);
        B.rect[2 * g] = has_rect ? rect[0] : 0xFFFFFFFFu;
        B.rect[2 * g + 1] = rect[1];
        if (B.small_tris) B.zmax[g] = zmax;
    }
    // the union of the rectangles
    const uint32_t u0 = wave_min_u16x2(has_rect ? rect[0] : ~0u), u1 = ~wave_min_u16x2(has_rect ? ~rect[1] : ~0u);
    if (B.small_tris) {
        // the group's bound, z through an order-preserving key with NaN above
        // all: one bound not known, and the group's is not (8 icosphere
        // frames: + 0.03 ms of 1.5 here, - 0.36 ms of 2.34 in the rasterizer)
        const uint32_t zb = f2u(zmax), key = has_rect ? (zb >> 31 ? ~zb : zb | 0x80000000u) : 0u;
        const uint32_t kmax = ~wave_min_u32(~key);
        GroupBound gb;
        gb.zmax = u2f(kmax >> 31 ? kmax & 0x7FFFFFFFu : ~kmax);
        gb.r0 = u0;
        gb.r1 = u1;
        gb.pad = 0;
        if (lane == 0) B.group_max[group] = gb;
    }
    // prims.o (render.rs:195; verts.o is 3 per primitive, derived in
    // scan_totals) and the small triangles' frags.i: one atomic each per wave
    // when the wave's triangles all belong to one frame, else one per lane,
    // into the group's partial counters
    {
        uint32_t fmin = 0, fmax = 0;
        if (uniform) {
            fmin = fmax = (uint32_t)__builtin_amdgcn_readfirstlane((int)I.frame);
        } else {
            fmin = wave_min_u32(nf > 0 ? frame : 0xFFFFFFFFu);
            fmax = ~wave_min_u32(nf > 0 ? ~frame : 0xFFFFFFFFu);
        }
        const uint32_t part = (group % PRIM_PARTS) * PRIM_PART_STRIDE;
        unsigned long long* c = B.prims_part + part;
        if (fmin == fmax) {
            c += (uint64_t)fmin * PRIM_PARTS * PRIM_PART_STRIDE;
            uint32_t tot, ftot;
            (void)wave_excl_scan(nf, &tot);
            (void)wave_excl_scan(frags, &ftot);  // at most 64 triangles x 32 rows x 16,384 columns
            if (lane == 0 && tot) atomicAdd(c, (unsigned long long)tot);
            if (lane == 0 && ftot) atomicAdd(c + 1, (unsigned long long)ftot);
        } else if (nf > 0) {
            c += (uint64_t)frame * PRIM_PARTS * PRIM_PART_STRIDE;
            atomicAdd(c, (unsigned long long)nf);
            if (frags) atomicAdd(c + 1, (unsigned long long)frags);
        }
    }
    // per-tile run counts
    // and the runs themselves, for k_bin
    const uint32_t multi = __ballot(has_rect && nf > 1u) ? RUNS_MULTI : 0u;
    auto put = [&](uint32_t k, uint32_t tile, unsigned long long mask, bool first) {
        if (lane < k) {
            atomicAdd(&B.run_count[run_slot(tile)], 1u);
            if (first && lane < PRE_RUNS) {
                B.tile_of[(uint64_t)group * PRE_RUNS + lane] = tile;
                B.mask_of[(uint64_t)group * PRE_RUNS + lane] = mask;
            }
        }
    };
    const uint32_t t0 = rect_tile(rect[0], twl, thl), t1 = rect_tile(rect[1], twl, thl);
    const uint32_t ut0 = rect_tile(u0, twl, thl), ut1 = rect_tile(u1, twl, thl);
    uint32_t n = 0;
    if (__ballot(has_rect) == 0ull) {
        // nothing to bin
    } else if (uniform && ((ut1 & 0xFFFFu) - (ut0 & 0xFFFFu) + 1) * ((ut1 >> 16) - (ut0 >> 16) + 1) <= (uint32_t)WAVE) {
        // the group's triangles lie together: ask of each tile of the union
        // who meets it, two comparisons a tile, rather than for the least next
        // tile of any lane, 30 instructions a tile met (8 icosphere frames: 353
        // of 1,770 VALU instructions a wave, 32-bit rectangles among them). A
        // wider union may hold few tiles that are met.
        const uint32_t base = (uint32_t)__builtin_amdgcn_readfirstlane((int)I.tile_base);
        const uint32_t ntx = (uint32_t)__builtin_amdgcn_readfirstlane((int)I.ntx);
        uint32_t my_tile = 0, my_lo = 0, my_hi = 0;
        for (uint32_t ty = ut0 >> 16; ty <= ut1 >> 16; ++ty) {
            const unsigned long long rows = __ballot(has_rect && t0 >> 16 <= ty && ty <= t1 >> 16);
            if (rows == 0ull) continue;
            for (uint32_t tx = ut0 & 0xFFFFu; tx <= (ut1 & 0xFFFFu); ++tx) {
                const unsigned long long m = rows & __ballot((t0 & 0xFFFFu) <= tx && tx <= (t1 & 0xFFFFu));
                if (m == 0ull) continue;
                const bool here = lane == n;
                my_tile = here ? base + ty * ntx + tx : my_tile;
                my_lo = here ? (uint32_t)m : my_lo;
                my_hi = here ? (uint32_t)(m >> 32) : my_hi;
                ++n;
            }
        }
        put(n, my_tile, my_lo | (unsigned long long)my_hi << 32, true);
    } else {
        n = for_each_tile(has_rect, t0, t1, I.tile_base, I.ntx, put);
    }
    if (lane == 0) B.n_runs[group] = n | multi;
}
#endif  // RF_RASTER_TU

__device__ __forceinline__ uint32_t find_frame_tile(const FrameDesc* f, uint32_t n, uint32_t t) {
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (f[mid].tile_base <= t) lo = mid; else hi = mid;
    }
    return lo;
}

// ---------------------------------------------------------------------------
// k_scan*: exclusive scan of the run counts over all tiles (the offsets of
// their run lists) and the lists of tiles the later kernels work through
// ---------------------------------------------------------------------------
// Launches are what a small frame waits for: up to SCAN_ONE tiles, one block
// does it all (k_scan: a 256 x 256 frame 11.9 -> 8.2 us); above, a block per
// 1024 tiles, the block totals, and their offsets added back (k_scan_local,
// k_scan_top, k_scan_add: 14 us at 16,320 tiles, where one block, two steps of
// 8 tiles a thread, took 47).
#ifndef RF_RASTER_TU
constexpr uint32_t SCAN_PER = 4;  // consecutive tiles a thread of k_scan takes
constexpr uint32_t SCAN_ONE = 1024 * SCAN_PER;

// Appends to a list: the place of each lane that wants one.
__device__ __forceinline__ uint32_t wave_append(uint32_t* count, bool want) {
    const unsigned long long m = __ballot(want);
    if (m == 0ull) return 0;
    const uint32_t first = (uint32_t)(__ffsll((long long)m) - 1);
    uint32_t at = 0;
    if (lane_id() == first) at = atomicAdd(count, (uint32_t)__popcll(m));
    at = (uint32_t)__builtin_amdgcn_readlane((int)at, (int)first);
    return at + (uint32_t)__popcll(m & ((1ull << lane_id()) - 1));
}

// A tile is heavy with 3 times the mean number of runs of the tiles with any,
// one of the heaviest with 12 times. The rasterizer takes these first, the
// heaviest before the others, so that no wave is left with one at the end (32
// mixed frames, in list order 7.2 ms, so 5.1).
struct HeavyMin {
    uint32_t heavy, heaviest;
    __device__ HeavyMin(uint32_t runs, uint32_t busy) {
        const unsigned long long r = runs, n = busy ? busy : 1u;
        heavy = (uint32_t)max(min(3ull * r / n, 0xFFFFFFFFull), (unsigned long long)WAVE);
        heaviest = (uint32_t)max(min(12ull * r / n, 0xFFFFFFFFull), (unsigned long long)WAVE);
    }
};

// Tile i's entries: n runs from off, `busy` tiles with runs before it. Called
// by whole waves (`in`: the lane has a tile); `c` counts the lists' entries
// (TileCount words).
__device__ __forceinline__ void place_tile(const BatchDesc& B, uint32_t* c, bool in, uint32_t i, uint32_t n, uint32_t off,
                                           uint32_t busy, uint32_t frame, const HeavyMin& h) {
    const uint32_t at = n ? busy : B.n_tiles - 1 - (i - busy);
    if (in) {
        B.run_off[i] = off;
        B.run_cursor[run_slot(i)] = off;
        B.tiles[at] = TileRec{i, frame, off, n};
    }
    const bool huge = in && n > HUGE_RUNS, is_long = in && n > LONG_RUNS && !huge;
    const bool top = in && n > h.heaviest, heavy = in && n > h.heavy && !top;
    uint32_t k = wave_append(c + TN_LONG, is_long);
    if (is_long) B.long_list[k] = at;
    k = wave_append(c + TN_HUGE, huge);
    if (huge) B.long_list[B.n_tiles - 1 - k] = at;
    k = wave_append(c + TN_HEAVIEST, top);
    if (top) B.heavy_list[k] = at;
    k = wave_append(c + TN_HEAVY, heavy);
    if (heavy) B.heavy_list[B.n_tiles - 1 - k] = at;
}

// Totals known: prims.o and the small triangles' frags.i of every frame from
// its partial counters (verts.o is 3 per primitive, render.rs:196), and the
// counters of the kernels that follow.
__device__ __forceinline__ void scan_totals(const BatchDesc& B, uint32_t runs, uint32_t busy, const HeavyMin& h) {
    for (uint32_t f = threadIdx.x; f < B.n_frames; f += blockDim.x) {
        unsigned long long p = 0, fr = 0;
        for (uint32_t k = 0; k < PRIM_PARTS; ++k) {
            const unsigned long long* c = &B.prims_part[((uint64_t)f * PRIM_PARTS + k) * PRIM_PART_STRIDE];
            p += c[0];
            fr += c[1];
        }
        B.stats[f].prims_o = p;
        B.stats[f].verts_o = 3ull * p;
        B.stats[f].frags_i = fr;
    }
    if (threadIdx.x == 0) {
        B.run_off[B.n_tiles] = runs;
        B.extra_count[RUNS_WORD] = runs;
        B.tile_counts[TN_BUSY] = busy;
        B.tile_counts[TN_HEAVY_MIN] = h.heavy;
        if (runs > B.runs_cap) atomicOr(B.err, ERRB_RUNS);
    }
}

__global__ __launch_bounds__(1024) void k_scan(BatchDesc B) {
    __shared__ uint32_t wave_tot[2][16];
    __shared__ uint32_t counts[TN_HEAVY_MIN];
    const uint32_t tid = threadIdx.x, w = tid / WAVE, i0 = tid * SCAN_PER;
    if (tid < TN_HEAVY_MIN) counts[tid] = 0;
    uint32_t n[SCAN_PER], v = 0, f = 0;
#pragma unroll
    for (uint32_t k = 0; k < SCAN_PER; ++k) {
        n[k] = i0 + k < B.n_tiles ? B.run_count[run_slot(i0 + k)] : 0u;
        v += n[k];
        f += n[k] ? 1u : 0u;
    }
    uint32_t frame = i0 < B.n_tiles ? find_frame_tile(B.frames, B.n_frames, i0) : 0u;
    uint32_t wt, wf, off = wave_excl_scan(v, &wt), busy = wave_excl_scan(f, &wf);
    if (lane_id() == 0) {
        wave_tot[0][w] = wt;
        wave_tot[1][w] = wf;
    }
    __syncthreads();
    uint32_t tot = 0, ftot = 0;
    for (uint32_t k = 0; k < 16; ++k) {
        if (k == w) {
            off += tot;
            busy += ftot;
        }
        tot += wave_tot[0][k];
        ftot += wave_tot[1][k];
    }
    const HeavyMin h(tot, ftot);
    for (uint32_t k = 0; k < SCAN_PER; ++k) {
        const uint32_t i = i0 + k;
        const bool in = i < B.n_tiles;
        while (in && frame + 1 < B.n_frames && B.frames[frame + 1].tile_base <= i) ++frame;
        place_tile(B, counts, in, i, n[k], off, busy, frame, h);
        off += n[k];
        busy += n[k] ? 1u : 0u;
    }
    __syncthreads();
    if (tid > TN_BUSY && tid < TN_HEAVY_MIN) B.tile_counts[tid] = counts[tid];
    scan_totals(B, tot, ftot, h);
}

__global__ __launch_bounds__(1024) void k_scan_local(BatchDesc B) {
    __shared__ uint32_t wave_tot[2][16];
    const uint32_t tid = threadIdx.x, lane = lane_id(), w = tid / WAVE;
    const uint32_t i = blockIdx.x * 1024 + tid;
    const uint32_t v = i < B.n_tiles ? B.run_count[run_slot(i)] : 0u;
    const uint32_t f = v != 0 ? 1u : 0u;
    uint32_t tot, ftot;
    const uint32_t ex = wave_excl_scan(v, &tot);
    const uint32_t fex = wave_excl_scan(f, &ftot);
    if (lane == 0) {
        wave_tot[0][w] = tot;
        wave_tot[1][w] = ftot;
    }
    __syncthreads();
    uint32_t off = 0, foff = 0;
    for (uint32_t k = 0; k < w; ++k) {
        off += wave_tot[0][k];
        foff += wave_tot[1][k];
    }
    if (i < B.n_tiles) {
        B.run_off[i] = off + ex;        // within the block until k_scan_add
        B.run_cursor[run_slot(i)] = foff + fex;
    }
    if (tid == 1023) {
        B.scan_blk[2 * blockIdx.x] = off + ex + v;
        B.scan_blk[2 * blockIdx.x + 1] = foff + fex + f;
    }
}

__global__ __launch_bounds__(1024) void k_scan_top(BatchDesc B) {
    __shared__ uint32_t wave_tot[2][16];
    __shared__ uint32_t carry[2];
    const uint32_t tid = threadIdx.x, lane = lane_id(), w = tid / WAVE;
    const uint32_t nb = (B.n_tiles + 1023) / 1024;
    if (tid < 2) carry[tid] = 0;
    __syncthreads();
    for (uint32_t base = 0; base < nb; base += 1024) {
        const uint32_t i = base + tid;
        const uint32_t v = i < nb ? B.scan_blk[2 * i] : 0u, f = i < nb ? B.scan_blk[2 * i + 1] : 0u;
        uint32_t tot, ftot;
        const uint32_t ex = wave_excl_scan(v, &tot);
        const uint32_t fex = wave_excl_scan(f, &ftot);
        if (lane == 0) {
            wave_tot[0][w] = tot;
            wave_tot[1][w] = ftot;
        }
        __syncthreads();
        uint32_t off = carry[0], foff = carry[1];
        for (uint32_t k = 0; k < w; ++k) {
            off += wave_tot[0][k];
            foff += wave_tot[1][k];
        }
        if (i < nb) {
            B.scan_blk[2 * i] = off + ex;
            B.scan_blk[2 * i + 1] = foff + fex;
        }
        __syncthreads();
        if (tid < 2)
            for (uint32_t k = 0; k < 16; ++k) carry[tid] += wave_tot[tid][k];
        __syncthreads();
    }
    scan_totals(B, carry[0], carry[1], HeavyMin(carry[0], carry[1]));
}

__global__ __launch_bounds__(1024) void k_scan_add(BatchDesc B) {
    const uint32_t i = blockIdx.x * 1024 + threadIdx.x;
    const bool in = i < B.n_tiles;
    const uint32_t off = (in ? B.run_off[i] : 0u) + B.scan_blk[2 * blockIdx.x];
    const uint32_t busy = (in ? B.run_cursor[run_slot(i)] : 0u) + B.scan_blk[2 * blockIdx.x + 1];
    place_tile(B, B.tile_counts, in, i, in ? B.run_count[run_slot(i)] : 0u, off, busy, in ? find_frame_tile(B.frames, B.n_frames, i) : 0u,
               HeavyMin(B.run_off[B.n_tiles], B.tile_counts[TN_BUSY]));
}
#endif  // RF_RASTER_TU

constexpr uint32_t SORT_LDS = 4096;  // run lists up to this long sort in LDS, a block each

// Sorts the runs held one per lane (lanes >= n hold none) by group: a bitonic
// network over the 64 lanes; lane i ends with the i-th run. Groups are
// distinct within a tile.
__device__ __forceinline__ void wave_sort_runs(uint32_t n, uint32_t& group, unsigned long long& mask,
                                               uint32_t& multi) {
    const uint32_t lane = lane_id();
    const bool in = lane < n;
    const uint32_t g = in ? group : 0xFFFFFFFFu;
    const uint32_t nextg = __shfl_down(g, 1, WAVE);
    if (!__ballot(in && lane + 1 < n && g > nextg)) return;  // already in order
    unsigned long long kk = ((unsigned long long)g << 6) | lane;
    for (uint32_t ksz = 2; ksz <= (uint32_t)WAVE; ksz <<= 1) {
        for (uint32_t js = ksz >> 1; js > 0; js >>= 1) {
            const unsigned long long other = __shfl_xor(kk, js, WAVE);
            const bool take_min = ((lane & js) == 0) == ((lane & ksz) == 0);
            kk = take_min ? (other < kk ? other : kk) : (other > kk ? other : kk);
        }
    }
    mask = __shfl(mask, (uint32_t)(kk & 63u), WAVE);
    multi = __shfl(multi, (uint32_t)(kk & 63u), WAVE);
    group = (uint32_t)(kk >> 6);
}

// Orders the runs of each tile with more than LONG_RUNS of them by group
// (k_bin appends them in arrival order; the rasterizer sorts shorter lists
// itself, in registers). Each block takes huge lists (more than HUGE_RUNS)
// until none is left, then its waves take long ones: keys sort in LDS, and the
// records move once, through registers; lists beyond SORT_LDS sort in place in
// global memory. Bound by the longest lists: 32 mixed frames, whose lists
// exceed 1,024 runs, took 0.72 to 1.0 ms with a wave for every list and 1,024
// keys in LDS, and take 0.37.
#ifndef RF_RASTER_TU
// Sorts keys [0, n) in LDS by `threads` threads, tid among them: an
// all-ascending bitonic network. The first step of each merge compares i with
// i ^ (k - 1), later steps i with i ^ j; indices >= n act as +inf keys.
template <class Barrier>
__device__ __forceinline__ void bitonic_lds(unsigned long long* key, uint32_t n, uint32_t tid, uint32_t threads,
                                            Barrier&& barrier) {
    uint32_t p2 = 1;
    while (p2 < n) p2 <<= 1;
    for (uint32_t ksz = 2; ksz <= p2; ksz <<= 1) {
        for (uint32_t js = ksz >> 1; js > 0; js >>= 1) {
            const uint32_t x = (js == (ksz >> 1)) ? (ksz - 1) : js;
            // the q-th index with bit js clear, and its partner
            for (uint32_t q = tid; q < p2 / 2; q += threads) {
                const uint32_t i = ((q & ~(js - 1)) << 1) | (q & (js - 1)), l = i ^ x;
                if (l < n) {
                    const unsigned long long a = key[i], c = key[l];
                    if (a > c) {
                        key[i] = c;
                        key[l] = a;
                    }
                }
            }
            barrier();
        }
    }
}
// Orders a list of n <= threads * 16 runs: keys in LDS, then the records. (A
// list without room, n = 0, has no first record either.)
template <class Barrier>
__device__ __forceinline__ void sort_runs(rf_u32x4* runs, uint32_t n, unsigned long long* key, uint32_t tid,
                                          uint32_t threads, Barrier&& barrier) {
    static_assert(sizeof(Run) == sizeof(rf_u32x4) && offsetof(Run, group) == 0, "a run moves as one 16-byte access");
    if (n < 2) return;
    for (uint32_t i = tid; i < n; i += threads) key[i] = ((unsigned long long)runs[i][0] << 32) | i;
    barrier();
    bitonic_lds(key, n, tid, threads, barrier);
    rf_u32x4 mine[16];
#pragma unroll
    for (uint32_t k = 0; k < 16; ++k) {
        const uint32_t i = tid + threads * k;
        if (threads * k < n) mine[k] = runs[i < n ? (uint32_t)key[i] : 0u];
    }
    barrier();
#pragma unroll
    for (uint32_t k = 0; k < 16; ++k)
        if (tid + threads * k < n) runs[tid + threads * k] = mine[k];
}

__global__ __launch_bounds__(256) void k_binsort(BatchDesc B) {
    __shared__ unsigned long long key[SORT_LDS];
    __shared__ uint32_t s_next;
    static_assert(HUGE_RUNS * 4 <= SORT_LDS && HUGE_RUNS <= 16 * WAVE && SORT_LDS <= 16 * 256, "see sort_runs");
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / WAVE;
    const uint32_t n_huge = B.tile_counts[TN_HUGE], n_long = B.tile_counts[TN_LONG];
    // a block's (wave's) first list is the one of its number; more come by a counter
    auto runs_of = [&](uint32_t place, uint32_t& n) {
        const TileRec T = B.tiles[place];
        n = T.off >= B.runs_cap ? 0u : min(T.nruns, B.runs_cap - T.off);
        return B.runs + T.off;
    };
    for (uint32_t k = blockIdx.x; k < n_huge;) {
        uint32_t n;
        Run* const runs = runs_of(B.long_list[B.n_tiles - 1 - k], n);
        if (n <= SORT_LDS) {
            sort_runs(reinterpret_cast<rf_u32x4*>(runs), n, key, tid, 256u, [] { __syncthreads(); });
        } else {
            uint32_t p2 = 1;
            while (p2 < n) p2 <<= 1;
            for (uint32_t ksz = 2; ksz <= p2; ksz <<= 1) {
                for (uint32_t js = ksz >> 1; js > 0; js >>= 1) {
                    const uint32_t x = (js == (ksz >> 1)) ? (ksz - 1) : js;
                    for (uint32_t q = tid; q < p2 / 2; q += 256) {
                        const uint32_t i = ((q & ~(js - 1)) << 1) | (q & (js - 1)), l = i ^ x;
                        if (l < n) {
                            const Run a = runs[i], c = runs[l];
                            if (a.group > c.group) {
                                runs[i] = c;
                                runs[l] = a;
                            }
                        }
                    }
                    __threadfence_block();
                    __syncthreads();
                }
            }
        }
        if (tid == 0) s_next = gridDim.x + atomicAdd(&B.tile_counter[TC_HUGE * TC_STRIDE], 1u);
        __syncthreads();
        k = s_next;
        __syncthreads();
    }
    for (uint32_t k = blockIdx.x * 4 + wave; k < n_long;) {
        uint32_t n;
        Run* const runs = runs_of(B.long_list[k], n);
        // a wave's LDS accesses are performed in order
        sort_runs(reinterpret_cast<rf_u32x4*>(runs), n, key + wave * HUGE_RUNS, lane, (uint32_t)WAVE,
                  [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); });
        uint32_t c = 0;
        if (lane == 0) c = atomicAdd(&B.tile_counter[TC_LONG * TC_STRIDE], 1u);
        k = gridDim.x * 4 + (uint32_t)__builtin_amdgcn_readfirstlane((int)c);
    }
}
#endif  // RF_RASTER_TU

// ---------------------------------------------------------------------------
// k_raster
// ---------------------------------------------------------------------------
// 16-byte framebuffer stores. The rasterizer writes every target pixel once
// and never reads it back in the launch, so with RF_NT_STORE the stores are
// streaming (non-temporal): a gigabyte of colour and depth per launch then
// does not displace from L2 the triangles, runs and texels that other tiles
// still read.
#ifndef RF_NT_STORE
#define RF_NT_STORE 1
#endif
__device__ __forceinline__ void st16(void* p, uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
#if RF_NT_STORE
    __builtin_nontemporal_store(rf_u32x4{a, b, c, d}, (rf_u32x4*)p);
#else
    *(uint4*)p = make_uint4(a, b, c, d);
#endif
}
__device__ __forceinline__ void st16f(float* p, float a, float b, float c, float d) {
    st16(p, __float_as_uint(a), __float_as_uint(b), __float_as_uint(c), __float_as_uint(d));
}

__device__ __forceinline__ void store_pixel(const FrameDesc& F, uint32_t x, uint32_t y, uint32_t v) {
    uint8_t* p = F.color + (uint64_t)y * F.color_stride;
    if (F.fmt == PIX_RGB8) {
        p += 3ull * x;
        p[0] = (uint8_t)v;
        p[1] = (uint8_t)(v >> 8);
        p[2] = (uint8_t)(v >> 16);
        return;
    }
    if (F.fmt >= PIX_RGBA4444) {
        *(uint16_t*)(p + 2ull * x) = (uint16_t)v;
        return;
    }
    *(uint32_t*)(p + 4ull * x) = v;
}


#ifndef RF_VEC_INIT
#define RF_VEC_INIT 1  // tile init of a cleared frame with 16-byte LDS fills
#endif
#ifndef RF_EMPTY_GRAB
#define RF_EMPTY_GRAB 32
#endif
constexpr int EMPTY_GRAB = RF_EMPTY_GRAB;  // tiles without runs a wave takes at once

// The fused clear (Frame::clear) of one tile that nothing draws into: 16-byte
// stores where whole rows of 4-byte pixels are aligned.
template <int TW, int TILE_H>
__device__ __forceinline__ void clear_tile(const FrameDesc& F, uint32_t tile, uint32_t lane) {
    const bool has_depth = F.depth != nullptr;
    if (!F.clear_color && !(has_depth && F.clear_depth)) return;
    const uint32_t lt = tile - F.tile_base;
    const uint32_t x0 = (lt % F.ntx) * TW, y0 = (lt / F.ntx) * TILE_H;
    const uint32_t ncols = min((uint32_t)TW, F.width - x0), nrows = min((uint32_t)TILE_H, F.height - y0);
    const bool vec = ncols == (uint32_t)TW && pixfmt_bytes(F.fmt) == 4u && ((uintptr_t)F.color & 15u) == 0 &&
                     (F.color_stride & 15u) == 0 &&
                     (!has_depth || (((uintptr_t)F.depth & 15u) == 0 && (F.depth_stride & 3u) == 0));
    if (vec) {
        constexpr uint32_t QR = TW / 4;  // quads per row
        const uint32_t cp = F.clear_pixel;
        const float cz = F.clear_depth_value;
        for (uint32_t q = lane; q < nrows * QR; q += WAVE) {
            const uint32_t r = q / QR, c = (q - r * QR) * 4;
            if (F.clear_color)
                st16(F.color + (uint64_t)(y0 + r) * F.color_stride + 4ull * (x0 + c), cp, cp, cp, cp);
            if (has_depth && F.clear_depth) st16f(F.depth + (uint64_t)(y0 + r) * F.depth_stride + x0 + c, cz, cz, cz, cz);
        }
    } else {
        for (uint32_t i = lane; i < ncols * nrows; i += WAVE) {
            const uint32_t r = i / ncols, c = i - r * ncols;
            if (F.clear_color) store_pixel(F, x0 + c, y0 + r, F.clear_pixel);
            if (has_depth && F.clear_depth)
                F.depth[(uint64_t)(y0 + r) * F.depth_stride + x0 + c] = F.clear_depth_value;
        }
    }
}

// Writes the runs to their tiles' lists, in arrival order. Two groups a wave: a
// lane takes one of the runs k_setup has kept. A group of more than PRE_RUNS is
// walked again (walking every group, a wave each: 0.27 ms for 8 icospheres1080
// frames, 0.74 for 32 mixed ones).
#ifndef RF_RASTER_TU
__global__ __launch_bounds__(256) void k_bin(BatchDesc B) {
    static_assert(PRE_RUNS * 2 == WAVE, "two groups a wave");
    const uint32_t lane = lane_id();
    const uint32_t g0 = 2 * (blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE);
    if (g0 >= B.n_groups) return;
    auto put = [&](uint32_t group, uint32_t multi, uint32_t tile, unsigned long long mask) {
        const uint32_t pos = atomicAdd(&B.run_cursor[run_slot(tile)], 1u);
        if (pos < B.runs_cap) {
            Run r;
            r.group = group;
            r.multi = multi;
            r.mask = mask;
            B.runs[pos] = r;
        }
    };
    const uint32_t mine = g0 + lane / PRE_RUNS;
    const uint32_t c = mine < B.n_groups ? B.n_runs[mine] : 0u, n = c & ~RUNS_MULTI;
    if (n <= PRE_RUNS && lane % PRE_RUNS < n) {
        const uint64_t k = (uint64_t)mine * PRE_RUNS + lane % PRE_RUNS;
        put(mine, c / RUNS_MULTI, B.tile_of[k], B.mask_of[k]);
    }
    for (uint32_t h = 0; h < 2; ++h) {
        const uint32_t cg = (uint32_t)__builtin_amdgcn_readlane((int)c, (int)(h * PRE_RUNS));
        if ((cg & ~RUNS_MULTI) <= PRE_RUNS) continue;
        const uint32_t group = g0 + h;
        const uint64_t g = (uint64_t)group * WAVE + lane;
        bool valid = false;
        uint32_t r0 = 0, r1 = 0, base = 0, ntx = 0;
        if (g < B.n_tris) {
            r0 = B.rect[2 * g];
            r1 = B.rect[2 * g + 1];
            valid = r0 != 0xFFFFFFFFu;
            const uint32_t twl = (uint32_t)__builtin_ctz(B.tile_w), thl = (uint32_t)__builtin_ctz(B.tile_h);
            r0 = rect_tile(r0, twl, thl);
            r1 = rect_tile(r1, twl, thl);
            if (valid) {
                const uint32_t di = draw_of_tri(B.draws, B.n_draws, B.group_draw[group], g);
                const FrameDesc& F = B.frames[B.draws[di].frame];
                base = F.tile_base;
                ntx = F.ntx;
            }
        }
        for_each_tile(valid, r0, r1, base, ntx, [&](uint32_t k, uint32_t tile, unsigned long long mask, bool) {
            if (lane < k) put(group, cg / RUNS_MULTI, tile, mask);
        });
    }
}
#endif  // RF_RASTER_TU
// Per-triangle data of a batch slot (64 B).
struct SlotP {
    float dv[2][4];        // d(z, a0, a1, a2)/dx of the upper and lower trapezoid
    uint32_t kind_tag;     // shader kind | (draw - the tile's draw base) << 16
    uint32_t p0, p1, p2;   // flat: packed colour; textured: width, height, row stride (texels)
    uint32_t rec;          // the triangle's first edge record in the batch
    int32_t ysplit;        // first row of the lower trapezoid (absolute)
    uint32_t rxb;          // pixel columns of the binned tiles, first | end << 16 (margin check)
    int32_t ra;            // row of that record, relative to the tile's first row (negative:
                           // a row above the target, folded onto row 0)
};
// Edge record of one (triangle, tile row): the left and right edge state
// after the serial row steps of ScanlineIter::next (raster.rs:84-113).
struct EdgeRec {
    float lx, rx, lz, l0, l1, l2;
};

// The tile's queues of fans (rings): those of its runs in order, and of them
// those to draw (n_slot + 64 at most). A run adds at most 64 fans, or, where triangles have several,
// 16 triangles at a time, at most 112.
constexpr int FQ_CAP = 192;

#ifndef RF_CELL_W
#define RF_CELL_W 8
#endif
constexpr int CELL_W = RF_CELL_W;    // pixel columns per ordering cell
// Triangles and edge records per batch. LDS decides how many one-wave
// workgroups a CU holds (registers allow eight), so a tile's batch takes what
// its pixels leave of the smallest share that holds 128 records: 1/8 of the
// CU's 160 KB, else 1/6, 1/5, 1/4 or 1/3 (in the allocation's 1,280-byte
// steps). Tiles of 64 rows, whose triangles are taller, ask for 384 (and hold
// 448, 480 and, of the third that is the largest share, 320). Longer batches
// start fewer half-empty rounds: at 32 x 32 tiles, 8 icospheres1080 frames, 128
// records and 32 triangles 2.63 ms, 192 and 64 2.55, 256 and 32 2.35. (A batch's
// first triangle has at most th rows in a tile, unless rows above the target
// fold onto row 0.)
constexpr int REC_BYTES = 25;  // an EdgeRec and its owner
constexpr int LDS_THIRD = 53760;
__host__ __device__ constexpr int lds_fixed(int tw, int th, int slots) {
    return 9 * tw * (th + 1) + 4 * th * (tw / CELL_W) + 4 * (FQ_CAP + 64) + 4 * (slots + WAVE) + 64 * slots;
}
__host__ __device__ constexpr int n_slot(int tw, int th) {
    return tw * th <= 512 || th > 32 ? 64 : 32;
}
__host__ __device__ constexpr int rec_cap(int tw, int th) {
    const int f = lds_fixed(tw, th, n_slot(tw, th)), min = f + (th > 32 ? 384 : 128) * REC_BYTES;
    const int share = min <= 20480 ? 20480 : min <= 26880 ? 26880 : min <= 32000 ? 32000 : min <= 40960 ? 40960 : LDS_THIRD;
    const int r = (share - f) / REC_BYTES / 32 * 32;
    return r < 480 ? r : 480;
}
#ifndef RF_KMAX
#define RF_KMAX 600
#endif
#ifndef RF_JSER
#define RF_JSER 256
#endif
constexpr int KMAX = RF_KMAX;  // row steps taken serially; more use the exact fast-forward
constexpr int JSER = RF_JSER;  // pixel steps taken serially; more use the exact fast-forward
#ifndef RF_REFILL_MIN
#define RF_REFILL_MIN 16
#endif
#ifndef RF_HIDE_RUNS
#define RF_HIDE_RUNS 64
#endif
// Tiles of more runs than this pass over hidden triangles. Measured at 16, 64
// and 128 on 14 icosphere and mixed batches: 64 is never behind (10 frames of
// 1,291 icospheres: raster 621, 674, 720 us, but 13 frames of 80: 220, 209, 210).
constexpr int HIDE_RUNS = RF_HIDE_RUNS;
constexpr int REFILL_MIN = RF_REFILL_MIN;  // free lanes that trigger a refill while others still work

// Tile rasterizer. One wave owns one tile (TILE_H rows x TW columns) at a
// time; the tile's depth and each pixel's colour source live in LDS.
// Triangles (clip fans) are consumed in submission order in batches of up to
// 64:
//   setup  lane = triangle: tri_fill/scan setup (raster.rs:185-302);
//   edges  lane = triangle: walks its rows inside the tile with the serial
//          edge recurrence (ScanlineIter::next, raster.rs:84-113), entering
//          the tile through the exact fast-forward when it starts far above,
//          and writes one span record per row, in triangle-major order; a
//          record's index is its order key;
//   spans  lanes take records in key order and keep one until it is done:
//          the varyings are stepped serially pixel by pixel from the span's
//          start (Scanline::fragments, raster.rs:61-68; the exact
//          fast-forward enters a tile far from the start). In rounds, every
//          record claims the (row, 8-column) cells its remaining pixels touch
//          with an LDS atomic minimum of its key, and a record whose next 8
//          pixels lie in cells it holds applies them: depth test, depth write
//          and colour source (rasterize_fb, target.rs:163-198). A cell held by
//          a record blocks every later one, so each pixel sees its fragments
//          in submission order; the record with the smallest key always
//          proceeds.
// A passing fragment that writes colour leaves in the pixel's record what its
// colour is made of: the colour itself for the flat and Gouraud shaders, the
// draw (relative to the tile's first draw) and the sampled texel's index for
// the textured ones (the samplers' coordinate arithmetic runs here; only the
// texel fetch waits). The colour a pixel ends with is that of its last
// passing fragment, so the fetches run once per written pixel at the end of
// the tile, all pixels in parallel, and colour and depth go straight to the
// target.
constexpr uint8_t TAG_NONE = 0xFFu;   // no fragment wrote colour
constexpr uint8_t TAG_COLOR = 0xFEu;  // payload is the colour; else tag = index in the tile's draws, payload = texel
// Draws a tile's colour sources can name at a time. One byte a pixel for the
// tag: at two, a 64 x 32 tile's workgroup holds 29 KB and five fit a CU; at
// one, with 32 slots, 26.6 KB and six (32 crates1080 frames: 0.680 -> 0.621 ms).
constexpr int N_TAGS = 62;
constexpr uint32_t LINE_TAG = 0x8000u;   // SlotP::kind_tag bit of a line primitive
constexpr uint32_t COUNTED_TAG = 0x4000u;  // and of a triangle whose frags.i k_setup counted

__device__ __forceinline__ uint32_t texel_pixel(const BatchDesc& B, uint32_t fmt, uint32_t draw, uint32_t texel) {
    const uint32_t t = ((const uint32_t*)B.draws[draw].tex)[texel];
    return pack_pixel(fmt, t & 0xFF, (t >> 8) & 0xFF, (t >> 16) & 0xFF, t >> 24);
}

// n serial additions of d to each of k values, serially for small n and
// through the exact fast-forward otherwise (only the first nlive values).
template <int K>
__device__ __forceinline__ void advance(float (&v)[K], const float (&d)[K], uint32_t n, uint32_t nser, int nlive) {
    if (n <= nser) {
        uint32_t q = 0;
        for (; q + 4 <= n; q += 4) {  // four steps per trip: fewer loop branches
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < K; ++i) v[i] = v[i] + d[i];
        }
        for (; q < n; ++q) {
#pragma unroll
            for (int i = 0; i < K; ++i) v[i] = v[i] + d[i];
        }
    } else {
#pragma unroll
        for (int i = 0; i < K; ++i)
            if (i < nlive) v[i] = ff_add(v[i], d[i], n);
    }
}

__device__ __forceinline__ int32_t wave_incl_max_i32(int32_t v) {
    // v >= -1: order-preserving shift to unsigned
    const uint32_t x = wave_incl_scan((uint32_t)(v + 1), 0u, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
    return (int32_t)x - 1;
}

// The depth test of Context::depth_test (ctx.rs:86-89) without branches.
__device__ __forceinline__ bool depth_pass_u(int32_t dt, float nz, float cur) {
    return (dt == DT_NONE) | ((dt == DT_LESS) & (cur < nz)) | ((dt == DT_EQUAL) & (cur == nz)) |
           ((dt == DT_GREATER) & (cur > nz));
}

#ifdef RF_RASTER_TU
// TW: tile width (16, 32, 64); CH: pixels per lane applied together in a span
// round (6 or 8: short spans waste fewer lanes' slots and registers at 6,
// long spans take fewer rounds at 8).
// LINES: the launch draws edges. The others carry neither the lines' set-up nor
// the one-pixel copy of a round (8 icosphere frames: 1.97 ms as one instance for
// both, 2.02 with that copy in it, 1.92 apart).
template <int TW, int CH, int TH, bool LINES>
__global__ __launch_bounds__(64, 2) void k_raster(BatchDesc B) {
    constexpr int TILE_H = TH;  // tile rows
    constexpr int REC_CAP = rec_cap(TW, TH);
    constexpr int NSLOT = n_slot(TW, TH);
    constexpr int DQ_CAP = NSLOT + WAVE;
    static_assert(REC_CAP >= TILE_H, "a batch's first triangle fits");
    static_assert(lds_fixed(TW, TH, NSLOT) + REC_CAP * REC_BYTES <= LDS_THIRD, "three workgroups a CU at least");
    constexpr int LD = TILE_H + 1;  // padded column stride in LDS (bank spread)
    constexpr int NPX = TW * LD;
    constexpr int CW = CELL_W < TW ? CELL_W : TW;  // ordering cell width in this tile
    constexpr int NCG = TW / CW;
    // depth, then the payloads, in one array: a chunk's depth reads run up to
    // CH - 1 columns past the last one, into the payloads (values never
    // used), so that they are unconditional and pair up (ds_read2)
    __shared__ __align__(16) float s_px[2 * NPX];
    float* const s_dep = s_px;
    uint32_t* const s_pay = reinterpret_cast<uint32_t*>(s_px + NPX);  // the pixel's colour source: payload
    static_assert((CH - 1) * LD + TILE_H <= NPX, "depth over-reads stay in the array");
    __shared__ __align__(16) uint8_t s_tag[NPX];   //   and tag
    static_assert((NPX * 4) % 16 == 0 && NPX % 16 == 0, "16-byte LDS fills");
    __shared__ SlotP s_slot[NSLOT];
    __shared__ EdgeRec s_rec[REC_CAP];
    __shared__ uint32_t s_fq[FQ_CAP];  // g << 3 | fan
    __shared__ uint32_t s_dq[DQ_CAP];
    __shared__ uint32_t s_draws[N_TAGS];
    __shared__ int8_t s_own[REC_CAP];  // slot whose records start here, or -1
    __shared__ __align__(16) uint32_t s_cell[TILE_H * NCG];

    const uint32_t lane = lane_id();
    for (uint32_t i = lane; i < (uint32_t)(TILE_H * NCG); i += WAVE) s_cell[i] = 0xFFFFFFFFu;
    // Tiles come from the heavy list, then from TILE_PARTS contiguous
    // partitions of all tiles with runs, with a counter each. Workgroups are
    // dispatched round-robin over the XCDs, so a workgroup starts on partition
    // blockIdx.x % TILE_PARTS: neighbouring tiles (which share triangles) meet
    // in one XCD's L2. A wave takes one tile per atomic and moves on to the
    // next partition when its own is done.
    // (The lists' lengths are read again for each tile: kept, they take scalar
    // registers that spill.)
    // The tiles without runs, EMPTY_GRAB per atomic, at the waves' end: their
    // fused clear is the only write.
    auto clear_empties = [&]() {
        const uint32_t n_empty = B.n_tiles - B.tile_counts[TN_BUSY];
        uint32_t ecur_fi = 0xFFFFFFFFu;
        FrameDesc E;
        for (;;) {
            uint32_t e0 = 0;
            if (lane == 0) e0 = atomicAdd(&B.tile_counter[TC_EMPTY * TC_STRIDE], (uint32_t)EMPTY_GRAB);
            e0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)e0);
            if (e0 >= n_empty) break;
            const uint32_t ne = min((uint32_t)EMPTY_GRAB, n_empty - e0);
            uint32_t my_tile = 0, my_fi = 0;
            if (lane < ne) {
                const TileRec T = B.tiles[B.n_tiles - 1 - (e0 + lane)];
                my_tile = T.tile;
                my_fi = T.frame;
            }
            {
                // ne consecutive full tiles of one tile row of one frame (the
                // common case: the list is in tile order): clear the row
                // segment they make, each store instruction 1 KB of one pixel row
                const uint32_t t0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)my_tile);
                const uint32_t f0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)my_fi);
                const bool run = __ballot(lane < ne && (my_tile != t0 + lane || my_fi != f0)) == 0ull;
                if (run) {
                    if (f0 != ecur_fi) {
                        E = B.frames[f0];
                        ecur_fi = f0;
                    }
                    const uint32_t lt = t0 - E.tile_base, tx = lt % E.ntx, ty = lt / E.ntx;
                    const uint32_t x0 = tx * TW, y0 = ty * TILE_H;
                    const bool has_depth = E.depth != nullptr;
                    const bool ok = tx + ne <= E.ntx && x0 + ne * TW <= E.width && y0 + TILE_H <= E.height &&
                                    pixfmt_bytes(E.fmt) == 4u && ((uintptr_t)E.color & 15u) == 0 &&
                                    (E.color_stride & 15u) == 0 &&
                                    (!has_depth || (((uintptr_t)E.depth & 15u) == 0 && (E.depth_stride & 3u) == 0));
                    if (ok) {
                        if (E.clear_color || (has_depth && E.clear_depth)) {
                            const uint32_t qpr = ne * (TW / 4);  // 16-byte quads per pixel row
                            const uint32_t cp = E.clear_pixel;
                            const float cz = E.clear_depth_value;
                            for (uint32_t q = lane; q < TILE_H * qpr; q += WAVE) {
                                const uint32_t r = q / qpr, c = (q - r * qpr) * 4;
                                if (E.clear_color)
                                    st16(E.color + (uint64_t)(y0 + r) * E.color_stride + 4ull * (x0 + c), cp, cp, cp,
                                         cp);
                                if (has_depth && E.clear_depth)
                                    st16f(E.depth + (uint64_t)(y0 + r) * E.depth_stride + x0 + c, cz, cz, cz, cz);
                            }
                        }
                        continue;
                    }
                }
            }
            for (uint32_t j = 0; j < ne; ++j) {
                const uint32_t tile = (uint32_t)__builtin_amdgcn_readlane((int)my_tile, (int)j);
                const uint32_t fi = (uint32_t)__builtin_amdgcn_readlane((int)my_fi, (int)j);
                if (fi != ecur_fi) {
                    E = B.frames[fi];
                    ecur_fi = fi;
                }
                clear_tile<TW, TH>(E, tile, lane);
            }
        }
    };
    // The wave's next tile: its atomic is in flight while the tile before is
    // written back.
    uint32_t stage = 0;  // 0: the heavy list, else the partitions in turn from the wave's own
    uint32_t claim = 0;
    auto take = [&]() {
        const uint32_t part = (blockIdx.x + stage - 1) % TILE_PARTS;
        if (lane == 0) claim = atomicAdd(&B.tile_counter[(stage ? part : TC_HEAVY) * TC_STRIDE], 1u);
    };
    if (B.tile_counts[TN_HEAVIEST] + B.tile_counts[TN_HEAVY] == 0) stage = 1;
    take();
    for (;;) {
        TileRec T;
        bool got = false;
        while (!got && stage <= TILE_PARTS) {
            const uint32_t t0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)claim);
            if (stage == 0) {
                const uint32_t n_top = B.tile_counts[TN_HEAVIEST];
                if (t0 < n_top + B.tile_counts[TN_HEAVY]) {
                    T = B.tiles[B.heavy_list[t0 < n_top ? t0 : B.n_tiles - 1 - (t0 - n_top)]];
                    got = true;
                }
            } else {
                const uint32_t part = (blockIdx.x + stage - 1) % TILE_PARTS, n_busy = B.tile_counts[TN_BUSY];
                const uint32_t pb = (uint32_t)(((uint64_t)n_busy * part) / TILE_PARTS);
                const uint32_t pe = (uint32_t)(((uint64_t)n_busy * (part + 1)) / TILE_PARTS);
                if (t0 < pe - pb) {
                    T = B.tiles[pb + t0];
                    got = T.nruns <= B.tile_counts[TN_HEAVY_MIN];  // the heavy ones are drawn already
                    if (!got) {
                        take();
                        continue;
                    }
                }
            }
            if (!got && ++stage <= TILE_PARTS) take();
        }
        if (!got) break;
        const uint32_t tile = (uint32_t)__builtin_amdgcn_readfirstlane((int)T.tile);
        const uint32_t fi = (uint32_t)__builtin_amdgcn_readfirstlane((int)T.frame);
        const FrameDesc F = B.frames[fi];
        const uint32_t lt = tile - F.tile_base;
        const uint32_t tx = lt % F.ntx, ty = lt / F.ntx;
        const uint32_t x0 = tx * TW, y0 = ty * TILE_H;
        const uint32_t off = (uint32_t)__builtin_amdgcn_readfirstlane((int)T.off);
        uint32_t nruns = (uint32_t)__builtin_amdgcn_readfirstlane((int)T.nruns);
        if (off >= B.runs_cap) nruns = 0;
        else if (off + nruns > B.runs_cap) nruns = B.runs_cap - off;
        const bool has_depth = F.depth != nullptr;
        const bool dwrite = has_depth && F.depth_write;
        const int32_t dtest = has_depth ? F.depth_test : (int32_t)DT_NONE;
        const uint32_t ncols = min((uint32_t)TW, F.width - x0);
        const uint32_t nrows = min((uint32_t)TILE_H, F.height - y0);
        const uint32_t npx = ncols * nrows;

        // 16-byte stores: whole tile row of 4-byte pixels, 16-byte aligned rows
        const bool vec = ncols == (uint32_t)TW && pixfmt_bytes(F.fmt) == 4u && ((uintptr_t)F.color & 15u) == 0 &&
                         (F.color_stride & 15u) == 0 && (!has_depth || (((uintptr_t)F.depth & 15u) == 0 &&
                                                                         (F.depth_stride & 3u) == 0));
        if (nruns == 0) {  // no room for its runs: the launch is done again
            take();
            continue;
        }

        // tile init (WAVE / TILE_H lanes per row, each a share of the columns):
        // depth from the fused clear or the target; no fragment yet
        if (RF_VEC_INIT && (F.clear_depth || !has_depth)) {
            // constant fills of the whole arrays (padding and any part beyond
            // the target included, never written back), 16 bytes a store
            const float cd = F.clear_depth_value;
            if (has_depth)
                for (uint32_t i = lane; i < (uint32_t)NPX / 4; i += WAVE)
                    reinterpret_cast<float4*>(s_dep)[i] = make_float4(cd, cd, cd, cd);
            for (uint32_t i = lane; i < (uint32_t)NPX / 16; i += WAVE)
                reinterpret_cast<uint4*>(s_tag)[i] = make_uint4(0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu);
        } else {
            constexpr uint32_t LPR = WAVE / TILE_H;  // lanes per row
            const uint32_t r = lane % TILE_H, part = lane / TILE_H;
            if (r < nrows) {
                const float* drow = has_depth ? F.depth + (uint64_t)(y0 + r) * F.depth_stride + x0 : nullptr;
                for (uint32_t c = part; c < ncols; c += LPR) {
                    if (has_depth) s_dep[c * LD + r] = F.clear_depth ? F.clear_depth_value : drow[c];
                    s_tag[c * LD + r] = TAG_NONE;
                }
            }
        }
        __syncthreads();

        unsigned long long fi_acc = 0, fo_acc = 0;
        uint32_t errs = 0;
        uint32_t fq_head = 0, fq_tail = 0;  // ring indices (wave-uniform)
        uint32_t dq_head = 0, dq_tail = 0;
        // Triangles that cannot pass the depth test anywhere in the tile are
        // passed over (see below) once a batch has been drawn.
        const bool hide = B.small_tris && dtest == (int32_t)DT_LESS && nruns > (uint32_t)HIDE_RUNS;
        bool drawn = false;
        uint32_t head_skip = 0;             // rows of the head triangle already taken (wave-uniform)
        uint32_t n_tags = 0, last_draw = 0;  // draws in s_draws, and the last of them

        // The tile's runs in group order, 64 at a time, one per lane (one by one
        // each waited for a load of its own): lists of up to 64 are sorted here;
        // longer ones were sorted by k_binsort. `live`: those still to be queued.
        uint32_t lrun_g = 0, lrun_x = 0, next_run = 0;
        unsigned long long lrun_m = 0, live = 0;
        auto load_runs = [&]() {
            const uint32_t n = min(nruns - next_run, (uint32_t)WAVE);
            if (lane < n) {
                const Run r = B.runs[off + next_run + lane];
                lrun_g = r.group;
                lrun_m = r.mask;
                lrun_x = r.multi;
            }
            live = __ballot(lane < n);
            next_run += n;
        };
        if (nruns <= (uint32_t)WAVE) {
            load_runs();
            wave_sort_runs(nruns, lrun_g, lrun_m, lrun_x);
        }
        // Batches of up to 64 fans follow one another without a pause: once a
        // batch has handed out its last record, the next one is set up while
        // the items in flight finish (an item keeps in registers all it needs
        // of its slot and record). Order keys run on across the batches.
        uint32_t rquarter = 0;    // next 16 triangles of the run being queued, if they have several fans
        uint32_t next = 0;        // next record of the current batch to hand out
        uint32_t nrec = 0;        // records of the current batch
        uint32_t key_base = 0;    // order key of the current batch's first record
        int32_t carry = -1;       // slot of the last record handed out
        bool have = false;
        uint32_t key = 0, row = 0, ikind = 0, ip0 = 0, ip1 = 0, ip2 = 0, itag = 0;
        float dz = 0, d0 = 0, d1 = 0, d2 = 0, z = 0, c0 = 0, c1 = 0, c2 = 0;
        int32_t xs = 0, jc = 0, j1 = 0;
        for (;;) {
            if (next >= nrec) {
                // The least depth of each of 4 x 4 blocks of the tile, four lanes
                // a block. Depths under the Less test only grow, so items in
                // flight can only raise it: a triangle whose fragments' z is
                // nowhere above its blocks' least depth fails at every pixel.
                // 8 icospheres1080 frames: 6.66 -> 2.35 ms (42.9M of 285M
                // fragments pass); with whole groups tested first 1.98 ms, and
                // 32 mixed frames 4.39 -> 3.50.
                float bmin = 0.0f;
                const bool test = hide && drawn && (live != 0ull || next_run < nruns);
                if (test) {
                    constexpr uint32_t BW = TW / 4, BH = TILE_H / 4;
                    const uint32_t bx = (lane >> 2 & 3u) * BW, by = (lane >> 4) * BH;
                    bmin = __builtin_inff();
#pragma unroll 4
                    for (uint32_t i = 0; i < BW * BH / 4; ++i) {
                        const uint32_t c = bx + (i * 4 + (lane & 3u)) / BH, r = by + (i * 4 + (lane & 3u)) % BH;
                        const float d = s_dep[c * LD + r];
                        bmin = c < ncols && r < nrows ? fminf(bmin, d) : bmin;
                    }
                    bmin = fminf(bmin, u2f(dpp_u32<DPP_QUAD_1032>(f2u(bmin), f2u(bmin))));
                    bmin = fminf(bmin, u2f(dpp_u32<DPP_QUAD_2301>(f2u(bmin), f2u(bmin))));
                }
                // Whether something of z up to `z` in a pixel rectangle may pass.
                // A z of NaN is not known: it passes everywhere, also where no
                // fragment can (depth of +inf or NaN, whose least is +inf here),
                // for such triangles' fragments and spans are counted and
                // checked only where they are drawn.
                auto may_pass = [&](bool in, float z, uint32_t r0, uint32_t r1) {
                    constexpr uint32_t BWL = __builtin_ctz(TW / 4), BHL = __builtin_ctz(TILE_H / 4);
                    const uint32_t cx0 = max(r0 & 0xFFFFu, x0) - x0, cx1 = min(r1 & 0xFFFFu, x0 + TW - 1) - x0;
                    const uint32_t cy0 = max(r0 >> 16, y0) - y0, cy1 = min(r1 >> 16, y0 + TILE_H - 1) - y0;
                    const uint32_t xm = (2u << (cx1 >> BWL)) - (1u << (cx0 >> BWL));
                    const uint32_t ym = (16u << 4 * (cy1 >> BHL)) - (1u << 4 * (cy0 >> BHL));
                    const uint32_t blocks = in ? xm * 0x1111u & ym : 0u;
                    float m = __builtin_inff();
#pragma unroll 2
                    for (int k = 0; k < 16; ++k) {
                        const float bm = u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(bmin), 4 * k));
                        m = blocks >> k & 1u ? fminf(m, bm) : m;
                    }
                    return in && !(z <= m);
                };
                // queue fans until a full batch is to be drawn (or none are left)
                while (!hide || dq_tail - dq_head < (uint32_t)NSLOT) {
                    while (fq_tail - fq_head < (uint32_t)WAVE) {
                        if (live == 0ull) {
                            if (next_run >= nruns) break;
                            load_runs();
                            if (test) {
                                // whole groups first: most of a deep list
                                const bool in = (live >> lane) & 1ull;
                                GroupBound gb{};
                                if (in) gb = B.group_max[lrun_g];
                                live = __ballot(may_pass(in, gb.zmax, gb.r0, gb.r1));
                            }
                            continue;
                        }
                        const int j = __ffsll((long long)live) - 1;
                        const uint32_t group = (uint32_t)__builtin_amdgcn_readlane((int)lrun_g, j);
                        const uint32_t multi = (uint32_t)__builtin_amdgcn_readlane((int)lrun_x, j);
                        const unsigned long long mask =
                            (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)lrun_m, j) |
                            (unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(lrun_m >> 32), j) << 32;
                        const uint64_t g = (uint64_t)group * WAVE + lane;
                        bool has = (mask >> lane) & 1ull;
                        if (!multi) {
                            // one fan a triangle: its place is its rank in the mask
                            const uint32_t pre = (uint32_t)__popcll(mask & ((1ull << lane) - 1));
                            if (has) s_fq[(fq_tail + pre) % FQ_CAP] = (uint32_t)g << 3;
                            fq_tail += (uint32_t)__popcll(mask);
                            live &= live - 1;
                        } else {
                            has = has && lane / 16 == rquarter;
                            const uint32_t nf = has ? (B.hdr[g] & 7u) : 0u;
                            uint32_t tot;
                            const uint32_t pre = wave_excl_scan(nf, &tot);
                            for (uint32_t k = 0; k < nf; ++k) s_fq[(fq_tail + pre + k) % FQ_CAP] = ((uint32_t)g << 3) | k;
                            fq_tail += tot;
                            if (++rquarter == 4) {
                                live &= live - 1;
                                rquarter = 0;
                            }
                        }
                    }
                    __syncthreads();
                    const uint32_t nq = min(fq_tail - fq_head, (uint32_t)WAVE);
                    if (!hide || nq == 0) break;
                    bool take = lane < nq;
                    const uint32_t e = take ? s_fq[(fq_head + lane) % FQ_CAP] : 0u;
                    if (test) {
                        float z = 0.0f;
                        uint32_t r0 = 0, r1 = 0;
                        if (take) {
                            const uint64_t gg = e >> 3;
                            z = B.zmax[gg];
                            r0 = B.rect[2 * gg];
                            r1 = B.rect[2 * gg + 1];
                        }
                        take = may_pass(take, z, r0, r1);
                    }
                    const unsigned long long tm = __ballot(take);
                    if (take) s_dq[(dq_tail + __popcll(tm & ((1ull << lane) - 1))) % DQ_CAP] = e;
                    dq_tail += __popcll(tm);
                    fq_head += nq;
                    __syncthreads();
                }
                drawn = true;
                const uint32_t avail = hide ? dq_tail - dq_head : fq_tail - fq_head;
                if (avail == 0) {
                    if (__ballot(have) == 0ull) break;  // the tile is done
                    goto rounds;
                }
                const uint32_t nb = avail < (uint32_t)NSLOT ? avail : (uint32_t)NSLOT;
                // ---- setup: lane = triangle
                const bool act = lane < nb;
                Slot S;
                uint32_t rows_in = 0, di = 0, kind = 0;
                int32_t ra = 0, rb = 0;
                uint32_t rx0b = 0, rx1b = 0;
                int na = 0;
                // a line (KIND_LINE): one record per pixel of its walk that lies in
                // the tile's columns (wide) or rows (tall), from step lka on
                bool is_line = false, lwide = false, counted = false;
                uint32_t lS = 0, lka = 0;
                float lbase = 0.0f, lstep = 0.0f, lz = 0.0f, la0 = 0.0f, la1 = 0.0f, la2 = 0.0f;
                if (act) {
                    const uint32_t e = hide ? s_dq[(dq_head + lane) % DQ_CAP] : s_fq[(fq_head + lane) % FQ_CAP];
                    const uint64_t gg = e >> 3;
                    const uint32_t j = e & 7u;
                    const ScrTri* st = (j == 0) ? &B.scr[gg] : &B.extra[(B.hdr[gg] >> 3) + j - 1];
                    float va[6], vb[6], vc[6];
#pragma unroll
                    for (int c = 0; c < 6; ++c) {
                        va[c] = st->v[0][c];
                        vb[c] = st->v[1][c];
                        vc[c] = st->v[2][c];
                    }
                    di = st->draw;
                    kind = st->kind & 0xFFu;
                    is_line = LINES && (st->kind & KIND_LINE) != 0u;
                    counted = (st->kind & KIND_COUNTED) != 0u;
                    na = kind_attrs(kind);
                    if (is_line) {
                        lS = f2u(vb[0]);
                        const uint32_t ln = f2u(vb[1]);
                        lbase = vb[2];
                        lstep = vb[3];
                        lwide = f2u(vb[4]) != 0u;
                        lz = va[2];
                        la0 = va[3];
                        la1 = va[4];
                        la2 = va[5];
                        const uint32_t lo = lwide ? x0 : y0, hi = lo + (lwide ? ncols : nrows);
                        lka = lo > lS ? lo - lS : 0u;
                        const uint32_t kend = hi > lS ? min(ln, hi - lS) : 0u;
                        rows_in = kend > lka ? kend - lka : 0u;
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            S.t[h].n = 0;
                            S.t[h].dvz = 0.0f;
                            for (int c = 0; c < 3; ++c) S.t[h].dva[c] = 0.0f;
                        }
                    } else {
                        tri_setup(S, va, vb, vc, na);
                        const uint32_t rr0 = B.rect[2 * gg], rr1 = B.rect[2 * gg + 1];
                        rx0b = (rr0 & 0xFFFFu) / TW * TW;
                        rx1b = ((rr1 & 0xFFFFu) / TW + 1) * TW;
                        // rows of the triangle in this tile; in the first tile
                        // row, the rows above the target too: `self.y as
                        // usize` folds each onto row 0 as a span of its own
                        // (raster.rs:106), in row order before row 0's own
                        ra = S.ylo - (int32_t)y0;
                        rb = S.yhi - (int32_t)y0;
                        if (y0 > 0 || ra > 0) ra = ra < 0 ? 0 : ra;
                        rb = rb > (int32_t)nrows ? (int32_t)nrows : rb;
                        if (lane == 0) ra += (int32_t)head_skip;  // rows an earlier batch took
                        rows_in = rb > ra ? (uint32_t)(rb - ra) : 0u;
                    }
                }
                // A triangle with more rows here than a batch holds (only
                // with folded rows: otherwise at most TILE_H) goes in parts
                // of REC_CAP rows, as the sole triangle of its batches.
                const bool split = lane == 0 && rows_in > (uint32_t)REC_CAP;
                if (split) rows_in = REC_CAP;
                const bool head_split = __ballot(split) != 0ull;
                uint32_t rec_tot;
                const uint32_t rec_base = wave_excl_scan(rows_in, &rec_tot);
                // the draws' tags (draws only grow along the triangle order)
                const uint32_t prev = __shfl_up(di, 1, WAVE);
                const bool fresh = act && (lane == 0 ? n_tags == 0 || di != last_draw : di != prev);
                const unsigned long long fm = __ballot(fresh);
                uint32_t tag = n_tags + (uint32_t)__popcll(fm & ((2ull << lane) - 1)) - 1;
                const uint32_t tag0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)tag);
                if (tag0 >= (uint32_t)N_TAGS) {
                    // no tag left for the first triangle: pending texels are
                    // resolved to colours, and the tags start over
                    if (__ballot(have) != 0ull) goto rounds;  // after the items in flight, which use the old ones
                    for (uint32_t i = lane; i < npx; i += WAVE) {
                        const uint32_t r = i / ncols, c = i - r * ncols;
                        const uint32_t li = c * LD + r;
                        const uint32_t tg = s_tag[li];
                        if (tg < TAG_COLOR) {
                            s_pay[li] = texel_pixel(B, F.fmt, s_draws[tg], s_pay[li]);
                            s_tag[li] = TAG_COLOR;
                        }
                    }
                    __syncthreads();
                    tag -= tag0;
                }
                // take the leading triangles whose records and tags fit (lane
                // 0 always does: it has at most REC_CAP rows)
                const bool fits = rec_base + rows_in <= (uint32_t)REC_CAP && tag < (uint32_t)N_TAGS;
                const unsigned long long nf_mask = ~__ballot(act && fits && !head_split);
                const uint32_t nuse = head_split ? 1u
                                    : nf_mask == 0ull ? (uint32_t)WAVE : (uint32_t)(__ffsll((long long)nf_mask) - 1);
                const bool use = lane < nuse;
                const uint32_t nrec_new = __shfl(rec_base + rows_in, nuse - 1, WAVE);
                if (use && (fresh || lane == 0)) s_draws[tag] = di;
                n_tags = __shfl(tag, nuse - 1, WAVE) + 1;
                last_draw = __shfl(di, nuse - 1, WAVE);
                for (uint32_t i = lane; i < nrec_new; i += WAVE) s_own[i] = -1;
                __syncthreads();
                if (use) {
                    SlotP& P = s_slot[lane];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        P.dv[h][0] = S.t[h].dvz;
                        for (int c = 0; c < 3; ++c) P.dv[h][1 + c] = S.t[h].dva[c];
                    }
                    P.kind_tag = kind | (is_line ? LINE_TAG : 0u) | (counted ? COUNTED_TAG : 0u) | (tag << 16);
                    const DrawDesc& D = B.draws[di];
                    if (kind == KIND_FLAT) {
                        const uint32_t fc = D.flat_rgba;
                        P.p0 = pack_pixel(F.fmt, fc & 0xFF, (fc >> 8) & 0xFF, (fc >> 16) & 0xFF, fc >> 24);
                    } else {
                        P.p0 = D.tex_w;
                    }
                    P.p1 = D.tex_h;
                    P.p2 = D.tex_stride;
                    P.rec = rec_base;
                    P.ra = ra;
                    P.ysplit = S.t[0].n ? (int32_t)S.t[0].y0i + (int32_t)S.t[0].n : -0x7FFFFFFF;
                    P.rxb = rx0b | (rx1b << 16);
                    if (rows_in) s_own[rec_base] = (int8_t)lane;
                }
                // ---- edges: lane = triangle, walk its rows in the tile
                if (use && rows_in && is_line) {
                    // the line's pixels: the walked coordinate is the pixel
                    // index, the stepped one goes on serially (raster.rs:138-175)
                    float lv[1] = {lbase};
                    const float ld[1] = {lstep};
                    advance<1>(lv, ld, lka, KMAX, 1);
                    EdgeRec* out = &s_rec[rec_base];
                    for (uint32_t k = 0; k < rows_in; ++k) {
                        const float pix = (float)(lS + lka + k);
                        out[k] = lwide ? EdgeRec{pix, lv[0], lz, la0, la1, la2} : EdgeRec{lv[0], pix, lz, la0, la1, la2};
                        lv[0] = lv[0] + lstep;
                    }
                } else if (use && rows_in) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const Trap& T = S.t[h];
                        if (T.n == 0) continue;
                        const int32_t ty0 = (int32_t)T.y0i;  // absolute first row
                        const int32_t rend = ra + (int32_t)rows_in;  // rows recorded in this batch
                        int32_t a = ty0 > (int32_t)y0 + ra ? ty0 : (int32_t)y0 + ra;
                        int32_t b = ty0 + (int32_t)T.n;
                        if (b > (int32_t)y0 + rend) b = (int32_t)y0 + rend;
                        if (a >= b) continue;
                        float ev[6] = {T.lx, T.rx, T.lz, T.la[0], T.la[1], T.la[2]};
                        const float ed[6] = {T.dlx, T.drx, T.dlz, T.dla[0], T.dla[1], T.dla[2]};
                        advance<6>(ev, ed, (uint32_t)(a - ty0), KMAX, 3 + na);
                        EdgeRec* out = &s_rec[rec_base + (uint32_t)(a - (int32_t)y0 - ra)];
                        int32_t y = a;
                        for (; y + 2 <= b; y += 2, out += 2) {  // two rows per trip
                            out[0] = EdgeRec{ev[0], ev[1], ev[2], ev[3], ev[4], ev[5]};
#pragma unroll
                            for (int i = 0; i < 6; ++i) ev[i] = ev[i] + ed[i];
                            out[1] = EdgeRec{ev[0], ev[1], ev[2], ev[3], ev[4], ev[5]};
#pragma unroll
                            for (int i = 0; i < 6; ++i) ev[i] = ev[i] + ed[i];
                        }
                        if (y < b) *out = EdgeRec{ev[0], ev[1], ev[2], ev[3], ev[4], ev[5]};
                    }
                }
                __syncthreads();

                key_base += nrec;
                nrec = nrec_new;
                next = 0;
                carry = -1;
                if (head_split) {
                    head_skip += REC_CAP;  // the same triangle heads the next batch
                } else {
                    if (hide) dq_head += nuse;
                    else fq_head += nuse;
                    head_skip = 0;
                }
            }
        rounds:
            const unsigned long long need = __ballot(!have);
            if (next < nrec && (uint32_t)__popcll(need) >= (uint32_t)REFILL_MIN) {
                uint32_t cnt;
                const uint32_t rank = wave_excl_scan(have ? 0u : 1u, &cnt);
                const uint32_t k = next + rank;
                const bool valid = !have && k < nrec;
                int32_t f = wave_incl_max_i32(valid ? (int32_t)s_own[k] : -1);
                f = f > carry ? f : carry;
                f = f < 0 ? 0 : f;  // every valid record has a slot at or before it
                carry = __shfl(f, WAVE - 1, WAVE);  // the scan is non-decreasing
                next = next + cnt < nrec ? next + cnt : nrec;
                if (valid) {
                    const EdgeRec R = s_rec[k];
                    const SlotP& P = s_slot[f];
                    if (LINES && (P.kind_tag & LINE_TAG)) {
                        // a line pixel (Scanline x..x + 1 with the first end's
                        // single varying value); only the tile holding it draws it
                        const uint32_t px = cvt_u32(R.lx), py = cvt_u32(R.rx);
                        if (px >= x0 && px < x0 + ncols && py >= y0 && py < y0 + nrows) {
                            fi_acc += 1;
                            ikind = P.kind_tag & 0xFFu;
                            dz = d0 = d1 = d2 = 0.0f;
                            z = R.lz;
                            c0 = R.l0;
                            c1 = R.l1;
                            c2 = R.l2;
                            have = true;
                            key = key_base + k;
                            row = py - y0;
                            xs = (int32_t)px;
                            jc = 0;
                            j1 = 1;
                            ip0 = P.p0;
                            ip1 = P.p1;
                            ip2 = P.p2;
                            itag = P.kind_tag >> 16;
                        }
                    } else {
                    const int32_t r = P.ra + (int32_t)(k - P.rec);
                    const int32_t y = (int32_t)y0 + r;  // absolute row; negative: folded onto row 0
                    const uint32_t ty = y > 0 ? (uint32_t)y : 0u;
                    const int h = y < P.ysplit ? 0 : 1;
                    ikind = P.kind_tag & 0xFFu;
                    dz = P.dv[h][0];
                    d0 = P.dv[h][1];
                    d1 = P.dv[h][2];
                    d2 = P.dv[h][3];
                    // the span of this row (ScanlineIter::next, raster.rs:84-113)
                    const float rx0 = round_up_to_half(R.lx), rx1 = round_up_to_half(R.rx);
                    // v0.lerp(&v0.step(&dv_dx), x0 - v0.x)
                    const float tw_ = rx0 - R.lx;
                    float vv[4] = {R.lz + ((R.lz + dz) - R.lz) * tw_, R.l0 + ((R.l0 + d0) - R.l0) * tw_,
                                   R.l1 + ((R.l1 + d1) - R.l1) * tw_, R.l2 + ((R.l2 + d2) - R.l2) * tw_};
                    // 32-bit saturating casts: any value the 64-bit `as usize`
                    // keeps apart from these is beyond the target and fails
                    // the bounds check the same way
                    const uint32_t cnt_f = cvt_u32(rx1 - rx0);
                    const uint32_t xs32 = cvt_u32(rx0);
                    uint32_t xe = cvt_u32(rx1);
                    if (xe < xs32) xe = xs32;
                    int32_t jj0 = 0, jj1 = 0;
                    if (xe > F.width || ty >= F.height) {
                        errs |= ERRB_BOUNDS;
                    } else {
                        if (xe > xs32 && (xs32 < (P.rxb & 0xFFFFu) || xe > (P.rxb >> 16))) errs |= ERRB_MARGIN;
                        // frags.i: the part of [xs, xe) inside this tile
                        const uint32_t pa = xs32 > x0 ? xs32 : x0;
                        const uint32_t pb = xe < x0 + TW ? xe : x0 + TW;
                        if (pb > pa && !(P.kind_tag & COUNTED_TAG)) fi_acc += pb - pa;
                        const uint32_t nfrag = cnt_f < xe - xs32 ? cnt_f : xe - xs32;
                        xs = (int32_t)xs32;
                        jj0 = (int32_t)x0 - xs > 0 ? (int32_t)x0 - xs : 0;
                        jj1 = (int32_t)x0 + TW - xs;
                        if (jj1 > (int32_t)nfrag) jj1 = (int32_t)nfrag;
                    }
                    if (jj0 < jj1) {
                        const float dd[4] = {dz, d0, d1, d2};
                        // the fragment iterator stepped jj0 times (Scanline::fragments)
                        advance<4>(vv, dd, (uint32_t)jj0, JSER, 1 + kind_attrs(ikind));
                        z = vv[0];
                        c0 = vv[1];
                        c1 = vv[2];
                        c2 = vv[3];
                        have = true;
                        key = key_base + k;
                        row = ty - y0;
                        jc = jj0;
                        j1 = jj1;
                        ip0 = P.p0;
                        ip1 = P.p1;
                        ip2 = P.p2;
                        itag = P.kind_tag >> 16;
                    }
                    }
                }
            }
            const unsigned long long busy = __ballot(have);
            if (busy == 0ull) continue;
            // claim every cell of the remaining pixels
            int32_t cl0 = 0, cl1 = -1, cw1 = -1;
            // a lane without a record reads and frees row 0's cells: harmless
            const uint32_t crow = have ? row : 0u;
            if (have) {
                cl0 = (xs + jc - (int32_t)x0) / CW;
                cl1 = (xs + j1 - 1 - (int32_t)x0) / CW;
                const int32_t je = jc + CH < j1 ? jc + CH : j1;
                cw1 = (xs + je - 1 - (int32_t)x0) / CW;
#pragma unroll
                for (int32_t c = 0; c < NCG; ++c)
                    if (c >= cl0 && c <= cl1) atomicMin(&s_cell[row * NCG + c], key);
            }
            // the row's cells in one (vector) read, after every lane's claims
            uint32_t cells[NCG];
            if constexpr (NCG % 4 == 0) {
#pragma unroll
                for (int32_t c = 0; c < NCG; c += 4) {
                    const uint4 q = *reinterpret_cast<const uint4*>(&s_cell[crow * NCG + c]);
                    cells[c] = q.x;
                    cells[c + 1] = q.y;
                    cells[c + 2] = q.z;
                    cells[c + 3] = q.w;
                }
            } else {
#pragma unroll
                for (int32_t c = 0; c < NCG; ++c) cells[c] = s_cell[crow * NCG + c];
            }
            bool win = have;
#pragma unroll
            for (int32_t c = 0; c < NCG; ++c)
                if (c >= cl0 && c <= cw1) win = win && cells[c] == key;
            // the next N pixels of the winners' records
            auto apply = [&](auto n_px) {
                constexpr int N = decltype(n_px)::value;
                const int32_t rem = j1 - jc;
                const uint32_t li = (uint32_t)(xs + jc - (int32_t)x0) * LD + row;
                float zz[N], v0[N], v1[N], v2[N], cur[N];
                bool ps[N];
#pragma unroll
                for (int p = 0; p < N; ++p) {
                    zz[p] = z;
                    v0[p] = c0;
                    v1[p] = c1;
                    v2[p] = c2;
                    z = z + dz;
                    c0 = c0 + d0;
                    c1 = c1 + d1;
                    c2 = c2 + d2;
                }
                // the pixels of one chunk are distinct: read all depths first
                if (has_depth) {
#pragma unroll
                    for (int p = 0; p < N; ++p) cur[p] = s_px[li + p * LD];  // p >= rem: unused
                } else {
#pragma unroll
                    for (int p = 0; p < N; ++p) cur[p] = 0.0f;
                }
                uint32_t npass = 0;
#pragma unroll
                for (int p = 0; p < N; ++p) {
                    ps[p] = (p < rem) & depth_pass_u(dtest, zz[p], cur[p]);
                    npass += ps[p] ? 1u : 0u;
                }
                if (ikind == KIND_TEX_ONCE) {
                    // the shader runs for every passing fragment, colour write or not
                    const float tw = (float)ip0, th = (float)ip1;
#pragma unroll
                    for (int p = 0; p < N; ++p)
                        if (ps[p] && (cvt_u32(tw * (v0[p] / zz[p])) >= ip0 || cvt_u32(th * (v1[p] / zz[p])) >= ip1))
                            errs |= ERRB_TEXEL;
                }
                if (F.color_write) {
                    fo_acc += npass;
                    // colour sources of the chunk's pixels (the shader kind is
                    // decided once per chunk)
                    uint32_t pay[N];
                    uint32_t tg;
                    if (ikind == KIND_FLAT) {
                        tg = TAG_COLOR;
#pragma unroll
                        for (int p = 0; p < N; ++p) pay[p] = ip0;
                    } else if (ikind == KIND_GOURAUD) {  // Color3f::to_color4 (color.rs:253-263)
                        tg = TAG_COLOR;
#pragma unroll
                        for (int p = 0; p < N; ++p)
                            pay[p] = pack_pixel(F.fmt, cvt_u8(256.0f * v0[p]), cvt_u8(256.0f * v1[p]),
                                                cvt_u8(256.0f * v2[p]), 0xFF);
                    } else {
                        tg = itag;
                        const float tw = (float)ip0, th = (float)ip1;
                        if (ikind == KIND_TEX_CLAMP) {  // SamplerClamp (tex.rs:280-303)
                            const float mu = tw - 1.0f, mv = th - 1.0f;
#pragma unroll
                            for (int p = 0; p < N; ++p) {
                                // Scanline::fragments z_div (raster.rs:61-68, vec.rs:666-676)
                                float su = (v0[p] / zz[p]) * tw, sv = (v1[p] / zz[p]) * th;
                                su = su < 0.0f ? 0.0f : su;
                                su = su > mu ? mu : su;
                                sv = sv < 0.0f ? 0.0f : sv;
                                sv = sv > mv ? mv : sv;
                                pay[p] = cvt_u32(floorf(sv)) * ip2 + cvt_u32(floorf(su));
                            }
                        } else if (ikind == KIND_TEX_REPEAT_POT) {  // SamplerRepeatPot (tex.rs:240-266)
#pragma unroll
                            for (int p = 0; p < N; ++p) {
                                const uint32_t ui = (uint32_t)cvt_i32(floorf(tw * (v0[p] / zz[p]))) & (ip0 - 1);
                                const uint32_t vi = (uint32_t)cvt_i32(floorf(th * (v1[p] / zz[p]))) & (ip1 - 1);
                                pay[p] = vi * ip2 + ui;
                            }
                        } else {  // SamplerOnce (tex.rs:343-357): `as u32`, no wrap
#pragma unroll
                            for (int p = 0; p < N; ++p) {
                                const uint32_t ui = cvt_u32(tw * (v0[p] / zz[p]));
                                const uint32_t vi = cvt_u32(th * (v1[p] / zz[p]));
                                // outside the texture the reference panics (checked
                                // below); never fetch there
                                pay[p] = (ui < ip0 && vi < ip1) ? vi * ip2 + ui : 0u;
                            }
                        }
                    }
#pragma unroll
                    for (int p = 0; p < N; ++p) {
                        if (ps[p]) {
                            s_tag[li + p * LD] = (uint8_t)tg;
                            s_pay[li + p * LD] = pay[p];
                        }
                    }
                }
                if (dwrite) {
#pragma unroll
                    for (int p = 0; p < N; ++p)
                        if (ps[p]) s_dep[li + p * LD] = zz[p];
                }
                jc += N;
                if (jc >= j1) have = false;
            };
            // lines' records are single pixels: rounds of them alone apply no
            // more (8 frames of 500 crates' edges over their fill: 0.264 ->
            // 0.225 ms; at two pixels 0.240)
            if (LINES && __ballot(win && j1 - jc > 1) == 0ull) {
                if (win) apply(std::integral_constant<int, 1>{});
            } else if (win) {
                apply(std::integral_constant<int, CH>{});
            }
            // release the claims: every lane frees its whole row (one vector
            // write). Every claimed cell lies in a claimant's row, so all
            // cells are free again, as each round needs them at its start.
#pragma unroll
            for (int32_t c = 0; c < NCG; ++c) s_cell[crow * NCG + c] = 0xFFFFFFFFu;
                }
        __syncthreads();

        take();
        // write-back: fetch the texels, colour and depth to the target
        if (vec && (F.clear_color || F.color_write)) {
            // four pixels per lane; every load of a quad is issued before use
            constexpr uint32_t QR = TW / 4;
            for (uint32_t q = lane; q < nrows * QR; q += WAVE) {
                const uint32_t r = q / QR, c = (q - r * QR) * 4;
                uint8_t* crow = F.color + (uint64_t)(y0 + r) * F.color_stride + 4ull * (x0 + c);
                uint32_t tg[4], py[4], px[4];
                const uint32_t* tp[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    tg[k] = s_tag[(c + k) * LD + r];
                    py[k] = s_pay[(c + k) * LD + r];
                }
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    tp[k] = tg[k] < TAG_COLOR ? (const uint32_t*)B.draws[s_draws[tg[k]]].tex : nullptr;
                uint4 old = make_uint4(0, 0, 0, 0);
                const bool keep = !F.clear_color && (tg[0] == TAG_NONE || tg[1] == TAG_NONE || tg[2] == TAG_NONE ||
                                                     tg[3] == TAG_NONE);
                if (keep) old = *(const uint4*)crow;
                const uint32_t oldk[4] = {old.x, old.y, old.z, old.w};
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    if (tg[k] == TAG_COLOR) {
                        px[k] = py[k];
                    } else if (tg[k] != TAG_NONE) {
                        const uint32_t t = tp[k][py[k]];
                        px[k] = pack_pixel(F.fmt, t & 0xFF, (t >> 8) & 0xFF, (t >> 16) & 0xFF, t >> 24);
                    } else {
                        px[k] = F.clear_color ? F.clear_pixel : oldk[k];
                    }
                }
                st16(crow, px[0], px[1], px[2], px[3]);
                if (has_depth)
                    st16f(F.depth + (uint64_t)(y0 + r) * F.depth_stride + x0 + c, s_dep[c * LD + r],
                          s_dep[(c + 1) * LD + r], s_dep[(c + 2) * LD + r], s_dep[(c + 3) * LD + r]);
            }
        } else {
            for (uint32_t i = lane; i < npx; i += WAVE) {
                const uint32_t r = i / ncols, c = i - r * ncols;
                const uint32_t li = c * LD + r;
                const uint32_t tg = s_tag[li];
                if (tg == TAG_COLOR) {
                    store_pixel(F, x0 + c, y0 + r, s_pay[li]);
                } else if (tg != TAG_NONE) {
                    store_pixel(F, x0 + c, y0 + r, texel_pixel(B, F.fmt, s_draws[tg], s_pay[li]));
                } else if (F.clear_color) {
                    store_pixel(F, x0 + c, y0 + r, F.clear_pixel);
                }
                if (has_depth) F.depth[(uint64_t)(y0 + r) * F.depth_stride + x0 + c] = s_dep[li];
            }
        }
        const unsigned long long fi_s = wave_sum_u64(fi_acc), fo_s = wave_sum_u64(fo_acc);
        if (lane == 0) {
            if (fi_s) atomicAdd(&B.stats[fi].frags_i, fi_s);
            if (fo_s) atomicAdd(&B.stats[fi].frags_o, fo_s);
        }
        uint32_t e = errs;
        for (int o = 32; o > 0; o >>= 1) e |= __shfl_xor(e, o, WAVE);
        if (lane == 0 && e) atomicOr(B.err, e);
        __syncthreads();
    }

    // Then the tiles without runs (waves that finish the busy tiles early
    // fill the tail with them).
    clear_empties();
}

// The rasterizer's instances: tile width {16, 32, 64} x span chunk {6, 8}
// x tile height {16, 32, 64}.
using RasterFn = void (*)(BatchDesc);
constexpr bool TU_LINES = RF_RASTER_TU != 0;
#define RF_K3(TW, CH) \
    {k_raster<TW, CH, 16, TU_LINES>, k_raster<TW, CH, 32, TU_LINES>, k_raster<TW, CH, 64, TU_LINES>}
static const RasterFn RASTER_FNS[3][2][3] = {
    {RF_K3(16, 6), RF_K3(16, 8)}, {RF_K3(32, 6), RF_K3(32, 8)}, {RF_K3(64, 6), RF_K3(64, 8)}};
#undef RF_K3
static int raster_index(uint32_t tw, uint32_t ch, uint32_t th, int* i, int* j, int* k) {
    *i = tw == 16 ? 0 : (tw == 32 ? 1 : 2);
    *j = ch == 6 ? 0 : 1;
    *k = th == 16 ? 0 : (th == 64 ? 2 : 1);
    return 0;
}

#if RF_RASTER_TU
#define RF_TU(name) name##_lines
#else
#define RF_TU(name) name##_tris
#endif
hipError_t RF_TU(launch_raster)(const BatchDesc& B, hipStream_t s, uint32_t raster_grid) {
    int i, j, k;
    raster_index(B.tile_w, B.chunk, B.tile_h, &i, &j, &k);
    hipLaunchKernelGGL(RASTER_FNS[i][j][k], dim3(raster_grid), dim3(64), 0, s, B);
    return hipGetLastError();
}

uint32_t RF_TU(raster_wg_per_cu)(uint32_t tile_w, uint32_t chunk, uint32_t tile_h) {
    // resident one-wave workgroups per CU of each instance (registers and
    // LDS decide), asked of the runtime once
    static int occ[3][2][3] = {};
    int i, j, k;
    raster_index(tile_w, chunk, tile_h, &i, &j, &k);
    int& n = occ[i][j][k];
    if (n == 0) {
        int v = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, RASTER_FNS[i][j][k], 64, 0) != hipSuccess || v <= 0)
            v = 4;
        n = v;
    }
    return (uint32_t)n;
}
#endif  // RF_RASTER_TU

#ifndef RF_RASTER_TU
// ---------------------------------------------------------------------------
// Depth sort (render.rs:180-183, 209-219), before to_screen and face culling:
//   k_fans        one thread per triangle: assembly and clipping as k_setup
//                 does, each resulting clip-space triangle (a clip fan, in
//                 the order clip_tris emits them) stored with its key:
//                 Render::depth, (a.z + b.z + c.z) / 3 (prim.rs:21-23), as a
//                 total_cmp order key, then the triangle and fan index, so
//                 equal depths keep submission order;
//   radix sort of (key, fan) pairs, the draw first in the key, so that each
//                 draw's fans are contiguous and in order (each render() call
//                 sorts its own primitives); where draw, depth and index exceed
//                 64 bits, a second, stable sort by draw;
//   k_fan_gather  vertex q of fan i of the sorted order becomes vertex slot
//                 3i' + q of its draw, i' its rank in the draw (screen
//                 vertices): the main pipeline then draws them as unclipped
//                 triangles, whose indices follow from their number.
// The sorted draws form a batch of their own (their original meshes); the
// gather writes into the main batch, whose descriptors of these draws hold
// the fan counts the planning run found.
// ---------------------------------------------------------------------------
// Fan f of the pass: its key, draw and clip-space vertices.
__device__ __forceinline__ void put_fan(const BatchDesc& B, const DrawDesc* D, uint32_t di, uint32_t f, const CV& a,
                                        const CV& b, const CV& c, uint64_t g, uint32_t j) {
    const float z = ((a.p[2] + b.p[2]) + c.p[2]) / 3.0f;
    uint32_t k = (uint32_t)total_key(z) ^ 0x80000000u;  // ascending total order as unsigned
    if (D->sort == 2) k = ~k;                           // back to front
    unsigned long long key = ((unsigned long long)k << B.fan_bits) | (g << 3) | j;
    if (B.fan_draw_keyed) key |= (unsigned long long)di << (32 + B.fan_bits);
    B.fan_keys[f] = key;
    B.fan_vals[f] = f;
    if (B.fan_draw) B.fan_draw[f] = di;
    float* o = B.fans + (uint64_t)f * FAN_FLOATS;
    const CV* v[3] = {&a, &b, &c};
    for (int q = 0; q < 3; ++q) {
        for (int e = 0; e < 4; ++e) o[7 * q + e] = v[q]->p[e];
        for (int e = 0; e < 3; ++e) o[7 * q + 4 + e] = v[q]->a[e];
    }
}

// Bound by the fan counter when every fan takes its index with an atomic of
// its own: atomics on one address serialise in L2 (640,000 triangles in 4
// draws: 6.71 ms, with one atomic a block 0.07). A block counts its fans first
// and takes one range of indices; the order of the indices is of no account,
// the sort keys are distinct. The per-draw counts, wanted by the planning run
// only, take one atomic a wave where the wave's triangles are of one draw.
__global__ __launch_bounds__(256) void k_fans(BatchDesc B) {
    __shared__ uint32_t s_tot[4], s_base;
    const uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t lane = lane_id(), wave = threadIdx.x / WAVE;
    uint32_t cnt = 0, di = 0;
    const DrawDesc* D = nullptr;
    CV poly[CLIP_MAX], tmp[CLIP_MAX];
    if (g < B.n_tris) {
        di = draw_of_tri(B.draws, B.n_draws, B.group_draw[g / WAVE], g);
        D = &B.draws[di];
        const uint64_t t = g - D->tri_base;
        if (B.any_cull && !B.draw_vis[di]) {
            // a draw the bounding-box test hid
        } else if (D->tris[3 * t] >= D->n_verts || D->tris[3 * t + 1] >= D->n_verts ||
                   D->tris[3 * t + 2] >= D->n_verts) {
            atomicOr(B.err, ERRB_INDEX);
        } else {
            uint32_t all_out = ~0u, any_out = 0;
            for (int k = 0; k < 3; ++k) {
                shade_vertex(D, D->tris[3 * t + k], poly[k]);
                all_out &= poly[k].oc;
                any_out |= poly[k].oc;
            }
            int n = 0;                                             // Hidden
            if (all_out == 0) n = any_out == 0 ? 3 : clip_polygon(poly, 3, tmp);  // Visible or Clipped
            if (n < 0) atomicOr(B.err, ERRB_CLIP);
            cnt = n >= 3 ? (uint32_t)(n - 2) : 0u;
        }
    }
    uint32_t tot;
    const uint32_t pre = wave_excl_scan(cnt, &tot);
    if (lane == 0) s_tot[wave] = tot;
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t all = s_tot[0] + s_tot[1] + s_tot[2] + s_tot[3];
        s_base = all ? atomicAdd(B.fan_count, all) : 0u;
    }
    __syncthreads();
    if (B.fan_cnt) {
        const uint32_t d0 = wave_min_u32(cnt ? di : 0xFFFFFFFFu), d1 = ~wave_min_u32(cnt ? ~di : 0xFFFFFFFFu);
        if (d0 == d1) {
            if (lane == 0) atomicAdd(&B.fan_cnt[d0], tot);
        } else if (cnt) {
            atomicAdd(&B.fan_cnt[di], cnt);
        }
    }
    uint32_t f = s_base + pre;
    for (uint32_t k = 0; k < wave; ++k) f += s_tot[k];
    if (cnt && f + cnt > B.fan_cap) {
        atomicOr(B.err, ERRB_EXTRA);
        return;
    }
    for (uint32_t k = 0; k < cnt; ++k) put_fan(B, D, di, f + k, poly[0], poly[k + 1], poly[k + 2], g, k);
}

// The second sort's keys: the draw of each fan in the first sort's order.
__global__ __launch_bounds__(256) void k_fan_draw_keys(const uint32_t* order, const uint32_t* fan_draw, uint32_t n,
                                                       uint32_t* keys) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) keys[i] = fan_draw[order[i]];
}

// Vertex q of fan i of the final order (of draw d: draws_of[i], else the fan's
// own where there are several) becomes vertex slot 3 rank + q of main draw
// map[2d + 1], rank = i - map[2d] (the draw's first position). A thread a
// vertex: the fans lie anywhere, and a thread that reads a fan's 84 bytes alone
// waits for them three times as long (290,000 fans: 0.112 ms).
__global__ __launch_bounds__(256) void k_fan_gather(BatchDesc P, BatchDesc M, const uint32_t* order,
                                                    const uint32_t* draws_of, const uint32_t* map, uint32_t n_fans) {
    const uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t i = (uint32_t)(v / 3), q = (uint32_t)(v - 3ull * i);
    if (i >= n_fans) return;
    const uint32_t f = order[i];
    const uint32_t d = P.n_draws < 2 ? 0u : draws_of ? draws_of[i] : P.fan_draw[f];
    const uint32_t rank = i - map[2 * d];
    const DrawDesc* D = &M.draws[map[2 * d + 1]];
    const float* src = P.fans + (uint64_t)f * FAN_FLOATS + 7 * q;
    CV c;
#pragma unroll
    for (int e = 0; e < 4; ++e) c.p[e] = src[e];
#pragma unroll
    for (int e = 0; e < 3; ++e) c.a[e] = src[4 + e];
    to_screen(c, D->vp, kind_persp(D->kind), M.sv + 6 * (D->vert_base + 3ull * rank + q));
}

// ---------------------------------------------------------------------------
// k_cull: one thread per draw. A draw that asks for it is skipped when its
// mesh's bounding box is Hidden: the 8 corners (BBox::verts, scene.rs:59-66)
// through the draw's ProjMat3 (scene.rs:81-87) and view_frustum::status
// (clip.rs:245-267) — all corners outside one same plane. What the skipped
// render() call would have counted is added to the frame's hidden totals.
// ---------------------------------------------------------------------------
// Bound by those totals when every hidden draw adds its own (4 frames of 1,000
// draws: 54 us): a wave whose hidden draws are of one frame adds once.
__global__ __launch_bounds__(256) void k_cull(BatchDesc B) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    bool hidden = false;
    uint32_t frame = 0;
    unsigned long long prims = 0, verts = 0;
    if (i < B.n_draws) {
        const DrawDesc* D = &B.draws[i];
        if (D->cull) {
            const float* m = D->mvp;
            uint32_t all_out = ~0u;
            for (int c = 0; c < 8; ++c) {
                const float px = D->bbox[(c & 4) ? 3 : 0], py = D->bbox[(c & 2) ? 4 : 1], pz = D->bbox[(c & 1) ? 5 : 2];
                const float x = dot4(m + 0, px, py, pz, 1.0f);
                const float y = dot4(m + 4, px, py, pz, 1.0f);
                const float z = dot4(m + 8, px, py, pz, 1.0f);
                const float w = dot4(m + 12, px, py, pz, 1.0f);
                all_out &= outcode(x, y, z, w);
            }
            if (all_out != 0) {
                hidden = true;
                frame = D->frame;
                // a depth-sorted draw holds its fans: its render() call's own counts
                prims = D->pre ? D->in_tris : D->n_tris;
                verts = D->pre ? D->in_verts : D->n_verts;
            }
        }
        B.draw_vis[i] = hidden ? 0u : 1u;
    }
    const uint32_t f0 = wave_min_u32(hidden ? frame : 0xFFFFFFFFu), f1 = ~wave_min_u32(hidden ? ~frame : 0xFFFFFFFFu);
    if (f0 == f1) {
        const uint32_t n = (uint32_t)__popcll(__ballot(hidden));
        prims = wave_sum_u64(prims);
        verts = wave_sum_u64(verts);
        if (lane_id() == 0) {
            FrameStats& st = B.stats[f0];
            atomicAdd(&st.hidden_draws, (unsigned long long)n);
            atomicAdd(&st.hidden_prims, prims);
            atomicAdd(&st.hidden_verts, verts);
        }
    } else if (hidden) {
        FrameStats& st = B.stats[frame];
        atomicAdd(&st.hidden_draws, 1ull);
        atomicAdd(&st.hidden_prims, prims);
        atomicAdd(&st.hidden_verts, verts);
    }
}

// Zeroes per-batch counters (a kernel, so it can live inside a captured graph).
__global__ void k_reset(BatchDesc B) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < B.n_tiles) B.run_count[run_slot(i)] = 0;
    // the draw of each group's first triangle
    if (i < B.n_groups) B.group_draw[i] = find_draw_tri(B.draws, B.n_draws, (uint64_t)i * WAVE);
    if (i < B.n_frames * PRIM_PARTS) {
        B.prims_part[(uint64_t)i * PRIM_PART_STRIDE] = 0;
        B.prims_part[(uint64_t)i * PRIM_PART_STRIDE + 1] = 0;
    }
    if (i < B.n_frames) {
        B.stats[i].prims_o = 0;
        B.stats[i].verts_o = 0;
        B.stats[i].frags_i = 0;
        B.stats[i].frags_o = 0;
        B.stats[i].hidden_draws = 0;
        B.stats[i].hidden_prims = 0;
        B.stats[i].hidden_verts = 0;
    }
    if (i == 0) {
        *B.extra_count = 0;
        *B.err = 0;
        if (B.fan_count) *B.fan_count = 0;
        for (uint32_t k = 0; k < N_TILE_COUNTERS; ++k) B.tile_counter[k * TC_STRIDE] = 0;
        for (uint32_t k = TN_BUSY; k <= TN_HEAVY_MIN; ++k) B.tile_counts[k] = 0;
    }
    if (B.fan_cnt && i < B.n_draws) B.fan_cnt[i] = 0;
}

// ---------------------------------------------------------------------------
// launch wrappers
// ---------------------------------------------------------------------------
static hipError_t launch_impl(const BatchDesc& B0, hipStream_t s, uint32_t raster_grid, hipEvent_t* ev) {
    BatchDesc B = B0;
    B.small_tris = B.n_tris > (uint64_t)RF_SMALL_TRIS * B.n_tiles;
    uint32_t reset_n = B.n_tiles > B.n_frames * PRIM_PARTS ? B.n_tiles : B.n_frames * PRIM_PARTS;
    reset_n = reset_n > B.n_groups ? reset_n : B.n_groups;
    auto mark = [&](int i) {
        if (ev) (void)hipEventRecord(ev[i], s);
    };
    hipError_t e = hipSuccess;
    auto chk = [&](hipError_t r) {
        if (r != hipSuccess && e == hipSuccess) e = r;
    };
    mark(0);
    hipLaunchKernelGGL(k_reset, dim3((reset_n + 255) / 256 + 1), dim3(256), 0, s, B);
    if (B.any_cull) hipLaunchKernelGGL(k_cull, dim3((B.n_draws + 255) / 256), dim3(256), 0, s, B);
    mark(1);
    if (B.n_groups) hipLaunchKernelGGL(k_setup, dim3((B.n_groups + 3) / 4), dim3(256), 0, s, B);
    mark(2);
    const uint32_t nb = (B.n_tiles + 1023) / 1024;
    if (B.n_tiles <= SCAN_ONE) {
        hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, s, B);
    } else {
        hipLaunchKernelGGL(k_scan_local, dim3(nb), dim3(1024), 0, s, B);
        hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, s, B);
        hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(1024), 0, s, B);
    }
    mark(3);
    if (B.n_groups) hipLaunchKernelGGL(k_bin, dim3((B.n_groups + 7) / 8), dim3(256), 0, s, B);
    mark(4);
    // no tile has more than 64 runs where there are no more groups
    if (B.n_groups > (uint32_t)WAVE)
        hipLaunchKernelGGL(k_binsort, dim3(B.n_tiles < 1024u ? B.n_tiles : 1024u), dim3(256), 0, s, B);
    mark(5);
    chk(hipGetLastError());
    chk(B.any_lines ? launch_raster_lines(B, s, raster_grid) : launch_raster_tris(B, s, raster_grid));
    mark(6);
    chk(hipGetLastError());
    return e;
}
hipError_t launch_fans(const BatchDesc& B, hipStream_t s) {
    if (B.n_tris && (!B.fans || !B.fan_keys || !B.fan_vals || !B.fan_count || !B.fan_cap)) return hipErrorInvalidValue;
    uint32_t reset_n = B.n_tiles > B.n_frames * PRIM_PARTS ? B.n_tiles : B.n_frames * PRIM_PARTS;
    reset_n = reset_n > B.n_groups ? reset_n : B.n_groups;
    reset_n = reset_n > B.n_draws ? reset_n : B.n_draws;
    hipLaunchKernelGGL(k_reset, dim3((reset_n + 255) / 256 + 1), dim3(256), 0, s, B);
    if (B.any_cull) hipLaunchKernelGGL(k_cull, dim3((B.n_draws + 255) / 256), dim3(256), 0, s, B);
    if (B.n_tris) hipLaunchKernelGGL(k_fans, dim3((uint32_t)((B.n_tris + 255) / 256)), dim3(256), 0, s, B);
    return hipGetLastError();
}
hipError_t launch_fan_draw_keys(const uint32_t* order, const uint32_t* fan_draw, uint32_t n, uint32_t* keys,
                                hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_fan_draw_keys, dim3((n + 255) / 256), dim3(256), 0, s, order, fan_draw, n, keys);
    return hipGetLastError();
}
hipError_t launch_fan_gather(const BatchDesc& P, const BatchDesc& M, const uint32_t* order, const uint32_t* draws_of,
                             const uint32_t* map, uint32_t n_fans, hipStream_t s) {
    if (n_fans && (!P.fans || !order || !map || !M.sv)) return hipErrorInvalidValue;
    if (n_fans)
        hipLaunchKernelGGL(k_fan_gather, dim3((uint32_t)((3ull * n_fans + 255) / 256)), dim3(256), 0, s, P, M, order, draws_of,
                           map, n_fans);
    return hipGetLastError();
}
hipError_t launch_pipeline(const BatchDesc& B, hipStream_t s, uint32_t raster_grid) {
    return launch_impl(B, s, raster_grid, nullptr);
}
hipError_t launch_pipeline_timed(const BatchDesc& B, hipStream_t s, uint32_t raster_grid, hipEvent_t* ev) {
    return launch_impl(B, s, raster_grid, ev);
}
#endif  // RF_RASTER_TU

}  // namespace rf
