// Device-side descriptors shared by the host runtime and the kernels.
//
// A *batch* is one or more frames; a frame is one render target, one context
// and an ordered list of draws; a draw is one `render()` call of the
// reference (core/src/render.rs:134-207): one mesh, one built-in shader kind,
// one uniform (the mvp matrix) and one `to_screen` matrix. Primitive
// submission order -- which decides depth-test ties -- is draw order, then
// triangle order within the draw, then clip-fan order (clip.rs:360-398).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace rf {

// The rasterizer's tiles are split into this many contiguous partitions, one
// per XCD (accelerator complex die, each with its own L2) of the MI355X.
constexpr uint32_t TILE_PARTS = 8;


// Shader kinds (the built-in vertex/fragment shader pairs).
enum ShaderKind : uint32_t {
    KIND_FLAT = 0,            // constant Color4, varying ()
    KIND_GOURAUD = 1,         // Color3f varying -> Color3f::to_color4
    KIND_TEX_CLAMP = 2,       // TexCoord varying (z-divided) -> SamplerClamp
    KIND_TEX_REPEAT_POT = 3,  // TexCoord varying (z-divided) -> SamplerRepeatPot
    KIND_TEX_ONCE = 4,        // TexCoord varying (z-divided) -> SamplerOnce
};
constexpr uint32_t KIND_LAST = KIND_TEX_ONCE;

// Primitive types of a draw (Render impls, prim.rs:11-60).
enum PrimType : uint32_t {
    PRIM_TRI = 0,   // Tri<usize>: index triples, tri_fill
    PRIM_EDGE = 1,  // Edge<usize>: index pairs, raster::line
};
// ScrTri::kind bit of a line (Edge) primitive: then v[0] is the line's first
// end (its z and varyings hold for every pixel) and v[1] its pixel walk
// (see k_setup).
constexpr uint32_t KIND_LINE = 0x100;
// ScrTri::kind bit of a triangle whose frags.i k_setup has counted (see
// small_tri): the rasterizer leaves it alone.
constexpr uint32_t KIND_COUNTED = 0x200;

__host__ __device__ inline int kind_attrs(uint32_t k) {
    return k == KIND_FLAT ? 0 : (k == KIND_GOURAUD ? 3 : 2);
}
__host__ __device__ inline bool kind_persp(uint32_t k) { return k >= KIND_TEX_CLAMP; }

// Colour buffer formats.
enum PixFmt : uint32_t {
    PIX_RGBA8 = 0,      // [u8; 4] r, g, b, a  (Buf2<Color4>, Rgba8888 bytes)
    PIX_RGB8 = 1,       // [u8; 3] r, g, b     (Buf2<Color3>)
    PIX_U32_RGBA = 2,   // u32 0xRRGGBBAA      (Rgba8888 into u32)
    PIX_U32_XRGB = 3,   // u32 0x00RRGGBB      (Xrgb8888)
    PIX_U32_ARGB = 4,   // u32 0xAARRGGBB      (Argb8888 into u32; Bgra8888 bytes)
    PIX_U32_BGRA = 5,   // u32 0xBBGGRRAA      (Bgra8888 into u32; Argb8888 bytes)
    PIX_RGBA4444 = 6,   // u16 rrrrggggbbbbaaaa (Rgba4444)
    PIX_RGB565 = 7,     // u16 rrrrrggggggbbbbb (Rgb565)
};
constexpr uint32_t PIX_LAST = PIX_RGB565;
__host__ __device__ inline uint32_t pixfmt_bytes(uint32_t fmt) {
    return fmt == PIX_RGB8 ? 3u : (fmt >= PIX_RGBA4444 ? 2u : 4u);
}

enum DepthTest : int32_t { DT_NONE = 0, DT_LESS = 1, DT_EQUAL = 2, DT_GREATER = 3 };
enum FaceCull : int32_t { FC_NONE = 0, FC_BACK = 1, FC_FRONT = 2 };

// Error bits raised by kernels (OR-ed into one device word per batch).
enum ErrBits : uint32_t {
    ERRB_INDEX = 1u << 0,      // a vertex index >= vertex count (prim.rs:17-19 panics)
    ERRB_BOUNDS = 1u << 1,     // a span outside the target (target.rs:173-174 panics)
    ERRB_MARGIN = 1u << 2,     // a span left the tiles its triangle was binned to
    ERRB_EXTRA = 1u << 3,      // clip-fan storage exhausted
    ERRB_RUNS = 1u << 4,       // bin-run storage exhausted
    ERRB_NONFINITE = 1u << 5,  // a screen-space vertex is NaN or infinite
    ERRB_NEGY = 1u << 6,       // a screen-space vertex lies above row -0.5
    ERRB_CLIP = 1u << 7,       // clipping produced more than 9 vertices
    ERRB_TEXEL = 1u << 8,      // SamplerOnce indexed outside the texture (buf.rs:731-733 panics)
};

struct DrawDesc {
    const float* pos;       // n_verts x (x, y, z)
    const float* attr;      // n_verts x kind_attrs(kind)
    const uint32_t* tris;   // n_tris x (i0, i1, i2), or x (i0, i1) for edges; a pre draw's are 3t, 3t + 1, 3t + 2
    const uint8_t* tex;     // Color4 texels (textured kinds)
    uint32_t n_verts, n_tris;
    uint32_t kind, frame;
    uint32_t tex_w, tex_h, tex_stride;  // stride in texels
    uint32_t flat_rgba;                 // r | g << 8 | b << 16 | a << 24
    uint32_t attr_stride;               // floats per vertex in `attr`
    uint32_t cull;                      // 1: skipped when BBox::visibility(mvp) is Hidden (scene.rs:81-87)
    uint32_t prim;                      // PrimType; n_tris counts primitives of that type
    uint32_t pre;                       // 1: vertex slots already filled (depth-sorted clip fans)
    uint32_t sort;                      // depth sort of this render() call: 0 none, 1 front to back, 2 back to front
    uint32_t in_tris, in_verts;         // a pre draw's render() input counts (prims.i, verts.i), for culled draws
    uint64_t vert_base;                 // a pre draw's first slot in the batch's screen vertices
    uint64_t tri_base;                  // first global triangle index
    float mvp[16];                      // row-major ProjMat3 (the uniform)
    float vp[16];                       // row-major Mat4<Ndc, Screen>
    float bbox[6];                      // the mesh's BBox::of (scene.rs:37-39): low x, y, z, high x, y, z
};

struct FrameDesc {
    uint8_t* color;          // device colour buffer
    float* depth;            // device depth buffer or null (colour-only target)
    uint64_t color_stride;   // bytes per row
    uint64_t depth_stride;   // floats per row
    uint32_t width, height, fmt;
    int32_t depth_test, face_cull, color_write, depth_write;
    int32_t clear_color, clear_depth;  // fused Frame::clear (front/src/lib.rs:103-120)
    uint32_t clear_pixel;              // clear colour already in the target format
    float clear_depth_value;           // 1 / depth_clear
    uint32_t ntx, nty;                 // tile grid
    uint32_t tile_base;                // first global tile index of this frame
    uint32_t pad;
};

// Per-frame statistics (stats.rs:16-40), accumulated by the kernels.
// prims.o, and frags.i of the small triangles, are counted in this many
// partial counters per frame, each pair on its own 128-byte line: atomics on
// one address serialise, and a frame of 3.2M small triangles has 50,000 setup
// waves adding to it.
constexpr uint32_t PRIM_PARTS = 16;
constexpr uint32_t PRIM_PART_STRIDE = 16;  // u64 words between partial counters (prims.o, frags.i)

struct FrameStats {
    unsigned long long prims_o, verts_o, frags_i, frags_o;
    unsigned long long hidden_draws, hidden_prims, hidden_verts;  // draws skipped by the bounding-box test
};

// Screen-space triangle as stored by the setup kernel: three vertices of
// (x, y, z, a0, a1, a2) plus the draw index.
struct ScrTri {
    float v[3][6];
    uint32_t draw;
    uint32_t kind;   // the draw's shader kind
};

// A bin run: the triangles of group `group` (64 consecutive global triangle
// indices) that touch one tile, as a bit mask.
struct Run {
    uint32_t group;
    uint32_t multi;  // 1: some triangle of the group has several clip fans (read its header)
    unsigned long long mask;
};

// Runs of a group that k_setup keeps for k_bin; a group of more is walked again.
constexpr uint32_t PRE_RUNS = 32;
constexpr uint32_t RUNS_MULTI = 1u << 31;  // n_runs bit: Run::multi

// Bounds of a group's binned triangles: the rasterizer drops a whole run by them.
struct alignas(16) GroupBound {
    float zmax;       // no fragment's z is above it (NaN: not known)
    uint32_t r0, r1;  // the union of their BatchDesc::rect
    uint32_t pad;
};

// A tile as the rasterizer takes it: all it needs to start, in one load.
struct alignas(16) TileRec {
    uint32_t tile, frame, off, nruns;  // its runs are runs[off .. off + nruns)
};
// Words of BatchDesc::tile_counts.
enum TileCount : uint32_t {
    TN_BUSY = 0,       // tiles with runs
    TN_LONG = 1,       // entries of long_list from its front
    TN_HUGE = 2,       // and from its end
    TN_HEAVIEST = 3,   // entries of heavy_list from its front
    TN_HEAVY = 4,      // and from its end
    TN_HEAVY_MIN = 5,  // tiles of more runs than this are in heavy_list
};
constexpr uint32_t LONG_RUNS = 64, HUGE_RUNS = 1024;  // run lists longer than these (see k_binsort)
// Work counters behind the partitions' (BatchDesc::tile_counter).
constexpr uint32_t TC_EMPTY = TILE_PARTS, TC_HEAVY = TILE_PARTS + 1, TC_LONG = TILE_PARTS + 2, TC_HUGE = TILE_PARTS + 3;
constexpr uint32_t N_TILE_COUNTERS = TILE_PARTS + 4;
// Words between them: on one line, with the tile counts that every wave reads,
// 22,000 atomics from eight dies made the rasterizer wait (32 crates1080 frames:
// 0.62 ms, on lines of their own 0.46).
constexpr uint32_t TC_STRIDE = 32;

// Atomics on one line of memory wait for each other: four counters of
// neighbouring tiles to a line of 128 bytes, where thirty-two took k_bin of 32
// mixed frames 1.22 ms and these 0.74 (k_setup 3.03 -> 2.76; eight a line 0.77
// and 2.83, one a line 0.70 and 2.75, but their scan 0.042 for 0.034).
constexpr uint32_t RUN_STRIDE = 8;  // words
__host__ __device__ inline uint64_t run_slot(uint32_t tile) { return (uint64_t)tile * RUN_STRIDE; }

struct BatchDesc {
    const DrawDesc* draws;
    const FrameDesc* frames;
    FrameStats* stats;
    uint32_t n_draws, n_frames;
    uint64_t n_verts;   // vertex slots of the pre draws
    uint64_t n_tris;    // total input triangles
    uint32_t n_groups;  // ceil(n_tris / 64)
    uint32_t n_tiles;   // total tiles over all frames
    uint32_t tile_w, tile_h;  // rasterizer tile: 16, 32 or 64 columns x 16, 32 or 64 rows
    uint32_t chunk;     // rasterizer span chunk: 6 or 8 pixels (anything else: 8)
    // scratch
    float* sv;           // screen vertex (x, y, z, a0, a1, a2) per slot of the pre draws
    uint32_t* hdr;       // per triangle: surviving fan count | extra base << 3
    ScrTri* scr;         // per triangle: first surviving fan
    ScrTri* extra;       // further fans of clipped triangles
    uint32_t* extra_count;
    uint32_t extra_cap;
    uint32_t* rect;      // per triangle: pixel rect (c0 | r0 << 16, c1 | r1 << 16; all ones: none), 2 words
    float* zmax;         // per triangle: no fragment's z is above it (NaN: not known)
    GroupBound* group_max;  // per group; written where small_tris is set
    uint32_t* tile_of;   // per group, PRE_RUNS: its runs' tiles, and
    unsigned long long* mask_of;  // masks, as k_setup has met them
    uint32_t* n_runs;    // per group: their number | RUNS_MULTI
    uint32_t* run_count; // per tile (run_slot)
    uint32_t* run_off;   // per tile + 1 (exclusive scan)
    uint32_t* run_cursor;  // per tile (run_slot): where its next run goes
    uint32_t* scan_blk;  // per 1024 tiles: run total, then its offset
    TileRec* tiles;        // the tiles with runs in tile order, then, from the end down, the others in tile order
    uint32_t* long_list;   // places in `tiles` of those with a long list of runs, from the front, and a huge one, from the end
    uint32_t* heavy_list;  // places in `tiles` of the heaviest, from the front, and of the heavy ones, from the end
    uint32_t* tile_counts; // TileCount words
    uint32_t small_tris;       // 1: k_setup counts and bounds the small triangles, the rasterizer passes over hidden ones
    uint32_t* group_draw;   // per 64-triangle group: the draw of its first triangle
    Run* runs;
    uint32_t runs_cap;
    uint32_t* tile_counter;  // work counters: one per tile partition, TC_* (N_TILE_COUNTERS)
    uint32_t* err;
    unsigned long long* prims_part;  // per frame: PRIM_PARTS partial counters (prims.o, frags.i)
    uint32_t* draw_vis;  // per draw: 0 if the bounding-box test hid it, else 1
    uint32_t any_cull;   // some draw asks for the bounding-box test
    uint32_t any_lines;  // some draw is of edges
    // depth sort (render.rs:180-183, 209-219): clip fans in clip space, their keys
    uint32_t depth_sort;              // 0 none, 1 front to back, 2 back to front
    uint32_t fan_cap;
    float* fans;                      // per fan: 3 x (x, y, z, w, a0, a1, a2)
    unsigned long long* fan_keys;     // per fan: draw (if it fits) | order key | triangle << 3 | fan
    uint32_t fan_bits;                // bits of the key's last field
    uint32_t fan_draw_keyed;          // 1: the draw is the key's first field
    uint32_t* fan_vals;               // per fan: its index in `fans`
    uint32_t* fan_count;
    uint32_t* fan_draw;               // per fan: its draw
    uint32_t* fan_cnt;                // per draw: its fans
};
constexpr int FAN_FLOATS = 21;

}  // namespace rf
